// PageRank-style driver: residual-push PageRank whose every iteration is
// one selector-dispatched SpMSpV. The reference has no such driver; its
// harnesses replay frontiers recorded from a PageRank run, one sparse x
// per line of pr_x_<matrix>.txt (la/test/test_application.cu:206-210,
// 252-256; la/test/new_test_app.cu:293-299). This produces those frontiers
// on the device and runs them.
//
// Transition matrix: column u of the CSC holds u's out-edges with weights
// a_vu; the walk moves from u to v with probability a_vu / w_u, where
// w_u = sum_v a_vu (unit weights give the usual PageRank; columns with no
// entries keep their mass). With teleport (1 - d) / n the ranks are the
// solution of (I - d A W^-1) p = (1 - d) / n.
//
// Residual push: p = 0, r = (1 - d) / n everywhere, every vertex active.
// Per iteration, for the active set S (sorted keys):
//   take:  p[u] += r[u]; x_u = r[u] / w_u; r[u] = 0          (u in S)
//   y = A x                    (the selector's slot, sorted output)
//   push:  r[v] += d * y_v; v joins the next S if r[v] > eps * (1 - d) / n
// (only vertices that received a push can cross the threshold: every
// other vertex above it was in S and is now at 0). At the end p += r.
// With every residual at most eps (1 - d) / n, sum|p - p*| <= eps * d.
//
// y's keys are sorted and distinct, so the vertices that cross the threshold
// come out in order: one kernel pushes, lists them and takes their residuals
// for the next iteration (k_pr_push). It reads y's count on the device, so the
// host waits once per iteration, for the next set's size. An iteration is
// launches and short kernels: with separate take, push, compaction and count
// kernels (6 to 20 us each, the push waiting on one atomic per vertex) and a
// second wait for y's count, R-MAT s18 at eps 1e-4 took 7,400 us, 85
// iterations, 5,300 us so.
#include <chrono>

#include "handle.hpp"

using namespace spmspv;

struct PrState {
  void* alloc = nullptr;
  float* w = nullptr;         // n: column weight sums
  float* r = nullptr;         // n: residuals
  int* fk[2] = {nullptr, nullptr};  // n: active keys (sorted)
  float* fv[2] = {nullptr, nullptr};  // n: x values of the active set
  int* yk = nullptr;          // m
  float* yv = nullptr;        // m
};

namespace {

constexpr int kPrNT = 256, kPrIPT = 8, kPrTile = kPrNT * kPrIPT;  // k_pr_push
static_assert(kPrTile >= kPrepTile, "the look-back words are laid out for k_prep's tiles");
constexpr int kLongCol = 1024;

// Weight sums of the columns of at most kLongCol entries, a team of 16 lanes
// per column.
__global__ __launch_bounds__(256) void k_col_weights(const int* __restrict__ colptr, const float* __restrict__ cval,
                                                     int n, float* __restrict__ w) {
  constexpr int TEAM = 16;
  const int tl = threadIdx.x & (TEAM - 1);
  const long long nt = (long long)gridDim.x * blockDim.x / TEAM;
  for (long long c = ((long long)blockIdx.x * blockDim.x + threadIdx.x) / TEAM; c < n; c += nt) {
    const int b = colptr[c], e = colptr[c + 1];
    if (e - b > kLongCol) continue;
    float s = 0.f;
    for (int i = b + tl; i < e; i += 4 * TEAM) {
      float v[4];
#pragma unroll
      for (int k = 0; k < 4; ++k) v[k] = i + k * TEAM < e ? cval[i + k * TEAM] : 0.f;
      s += (v[0] + v[1]) + (v[2] + v[3]);
    }
#pragma unroll
    for (int o = TEAM / 2; o > 0; o >>= 1) s += __shfl_xor(s, o, TEAM);
    if (tl == 0) w[c] = s;
  }
}

// The longer ones, a workgroup per column (one wave per hub column took 480 us
// at R-MAT s18). Each workgroup looks through its own stride of columns, so
// that hubs beside each other spread over the workgroups; the number of
// workgroups is prime, since R-MAT's hubs also share their low bits.
template <int NT>
__global__ __launch_bounds__(NT) void k_long_col_weights(const int* __restrict__ colptr,
                                                         const float* __restrict__ cval, int n,
                                                         float* __restrict__ w) {
  __shared__ int s_cols[NT];
  __shared__ int s_i[NT / kWave];
  __shared__ float s_f[NT / kWave];
  for (long long k0 = 0; k0 * gridDim.x + blockIdx.x < n; k0 += NT) {
    const long long c = (k0 + threadIdx.x) * gridDim.x + blockIdx.x;
    const int is_long = c < n && colptr[c + 1] - colptr[c] > kLongCol ? 1 : 0;
    int tot;
    const int pos = block_excl_sum<NT, int>(is_long, s_i, &tot);
    if (is_long) s_cols[pos] = (int)c;
    __syncthreads();
    for (int q = 0; q < tot; ++q) {
      const int col = s_cols[q], b = colptr[col], e = colptr[col + 1];
      float s = 0.f;
      for (int i = b + (int)threadIdx.x; i < e; i += 4 * NT) {
        float v[4];
#pragma unroll
        for (int k = 0; k < 4; ++k) v[k] = i + k * NT < e ? cval[i + k * NT] : 0.f;
        s += (v[0] + v[1]) + (v[2] + v[3]);
      }
      s = block_sum<NT, float>(s, s_f);
      if (threadIdx.x == 0) w[col] = s;
    }
    __syncthreads();
  }
}

__device__ __forceinline__ float share(float r, float w) { return w > 0.f ? r / w : 0.f; }

// p, r, and the first active set (every vertex) with its residuals taken.
__global__ void k_pr_init(int n, float r0, const float* __restrict__ w, float* __restrict__ p,
                          float* __restrict__ r, int* __restrict__ fk, float* __restrict__ fv) {
  for (int v = blockIdx.x * blockDim.x + threadIdx.x; v < n; v += gridDim.x * blockDim.x) {
    p[v] = r0;
    r[v] = 0.f;
    fk[v] = v;
    fv[v] = share(r0, w[v]);
  }
}

// r[v] += d * y_v; the vertices over the threshold, in y's (ascending) order,
// are the next active set: listed with their x value, their residual taken.
// Tiles of kPrTile entries of y with decoupled look-back; the last one sends
// the set's size to the host, which only queues further work on this stream.
__global__ __launch_bounds__(kPrNT) void k_pr_push(const int* __restrict__ yk, const float* __restrict__ yv,
                                                   Ctl* ctl, float d, float thr, const float* __restrict__ w,
                                                   float* __restrict__ p, float* __restrict__ r,
                                                   int* __restrict__ fk, float* __restrict__ fv,
                                                   unsigned long long* state, Ep ep, long long* sig) {
  __shared__ unsigned long long s_pre;
  __shared__ int s_w[kPrNT / kWave];
  const int cnt = ctl->ynnz;  // y's keys are distinct: one writer per r[v]
  const unsigned ntiles = (unsigned)((cnt + kPrTile - 1) / kPrTile);
  const unsigned t = blockIdx.x;
  if (t >= ntiles) {
    if (ntiles == 0 && t == 0 && threadIdx.x == 0) *sig = 0;
    return;
  }
  const int wv = threadIdx.x / kWave;
  const int i0 = (int)t * kPrTile + wv * kWave * kPrIPT + lane();
  int v[kPrIPT];
  float nr[kPrIPT], wt[kPrIPT];
  // entries past the end repeat the last one and are not stored
#pragma unroll
  for (int j = 0; j < kPrIPT; ++j) {
    const int i = min(i0 + j * kWave, cnt - 1);
    v[j] = yk[i];
    nr[j] = yv[i];
  }
#pragma unroll
  for (int j = 0; j < kPrIPT; ++j) {
    nr[j] = r[v[j]] + d * nr[j];
    wt[j] = w[v[j]];
  }
  const uint64_t lt = lane() == 0 ? 0ull : (~0ull >> (kWave - lane()));
  int rank[kPrIPT], mine = 0;
  bool over[kPrIPT];
#pragma unroll
  for (int j = 0; j < kPrIPT; ++j) {
    const bool in = i0 + j * kWave < cnt;
    over[j] = in && nr[j] > thr;
    const uint64_t bal = __ballot(over[j]);
    rank[j] = mine + __popcll(bal & lt);
    mine += __popcll(bal);
    if (in) r[v[j]] = over[j] ? 0.f : nr[j];
    if (over[j]) p[v[j]] += nr[j];
  }
  if (lane() == 0) s_w[wv] = mine;
  __syncthreads();
  int before = 0, tot = 0;
#pragma unroll
  for (int k = 0; k < kPrNT / kWave; ++k) {
    before += k < wv ? s_w[k] : 0;
    tot += s_w[k];
  }
  const long long pre = (long long)tile_prefix(state, t, ep_of(ctl, ep), (unsigned long long)tot, &s_pre);
#pragma unroll
  for (int j = 0; j < kPrIPT; ++j) {
    if (over[j]) {
      const long long o = pre + before + rank[j];
      fk[o] = v[j];
      fv[o] = share(nr[j], wt[j]);
    }
  }
  if (t == ntiles - 1 && threadIdx.x == 0) *sig = pre + tot;
}

__global__ void k_pr_finish(int n, float* __restrict__ p, const float* __restrict__ r) {
  for (int v = blockIdx.x * blockDim.x + threadIdx.x; v < n; v += gridDim.x * blockDim.x) p[v] += r[v];
}

int grid_of(long long items) {
  return (int)std::max<long long>(1, std::min<long long>(4096, (items + 255) / 256));
}

}  // namespace

namespace spmspv {
// PageRank buffers, sized by m and n: allocated once per handle.
int pr_alloc(spmspv_handle_t h) {
  if (h->pr) return SPMSPV_SUCCESS;
  auto* st = new PrState();
  const size_t n = h->n, m = h->m;
  size_t off = 0;
  auto take = [&](size_t bytes) {
    const size_t o = off;
    off = (off + bytes + 255) / 256 * 256;
    return o;
  };
  const size_t ow = take(n * 4), orr = take(n * 4), of0 = take(n * 4), of1 = take(n * 4);
  const size_t ov0 = take(n * 4), ov1 = take(n * 4);
  const size_t oyk = take(m * 4), oyv = take(m * 4);
  if (hipMalloc(&st->alloc, off) != hipSuccess) {
    delete st;
    return set_error(h, SPMSPV_OUT_OF_MEMORY, "pagerank buffers");
  }
  char* p = static_cast<char*>(st->alloc);
  st->w = reinterpret_cast<float*>(p + ow);
  st->r = reinterpret_cast<float*>(p + orr);
  st->fk[0] = reinterpret_cast<int*>(p + of0);
  st->fk[1] = reinterpret_cast<int*>(p + of1);
  st->fv[0] = reinterpret_cast<float*>(p + ov0);
  st->fv[1] = reinterpret_cast<float*>(p + ov1);
  st->yk = reinterpret_cast<int*>(p + oyk);
  st->yv = reinterpret_cast<float*>(p + oyv);
  h->pr = st;
  return SPMSPV_SUCCESS;
}

void pr_release(spmspv_handle_t h) {
  if (!h || !h->pr) return;
  if (h->pr->alloc) (void)hipFree(h->pr->alloc);
  delete h->pr;
  h->pr = nullptr;
}
}  // namespace spmspv

extern "C" {

int spmspv_pagerank(spmspv_handle_t h, float damping, float eps, int max_iter, int policy,
                    float* d_rank, double stats[4], int* sizes) {
  if (!h) return set_error(nullptr, SPMSPV_INVALID_ARGUMENT, "null handle");
  if (!d_rank || !(damping > 0.f && damping < 1.f) || !(eps > 0.f) || max_iter < 1 || policy < -1 ||
      policy >= SPMSPV_NUM_SLOTS)
    return set_error(h, SPMSPV_INVALID_ARGUMENT, "pagerank: bad damping, eps, max_iter, policy or rank");
  if (h->m != h->n) return set_error(h, SPMSPV_INVALID_ARGUMENT, "pagerank needs a square matrix");
  int rc;
  if ((rc = ensure_arena(h)) || (rc = need_csc(h)) || (rc = ensure_mat_features(h)) || (rc = pr_alloc(h)))
    return rc;
  PrState* st = h->pr;
  hipStream_t s = h->stream;
  const int n = h->n;
  const int saved_mode = h->sel_mode, saved_fixed = h->sel_fixed;
  if (policy >= 0) {
    h->sel_mode = 2;
    h->sel_fixed = policy;
  }
  struct Restore {
    spmspv_handle_t h;
    int mode, fixed;
    ~Restore() {
      h->sel_mode = mode;
      h->sel_fixed = fixed;
      unset_x(h);  // x was the driver's own buffer
    }
  } restore{h, saved_mode, saved_fixed};
  const auto t0 = std::chrono::steady_clock::now();
  hipLaunchKernelGGL(k_col_weights, dim3(grid_of((long long)n * 16)), dim3(256), 0, s, h->csc_colptr, h->csc_val, n,
                     st->w);
  if (h->nnz > kLongCol)
    hipLaunchKernelGGL(k_long_col_weights<512>, dim3(509), dim3(512), 0, s, h->csc_colptr, h->csc_val, n, st->w);
  const float r0 = (1.f - damping) / (float)n;
  const float thr = eps * r0;
  hipLaunchKernelGGL(k_pr_init, dim3(grid_of(n)), dim3(256), 0, s, n, r0, st->w, d_rank, st->r, st->fk[0], st->fv[0]);
  HIP_TRY(h, hipGetLastError());
  int cur = 0, cnt = n, it = 0;
  double pushes = 0.0;
  while (cnt > 0 && it < max_iter) {
    if (sizes) sizes[it] = cnt;
    pushes += cnt;
    if ((rc = spmspv_set_sparse_x(h, st->fk[cur], st->fv[cur], cnt))) return rc;
    int used = -1;
    if ((rc = spmspv_run_auto(h, 1.f, nullptr, st->yk, st->yv, nullptr, &used))) return rc;
    __atomic_store_n(h->sig + 3, kSigPending, __ATOMIC_RELEASE);
    hipLaunchKernelGGL(k_pr_push, dim3((unsigned)((h->m + kPrTile - 1) / kPrTile)), dim3(kPrNT), 0, s, st->yk, st->yv,
                       h->ctl, damping, thr, st->w, d_rank, st->r, st->fk[cur ^ 1], st->fv[cur ^ 1], h->scan_state,
                       next_ep(h, 1), h->sig_dev + 3);
    HIP_TRY(h, hipGetLastError());
    long long next = 0;
    if ((rc = wait_signal(h, 3, &next))) return rc;
    cnt = (int)next;
    cur ^= 1;
    ++it;
  }
  hipLaunchKernelGGL(k_pr_finish, dim3(grid_of(n)), dim3(256), 0, s, n, d_rank, st->r);
  HIP_TRY(h, hipGetLastError());
  HIP_TRY(h, hipStreamSynchronize(s));
  if (stats) {
    stats[0] = it;
    stats[1] = std::chrono::duration<double>(std::chrono::steady_clock::now() - t0).count();
    stats[2] = pushes;
    stats[3] = cnt;  // vertices still above the threshold (0 when converged)
  }
  return SPMSPV_SUCCESS;
}

}  // extern "C"
