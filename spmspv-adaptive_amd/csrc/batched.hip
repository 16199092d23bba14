// Batched multi-vector SpMSpV: nvec sparse vectors against one matrix with
// two host synchronisations for the whole batch instead of two per call.
//   1. one launch selects for every vector (exact bin_len and choice per
//      vector); one readback;
//   2. one launch scans the columns of every vector whose slot reads the
//      scan, of as many at a time as the workspace holds (a vector that does
//      not fit alone is scanned in its own pipeline, as a single call is);
//      then every vector's chosen pipeline is queued back to back with
//      its bin_len already known (no readback inside), results at the
//      caller's offsets. Each vector has its own control block, so
//      nothing is copied between two pipelines, and one launch at the end
//      hands all the counts to d_ynnz;
//   3. one final synchronisation.
// 48 vectors of densities 2e-4 to 0.2 on R-MAT s20: 3,270 us with a selector
// launch, a scan and a count copy per vector (12, 10 and 4 us), 2,190 us so.
// No reference counterpart (the reference runs one vector per call).
#include <algorithm>
#include <vector>

#include "handle.hpp"

using namespace spmspv;

// Workspace: the vectors' descriptors, control blocks and selector words, their
// tiles, and the scans of one group of vectors. Reserved for kBatchVecs vectors
// of any size, grown by a batch of more vectors, freed with the handle.
struct BatchState {
  char* mem = nullptr;
  size_t bytes = 0;
};

namespace {

// Places of a group's scans and splits: 48 vectors of R-MAT s20 hold 1.4 M keys.
constexpr int kBatchVecs = 4096, kBatchKeys = 1 << 21, kBatchSplits = 1 << 18;

__global__ void k_batch_counts(const Ctl* __restrict__ ctls, int nvec, int* __restrict__ ynnz) {
  const int v = blockIdx.x * blockDim.x + threadIdx.x;
  if (v < nvec) ynnz[v] = ctls[v].ynnz;
}

size_t up256(size_t v) { return (v + 255) & ~size_t(255); }

// Device layout for nvec vectors in `tiles` tiles, scanned in groups of `places`
// places; the control blocks and arrival counts, which start at zero, come first.
struct Layout {
  size_t ctls, arrive, zeroed, stash, vec, tile_vec, list, tsum, tmax, ptr, xbeg, split, bytes;
  Layout(size_t nvec, size_t tiles, size_t places) {
    size_t o = 0;
    auto take = [&](size_t b) {
      const size_t r = o;
      o = up256(o + b);
      return r;
    };
    ctls = take(nvec * sizeof(Ctl));
    arrive = take(nvec * sizeof(unsigned));
    zeroed = o;
    stash = take(nvec * sizeof(long long));
    vec = take(nvec * sizeof(BatchVec));
    tile_vec = take(tiles * sizeof(int));
    list = take(tiles * sizeof(int));
    tsum = take(tiles * sizeof(long long));
    tmax = take(tiles * sizeof(int));
    ptr = take(places * sizeof(int));
    xbeg = take(places * sizeof(int));
    split = take(kBatchSplits * sizeof(int));
    bytes = o;
  }
};

size_t tiles_of(size_t keys) { return std::max<size_t>(1, (keys + kWideTile - 1) / kWideTile); }

int grow(spmspv_handle_t h, size_t bytes) {
  if (!h->batch) h->batch = new BatchState();
  BatchState* b = h->batch;
  if (b->bytes >= bytes) return SPMSPV_SUCCESS;
  HIP_TRY(h, hipStreamSynchronize(h->stream));
  if (b->mem) HIP_TRY(h, hipFree(b->mem));
  b->mem = nullptr;
  b->bytes = 0;
  HIP_TRY(h, hipMalloc((void**)&b->mem, bytes));
  b->bytes = bytes;
  return SPMSPV_SUCCESS;
}

}  // namespace

namespace spmspv {
int batch_alloc(spmspv_handle_t h) {
  // the vectors' offsets are ints: all their keys lie in 2^31
  const size_t tiles = std::min(kBatchVecs * tiles_of((size_t)h->n), (size_t{1} << 31) / kWideTile + kBatchVecs);
  return grow(h, Layout(kBatchVecs, tiles, kBatchKeys).bytes);
}

void batch_release(spmspv_handle_t h) {
  if (!h || !h->batch) return;
  if (h->batch->mem) (void)hipFree(h->batch->mem);
  delete h->batch;
  h->batch = nullptr;
}
}  // namespace spmspv

extern "C" {

int spmspv_run_batched(spmspv_handle_t h, int nvec, const int* d_vptr, const int* d_vkey,
                       const float* d_vval, const long long* d_yoff, int* d_ykey, float* d_yval,
                       int* d_ynnz, int* kernel_used) {
  if (!h) return set_error(nullptr, SPMSPV_INVALID_ARGUMENT, "null handle");
  if (nvec < 0 || (nvec > 0 && (!d_vptr || !d_yoff || !d_ykey || !d_yval || !d_ynnz)))
    return set_error(h, SPMSPV_INVALID_ARGUMENT, "run_batched: bad arguments");
  if (nvec == 0) return SPMSPV_SUCCESS;
  int rc;
  if ((rc = ensure_arena(h)) || (rc = need_csc(h)) || (rc = ensure_mat_features(h))) return rc;
  hipStream_t s = h->stream;
  std::vector<int> vptr(nvec + 1);
  std::vector<long long> yoff(nvec + 1);
  HIP_TRY(h, hipMemcpyAsync(vptr.data(), d_vptr, sizeof(int) * (nvec + 1), hipMemcpyDeviceToHost, s));
  HIP_TRY(h, hipMemcpyAsync(yoff.data(), d_yoff, sizeof(long long) * (nvec + 1), hipMemcpyDeviceToHost, s));
  HIP_TRY(h, hipStreamSynchronize(s));
  size_t tiles = 0;
  for (int v = 0; v < nvec; ++v) {
    const int xn = vptr[v + 1] - vptr[v];
    if (vptr[v] < 0 || xn < 0 || xn > h->n)
      return set_error(h, SPMSPV_INVALID_ARGUMENT, "run_batched: vector offsets out of range");
    if (xn > 0 && (!d_vkey || !d_vval))
      return set_error(h, SPMSPV_INVALID_ARGUMENT, "run_batched: null vector arrays");
    if (yoff[v] < 0 || yoff[v + 1] < yoff[v])
      return set_error(h, SPMSPV_INVALID_ARGUMENT, "run_batched: output offsets not ascending");
    tiles += tiles_of((size_t)xn);
  }
  const size_t keys = (size_t)(vptr[nvec] - vptr[0]);
  const int places = (int)std::min<size_t>(kBatchKeys, keys + nvec);
  const Layout at((size_t)nvec, tiles, places);
  if ((rc = grow(h, at.bytes))) return rc;
  BatchState* b = h->batch;
  auto* ctls = reinterpret_cast<Ctl*>(b->mem + at.ctls);
  auto* stash = reinterpret_cast<long long*>(b->mem + at.stash);
  auto* d_vec = reinterpret_cast<BatchVec*>(b->mem + at.vec);
  auto* d_tile_vec = reinterpret_cast<int*>(b->mem + at.tile_vec);
  auto* d_list = reinterpret_cast<int*>(b->mem + at.list);
  auto* tsum = reinterpret_cast<long long*>(b->mem + at.tsum);
  auto* ptr = reinterpret_cast<int*>(b->mem + at.ptr);
  auto* xbeg = reinterpret_cast<int*>(b->mem + at.xbeg);
  auto* split = reinterpret_cast<int*>(b->mem + at.split);
  std::vector<BatchVec> h_vec(nvec);
  std::vector<long long> st(nvec);
  std::vector<int> h_tile_vec(tiles), h_list(tiles);
  // 1. selection (the arrival counts and control blocks start at zero)
  int tile = 0;
  for (int v = 0; v < nvec; ++v) {
    const int xn = vptr[v + 1] - vptr[v];
    const int nt = (int)tiles_of((size_t)xn);
    h_vec[v] = BatchVec{vptr[v], xn, tile, nt, 0, 0};
    std::fill_n(h_tile_vec.begin() + tile, nt, v);
    tile += nt;
  }
  HIP_TRY(h, hipMemcpyAsync(d_vec, h_vec.data(), nvec * sizeof(BatchVec), hipMemcpyHostToDevice, s));
  HIP_TRY(h, hipMemcpyAsync(d_tile_vec, h_tile_vec.data(), tiles * sizeof(int), hipMemcpyHostToDevice, s));
  const SelectorArgs sel{h->have_weights ? h->weights_dev : nullptr, h->mat, h->sel_mode, h->sel_fixed,
                         nullptr, 0, -1, 0.f, h->bucket_lo, h->bucket_hi};
  launch_fill_i32(s, reinterpret_cast<int*>(b->mem), (long long)(at.zeroed / 4), 0);
  launch_batch_select(s, h->csc_colptr, d_vkey, h->n, (int)tiles, d_tile_vec, d_vec, tsum,
                      reinterpret_cast<int*>(b->mem + at.tmax), reinterpret_cast<unsigned*>(b->mem + at.arrive), ctls,
                      sel, stash);
  h->launches++;
  HIP_TRY(h, hipGetLastError());
  HIP_TRY(h, hipMemcpyAsync(st.data(), stash, sizeof(long long) * nvec, hipMemcpyDeviceToHost, s));
  HIP_TRY(h, hipStreamSynchronize(s));
  for (int v = 0; v < nvec; ++v) {
    const long long need = std::min<long long>(h->m, sel_word_binlen(st[v]));
    if (yoff[v + 1] - yoff[v] < need)
      return set_error(h, SPMSPV_INVALID_ARGUMENT,
                       "run_batched: output capacity of vector " + std::to_string(v) + " is " +
                           std::to_string(yoff[v + 1] - yoff[v]) + ", needs " + std::to_string(need));
    const int kid = sel_word_choice(st[v]);
    if (kid < 0 || kid > SPMSPV_K_COL_BUCKET)
      return set_error(h, SPMSPV_DEVICE_ERROR, "run_batched: selector returned no slot");
  }
  // x for vector v, with what the selection found
  auto set_x = [&](int v) -> int {
    int r = spmspv_set_sparse_x(h, const_cast<int*>(d_vkey) + vptr[v], const_cast<float*>(d_vval) + vptr[v],
                                vptr[v + 1] - vptr[v]);
    h->binlen_host = sel_word_binlen(st[v]);
    return r;
  };
  struct Unset {
    spmspv_handle_t h;
    ~Unset() { unset_x(h); }
  } unset{h};
  // 2. scans: of the vectors whose slot reads one (the small-x path makes its
  // own), in groups that fit the workspace; a vector's group, -1: none
  std::vector<int> group(nvec, -1), group_list{0};
  int nlist = 0, place = 0, nsplit = 0;
  for (int v = 0; v < nvec; ++v) {
    const int kid = sel_word_choice(st[v]);
    if ((rc = set_x(v))) return rc;
    if (!needs_scan(kid) || takes_small_path(h, kid)) continue;
    const long long sp = (h->xnnz + h->binlen_host) / kLbTile + 3;
    if (h->xnnz >= places || sp > kBatchSplits) continue;
    if (place + h->xnnz + 1 > places || nsplit + sp > kBatchSplits) {
      group_list.push_back(nlist);
      place = nsplit = 0;
    }
    h_vec[v].scan0 = place;
    h_vec[v].split0 = nsplit;
    place += h->xnnz + 1;
    nsplit += (int)sp;
    group[v] = (int)group_list.size() - 1;
    for (int t = 0; t < h_vec[v].ntiles; ++t) h_list[nlist++] = h_vec[v].tile0 + t;
  }
  group_list.push_back(nlist);
  if (nlist > 0) {
    HIP_TRY(h, hipMemcpyAsync(d_vec, h_vec.data(), nvec * sizeof(BatchVec), hipMemcpyHostToDevice, s));
    HIP_TRY(h, hipMemcpyAsync(d_list, h_list.data(), nlist * sizeof(int), hipMemcpyHostToDevice, s));
  }
  // queued pipelines, each on its own control block and scan; a group's scans
  // come before its first vector, after the pipelines of the group before it
  {
    struct Restore {
      spmspv_handle_t h;
      Ctl* ctl;
      int *ptr, *xbeg, *split;
      ~Restore() {
        h->ctl = ctl;
        h->ptr = ptr;
        h->xbeg = xbeg;
        h->split = split;
        h->prep_valid = false;
      }
    } own{h, h->ctl, h->ptr, h->xbeg, h->split};
    int scanned = -1;
    for (int v = 0; v < nvec; ++v) {
      const int kid = sel_word_choice(st[v]);
      if (kernel_used) kernel_used[v] = kid;
      if (group[v] > scanned) {
        scanned = group[v];
        const int l0 = group_list[scanned], l1 = group_list[scanned + 1];
        launch_batch_scan(s, h->csc_colptr, d_vkey, h->n, l1 - l0, d_list + l0, d_tile_vec, d_vec, tsum, ptr, xbeg,
                          split);
        h->launches++;
        HIP_TRY(h, hipGetLastError());
      }
      if ((rc = set_x(v))) return rc;
      const bool in = group[v] >= 0;
      h->ctl = ctls + v;
      h->ptr = in ? ptr + h_vec[v].scan0 : own.ptr;
      h->xbeg = in ? xbeg + h_vec[v].scan0 : own.xbeg;
      h->split = in ? split + h_vec[v].split0 : own.split;
      h->prep_valid = in;
      if ((rc = run_kernel(h, kid, nullptr, d_ykey + yoff[v], d_yval + yoff[v], true))) return rc;
    }
    hipLaunchKernelGGL(k_batch_counts, dim3((nvec + 255) / 256), dim3(256), 0, s, ctls, nvec, d_ynnz);
    HIP_TRY(h, hipGetLastError());
  }
  // 3. the batch is complete when this returns; x is left unset
  HIP_TRY(h, hipStreamSynchronize(s));
  return SPMSPV_SUCCESS;
}

}  // extern "C"
