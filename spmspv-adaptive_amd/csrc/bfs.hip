// Level-synchronous BFS on the boolean (OR, AND) semiring, one SpMSpV per
// level with the frontier as sparse x. The reference has no BFS loop: it
// replays frontier files recorded elsewhere (la/test/test_application.cu:
// 207-261, frontier format readsvmdata.hpp:308-348), so this driver is new.
//
// A level runs the boolean form of the slot chosen for it (row and column
// indices only: no matrix value is read and no FP32 arithmetic is done):
//   K0/K2  top-down: frontier vertices scan their columns and mark
//          unvisited rows (naive team per vertex / merge-path balanced);
//   K1/K3  top-down gather of all neighbours' row keys, in-house radix sort
//          of the keys alone, then each distinct row marked;
//   K4/K5/K7  by direction: where the frontier holds more than 1 / kTopDown of
//          the edges, bottom-up: each unvisited row scans its neighbours and
//          stops at the first frontier member (on booleans the masked and
//          unmasked load-balanced row products coincide, and a row's result is
//          known at its first hit: the merge-path scan of every nonzero that
//          K5/K7 ran before took 420 us at a large level of R-MAT s22, this 60
//          to 120 us). Below that few rows stop early and K2's kernels run;
//   K6     naive row scan without early exit.
// Every slot marks the rows it reaches in the next frontier's bit array;
// one collect pass then takes the unvisited ones among them, writes their
// levels and lists them, with one list append per workgroup round: device
// atomics on one address take 16 ns each, and an append per wave in every
// slot kernel had made those kernels wait for the counter. R-MAT s22, one
// source: 1,440 -> 450 us.
// Levels are int32 and unique, so any order of claims gives the same
// levels. The selector for level L+1 runs in the same stream right after
// level L (column scan and features of the new frontier + MLP, one launch),
// whose selecting workgroup writes the frontier's features and then its size
// and the choice, tagged with the level counter, into host-coherent words; the
// host polls the last one (no stream wait, no copies); with graphs on, each
// (slot, parity) level sequence is captured once as a hipGraph and replayed.
// Every kernel reads the frontier size from device memory, which is what makes
// the capture valid for any level.
#include <hip/hip_runtime.h>

#include <chrono>
#include <cmath>
#include <cstring>

#include "handle.hpp"
#include "selector.hpp"

using namespace spmspv;

struct BfsState {
  unsigned* visited = nullptr;              // n bits
  unsigned* fbits[2] = {nullptr, nullptr};  // frontier bit arrays
  int* front[2] = {nullptr, nullptr};       // frontier lists
  int* cnt = nullptr;                       // [0],[1] sizes, [2] level, [3] bottom-up queue size
  int2* queue = nullptr;                    // bottom-up: (row, chunk) items the head left undecided
  unsigned long long* reached = nullptr;    // [0] vertices, [1] degree sum
  void* alloc = nullptr;
  hipStream_t own_stream = nullptr;
  int* levels_bound = nullptr;              // levels array the graphs were captured with
  int bound_mode = -9, bound_fixed = -9;    // selector settings captured in the graphs
  const float* bound_weights = nullptr;
  hipGraphExec_t graph[8][2] = {};
};

namespace {

constexpr int kBfsGrid = 2048;
constexpr int kBfsNT = 256;
constexpr int kBuBatch = 8;    // neighbours each row tests in the bottom-up head pass
constexpr int kBuTeam = 16;    // lanes per queued item in the bottom-up tail pass
constexpr int kBuChunk = 256;  // neighbours per queued item
constexpr int kBuUnroll = 4;   // neighbours a lane has in flight
constexpr int kBuRows = 8;     // most rows per thread and queue append

// The row slots' direction: top-down up to this part of the edges in the
// frontier. A level in us, top-down / bottom-up / every nonzero by merge path
// (frontier's edges of all): R-MAT s22 16 / 679 / 385 (1 of 128 M), 62 / 369 /
// 470 (0.13 %), 94 / 335 / 493 (1.1 %), 414 / 151 / 511 (17 %); s20 37 / 217 /
// 131 (0.2 %), 246 / 50 / 141 (33 %); s18 41 / 46 / 52 (0.33 %), 66 / 40 / 58
// (7.8 %); uniform, 1 M vertices 103 / 179 / 145 (2.8 %), 246 / 117 / 157
// (10.5 %); a 1,000 x 1,000 grid 17 / 27 / 34.
constexpr int kTopDown = 32;

// Marks row v in the next frontier unless it is visited or marked already
// (visited is constant while a slot's kernels run).
__device__ __forceinline__ void mark_row(const unsigned* __restrict__ visited, unsigned* nbits, int v) {
  const unsigned bit = 1u << (v & 31);
  if (visited[v >> 5] & bit) return;
  unsigned* w = nbits + (v >> 5);
  if (__hip_atomic_load(w, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) & bit) return;
  atomicOr(w, bit);
}

__global__ void k_bfs_init(int* levels, int n, unsigned* visited, unsigned* fb0, unsigned* fb1,
                           int* front0, int* cnt, unsigned long long* reached, int src) {
  const int words = (n + 31) >> 5;
  for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x)
    levels[i] = i == src ? 0 : -1;
  for (int w = blockIdx.x * blockDim.x + threadIdx.x; w < words; w += gridDim.x * blockDim.x) {
    const unsigned b = (w == (src >> 5)) ? (1u << (src & 31)) : 0u;
    visited[w] = b;
    fb0[w] = b;
    fb1[w] = 0u;
  }
  if (blockIdx.x == 0 && threadIdx.x == 0) {
    front0[0] = src;
    cnt[0] = 1;
    cnt[1] = 0;
    cnt[2] = 0;
    cnt[3] = 0;
    reached[0] = 0;
    reached[1] = 0;
    reached[2] = 0;
  }
}

// K0: top-down, a team of 2^lg lanes per frontier vertex.
__global__ __launch_bounds__(kBfsNT) void k_td_naive(const int* __restrict__ colptr,
                                                     const int* __restrict__ crow,
                                                     const int* __restrict__ f, const int* __restrict__ cnt,
                                                     int cur, int lg, const unsigned* __restrict__ visited,
                                                     unsigned* nbits) {
  const int fsz = cnt[cur];
  const int team = 1 << lg;
  const int tl = threadIdx.x & (team - 1);
  const long long t0 = ((long long)blockIdx.x * blockDim.x + threadIdx.x) >> lg;
  const long long nt = ((long long)gridDim.x * blockDim.x) >> lg;
  for (long long i = t0; i < fsz; i += nt) {
    const int u = f[i];
    const int b = colptr[u], e = colptr[u + 1];
    for (int k = b + tl; k < e; k += team) mark_row(visited, nbits, crow[k]);
  }
}

// K2: top-down over merge-path tiles of (frontier entries + edges), using
// the splits k_prep wrote for the frontier.
template <int NT, int VT>
__global__ __launch_bounds__(NT) void k_td_lb(const int* __restrict__ ptr,
                                              const int* __restrict__ xbeg,
                                              const int* __restrict__ split,
                                              const int* __restrict__ crow, const Ctl* ctl,
                                              const int* __restrict__ cnt, int cur,
                                              const unsigned* __restrict__ visited, unsigned* nbits) {
  constexpr int T = NT * VT;
  __shared__ int s_ptr[T + 2];
  __shared__ int s_beg[T + 2];
  __shared__ int s_seg[T];
  const int xnnz = cnt[cur];
  const long long ntiles = ctl->n_tiles;
  const long long W = (long long)xnnz + ctl->bin_len;
  for (long long t = blockIdx.x; t < ntiles; t += gridDim.x) {
    const long long d0 = t * T, d1 = min(d0 + T, W);
    const int a0 = split[t], a1 = split[t + 1];
    const long long b0 = d0 - a0, b1 = d1 - a1;
    const int sa = a0 > 0 ? a0 - 1 : 0;
    const int nseg = a1 - sa + 1;
    for (int k = threadIdx.x; k < nseg; k += NT) {
      s_ptr[k] = ptr[sa + k];
      if (sa + k < xnnz) s_beg[k] = xbeg[sa + k];
    }
    __syncthreads();
    long long D = d0 + (long long)threadIdx.x * VT;
    if (D < d1) {
      int lo = a0, hi = a1;
      while (lo < hi) {
        const int mid = (lo + hi) >> 1;
        if ((long long)mid + s_ptr[mid - sa] < D) lo = mid + 1;
        else hi = mid;
      }
      int i = lo;
      long long p = D - i;
      for (int k = 0; k < VT && D < d1; ++k, ++D) {
        if (i < a1 && (long long)i + s_ptr[i - sa] == D) ++i;
        else s_seg[(p++) - b0] = i - 1 - sa;
      }
    }
    __syncthreads();
    // all of a thread's rows are loaded before the first is tested
    const int np = (int)(b1 - b0);
    int v[VT];
#pragma unroll
    for (int j = 0; j < VT; ++j) {
      const int q = j * NT + threadIdx.x;
      v[j] = -1;
      if (q < np) {
        const int sg = s_seg[q];
        v[j] = crow[s_beg[sg] + (int)(b0 + q - s_ptr[sg])];
      }
    }
#pragma unroll
    for (int j = 0; j < VT; ++j)
      if (v[j] >= 0) mark_row(visited, nbits, v[j]);
    __syncthreads();
  }
}

// After the sort slots: marks the distinct rows of a sorted key list of
// *n_dev items (repeats are skipped without a test).
__global__ void k_mark_sorted(const unsigned* __restrict__ keys, const long long* __restrict__ n_dev,
                              const unsigned* __restrict__ visited, unsigned* nbits) {
  const long long k = *n_dev;
  for (long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x; i < k;
       i += (long long)gridDim.x * blockDim.x) {
    const unsigned v = keys[i];
    if (i == 0 || keys[i - 1] != v) mark_row(visited, nbits, (int)v);
  }
}

// Bottom-up step of a direction-optimising BFS, in two passes. Head: one
// lane per unvisited row tests its first B neighbours (the column loads, then
// the frontier-bit loads, each issued together); a wave owns 64 rows and
// stores their two bit words without atomics. A row with no hit among more
// than B neighbours is queued in chunks of kBuChunk neighbours, with one
// append per workgroup and `rows` (<= kBuRows) rows per thread. Tail: a team
// of kBuTeam lanes per queued chunk, kBuTeam * kBuUnroll neighbours per step,
// stops at the first hit (its own, or one that another chunk of the row
// has marked when it starts). A team per row for every row keeps a whole wave
// on a row until each of its lanes is done (64 ms for a small-frontier level
// of R-MAT s22 with one wave per row), and one lane per row for every row
// leaves a wave waiting on its longest row (86 ms); in R-MAT rows the hubs
// come first (low ids), so once the frontier holds them most rows stop in the
// head.
template <int B>
__global__ __launch_bounds__(kBfsNT) void k_bu_head(const int* __restrict__ row_ptr,
                                                    const int* __restrict__ col, int m, int rows,
                                                    const unsigned* __restrict__ fbits,
                                                    const unsigned* __restrict__ visited, unsigned* nbits,
                                                    int2* queue, int* qcount) {
  __shared__ int s_i[kBfsNT / kWave];
  __shared__ int s_base;
  const long long step = (long long)kBfsNT * rows;
  for (long long b0 = (long long)blockIdx.x * step; b0 < m; b0 += (long long)gridDim.x * step) {
    int nc[kBuRows];
    int mine = 0;
#pragma unroll
    for (int k = 0; k < kBuRows; ++k) {
      nc[k] = 0;
      if (k >= rows) continue;
      const long long r = b0 + (long long)k * kBfsNT + threadIdx.x;
      int b = 0, e = 0;
      if (r < m && !((visited[r >> 5] >> (r & 31)) & 1u)) {
        b = row_ptr[r];
        e = row_ptr[r + 1];
      }
      bool found = false;
      if (b < e) {
        int u[B];
#pragma unroll
        for (int j = 0; j < B; ++j) u[j] = col[min(b + j, e - 1)];
        unsigned w[B];
#pragma unroll
        for (int j = 0; j < B; ++j) w[j] = fbits[(unsigned)u[j] >> 5];
#pragma unroll
        for (int j = 0; j < B; ++j) found = found || ((w[j] >> (u[j] & 31)) & 1u);
        if (!found && e - b > B) nc[k] = (e - b - B + kBuChunk - 1) / kBuChunk;
        mine += nc[k];
      }
      const uint64_t bal = __ballot(found);
      const unsigned half = lane() < 32 ? (unsigned)bal : (unsigned)(bal >> 32);
      if ((lane() & 31) == 0 && half) nbits[r >> 5] = half;
    }
    int tot;
    int pos = block_excl_sum<kBfsNT, int>(mine, s_i, &tot);
    if (tot == 0) continue;  // the same in every thread
    if (threadIdx.x == 0) s_base = atomicAdd(qcount, tot);
    __syncthreads();
    pos += s_base;
    __syncthreads();
#pragma unroll
    for (int k = 0; k < kBuRows; ++k) {
      const int r = (int)(b0 + (long long)k * kBfsNT + threadIdx.x);
      for (int q = 0; q < nc[k]; ++q) queue[pos++] = make_int2(r, q);
    }
  }
}

template <int B>
__global__ __launch_bounds__(kBfsNT) void k_bu_tail(const int* __restrict__ row_ptr,
                                                    const int* __restrict__ col,
                                                    const unsigned* __restrict__ fbits, unsigned* nbits,
                                                    const int2* __restrict__ queue,
                                                    const int* __restrict__ qcount) {
  const int nq = *qcount;
  const int tl = threadIdx.x & (kBuTeam - 1);
  const long long team = ((long long)blockIdx.x * blockDim.x + threadIdx.x) / kBuTeam;
  const long long nteams = (long long)gridDim.x * blockDim.x / kBuTeam;
  const long long wbase = team - (team % (kWave / kBuTeam));
  for (long long t0 = wbase; t0 < nq; t0 += nteams) {
    const long long t = t0 + (team - wbase);
    int r = 0, b = 0, e = 0;
    bool open = false;
    if (t < nq) {
      const int2 it = queue[t];
      r = it.x;
      b = row_ptr[r] + B + it.y * kBuChunk;
      e = min(b + kBuChunk, row_ptr[r + 1]);
      const unsigned w = __hip_atomic_load(nbits + (r >> 5), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      open = !((w >> (r & 31)) & 1u);
    }
    int found = 0;
    // wave-uniform trips: until every team's chunk ends or has a hit
    for (int k0 = b; __ballot(open && !found && k0 < e) != 0ull; k0 += kBuTeam * kBuUnroll) {
      int u[kBuUnroll];
#pragma unroll
      for (int j = 0; j < kBuUnroll; ++j) {
        const int k = k0 + j * kBuTeam + tl;
        u[j] = open && !found && k < e ? col[k] : -1;
      }
#pragma unroll
      for (int j = 0; j < kBuUnroll; ++j)
        if (u[j] >= 0) found |= (int)((fbits[(unsigned)u[j] >> 5] >> (u[j] & 31)) & 1u);
#pragma unroll
      for (int o = kBuTeam >> 1; o > 0; o >>= 1) found |= __shfl_xor(found, o, kWave);
    }
    if (found && tl == 0) atomicOr(nbits + (r >> 5), 1u << (r & 31));
  }
}

// Ends a level: of the marked rows the unvisited ones (they stay marked: the
// next frontier's bits) become visited, get their level and are listed; the
// consumed frontier's bits are cleared for the level after the next. A thread
// takes a word of 32 rows; where a wave's words hold many rows, its lanes
// take the rows of two words at a time, so that levels and list entries
// leave as adjacent words.
__global__ __launch_bounds__(kBfsNT) void k_bfs_collect(unsigned* nbits, unsigned* cbits, int n, int* cnt, int cur,
                                                        unsigned* visited, int* __restrict__ levels,
                                                        int* __restrict__ nf) {
  __shared__ int s_i[kBfsNT / kWave];
  __shared__ int s_base;
  const int level = cnt[2];
  const int words = (n + 31) >> 5;
  for (int w0 = blockIdx.x * kBfsNT; w0 < words; w0 += gridDim.x * kBfsNT) {
    const int w = w0 + threadIdx.x;
    unsigned nw = 0;
    if (w < words) {
      cbits[w] = 0u;
      const unsigned h = nbits[w];
      if (h) {
        const unsigned vis = visited[w];
        nw = h & ~vis;
        if (nw != h) nbits[w] = nw;
        if (nw) visited[w] = vis | nw;
      }
    }
    const int c = __popc(nw);
    int tot;
    int pos = block_excl_sum<kBfsNT, int>(c, s_i, &tot);
    if (tot == 0) continue;  // the same in every thread
    if (threadIdx.x == 0) s_base = atomicAdd(cnt + (cur ^ 1), tot);
    __syncthreads();
    pos += s_base;
    __syncthreads();
    if (wave_sum(c) > 2 * kWave) {
      const int wb = w0 + (threadIdx.x & ~(kWave - 1));
      const int bit = lane() & 31;
#pragma unroll 4
      for (int k = 0; k < kWave / 2; ++k) {
        const int src = 2 * k + (lane() >> 5);
        const unsigned word = __shfl(nw, src, kWave);
        const int p = __shfl(pos, src, kWave);
        if ((word >> bit) & 1u) {
          const int v = ((wb + src) << 5) + bit;
          levels[v] = level;
          nf[p + __popc(word & ((1u << bit) - 1u))] = v;
        }
      }
    } else {
      while (nw) {
        const int v = (w << 5) + __ffs(nw) - 1;
        nw &= nw - 1;
        levels[v] = level;
        nf[pos++] = v;
      }
    }
  }
}

// Graph500 edge count: sum of degrees over reached vertices.
template <int NT>
__global__ __launch_bounds__(NT) void k_reached(const int* __restrict__ levels, const int* __restrict__ colptr,
                                                int n, unsigned long long* out, long long* sig) {
  __shared__ long long s_l[NT / kWave];
  long long c = 0, d = 0;
  for (int v = blockIdx.x * blockDim.x + threadIdx.x; v < n; v += gridDim.x * blockDim.x) {
    const int len = colptr[v + 1] - colptr[v];
    if (levels[v] >= 0) {
      ++c;
      d += len;
    }
  }
  c = block_sum<NT, long long>(c, s_l);
  d = block_sum<NT, long long>(d, s_l);
  if (threadIdx.x == 0) count_to_host((unsigned long long)c, (unsigned long long)d, out, sig);
}

int lg2(int t) {
  int l = 0;
  while ((1 << l) < t && l < 6) ++l;
  return l;
}

// Enqueues one level on stream s: the slot's kernels on frontier `cur`, the
// collect pass, and the column scan of the new frontier with the selector and
// the host's words.
void enqueue_level(spmspv_handle_t h, hipStream_t s, int slot, int cur, int* levels,
                   const SelectorArgs& sel) {
  BfsState* b = h->bfs;
  const int nxt = cur ^ 1;
  const int words = (h->n + 31) / 32;
  int* f = b->front[cur];
  int* nf = b->front[nxt];
  unsigned* nbits = b->fbits[nxt];
  switch (slot) {
    case SPMSPV_K_COL_NAIVE_ATOMIC:
      hipLaunchKernelGGL(k_td_naive, dim3(kBfsGrid), dim3(kBfsNT), 0, s, h->csc_colptr, h->csc_row, f,
                         b->cnt, cur, lg2(h->team_col), b->visited, nbits);
      break;
    case SPMSPV_K_COL_LB_ATOMIC:
      hipLaunchKernelGGL((k_td_lb<kLbNT, kLbVT>), dim3(kBfsGrid), dim3(kLbNT), 0, s, h->ptr, h->xbeg,
                         h->split, h->csc_row, h->ctl, b->cnt, cur, b->visited, nbits);
      break;
    case SPMSPV_K_COL_NAIVE_SORT:
    case SPMSPV_K_COL_LB_SORT: {
      // boolean: the neighbours' row keys alone, sorted, then each distinct
      // row marked
      int* bk = reinterpret_cast<int*>(h->sb.keyA);
      if (slot == SPMSPV_K_COL_NAIVE_SORT)
        launch_naive_col(s, 2, h->csc_colptr, h->csc_row, nullptr, f, nullptr, h->ptr, h->n, 0,
                         b->cnt + cur, h->team_col, nullptr, nullptr, bk, nullptr);
      else
        launch_lb_gather(s, 2, h->ptr, h->xbeg, nullptr, h->split, h->csc_row, nullptr, h->ctl, 0,
                         b->cnt + cur, nullptr, nullptr, bk, nullptr, -1);
      SortBufs kb = h->sb;
      kb.valA = kb.valB = nullptr;
      const int fb = launch_radix_sort(s, kb, h->m, &h->ctl->bin_len, h->ctl, -1, h->nnz, false, Ep{0, 1},
                                       Gate{}, h->small_sort_cap);
      hipLaunchKernelGGL(k_mark_sorted, dim3(kBfsGrid), dim3(kBfsNT), 0, s, fb ? kb.keyB : kb.keyA,
                         &h->ctl->bin_len, b->visited, nbits);
      break;
    }
    case SPMSPV_K_SPMV_NAIVE:
      launch_row_naive(s, true, true, h->csr_row, h->csr_col, nullptr, nullptr, b->fbits[cur],
                       h->m, h->team_row, nullptr, nbits);
      break;
    default:  // 4, 5, 7 on a frontier of many edges: bottom-up
      if (h->nnz > 0) {
        // rows per thread and queue append: as many as leave every CU its workgroups
        const int rows = std::max(1, std::min(kBuRows, h->m / (kBfsNT * 1024)));
        const long long blocks = ((long long)h->m + (long long)kBfsNT * rows - 1) / (kBfsNT * rows);
        hipLaunchKernelGGL((k_bu_head<kBuBatch>), dim3((unsigned)std::min<long long>(kBfsGrid, blocks)),
                           dim3(kBfsNT), 0, s, h->csr_row, h->csr_col, h->m, rows, b->fbits[cur], b->visited,
                           nbits, b->queue, b->cnt + 3);
        hipLaunchKernelGGL((k_bu_tail<kBuBatch>), dim3(kBfsGrid), dim3(kBfsNT), 0, s, h->csr_row, h->csr_col,
                           b->fbits[cur], nbits, b->queue, b->cnt + 3);
      }
      break;
  }
  hipLaunchKernelGGL(k_bfs_collect, dim3(std::min(kBfsGrid, (words + kBfsNT - 1) / kBfsNT)), dim3(kBfsNT), 0, s,
                     nbits, b->fbits[cur], h->n, b->cnt, cur, b->visited, levels, nf);
  launch_prep(s, h->csc_colptr, nf, h->n, 0, b->cnt + nxt, h->ptr, h->xbeg, h->split, h->scan_state,
              h->tile_mm, h->ctl, &sel, Ep{0, 0}, h->prep_samp, false, LevelOpen{b->cnt, nxt, h->sig_dev + kSigBfs});
}

}  // namespace

namespace spmspv {
// BFS buffers (visited and frontier bit arrays, frontier lists, the
// bottom-up queue): sized by m and n, so allocated once per handle.
int bfs_alloc(spmspv_handle_t h) {
  if (h->bfs) return SPMSPV_SUCCESS;
  auto* b = new BfsState();
  const size_t n = h->n, m = h->m, words = (std::max(n, m) + 31) / 32 + 2;
  size_t off = 0;
  auto take = [&](size_t bytes) {
    const size_t o = off;
    off = (off + bytes + 255) / 256 * 256;
    return o;
  };
  const size_t o_vis = take(words * 4), o_fb0 = take(words * 4), o_fb1 = take(words * 4);
  const size_t o_f0 = take(n * 4 + 4), o_f1 = take(n * 4 + 4), o_cnt = take(64), o_r = take(64);
  // at most one item per row and one more per kBuChunk of its neighbours
  const size_t o_q = take((m + (size_t)h->nnz / kBuChunk + 64) * sizeof(int2));
  if (hipMalloc(&b->alloc, off) != hipSuccess) {
    delete b;
    return set_error(h, SPMSPV_OUT_OF_MEMORY, "bfs buffers");
  }
  char* p = static_cast<char*>(b->alloc);
  b->visited = reinterpret_cast<unsigned*>(p + o_vis);
  b->fbits[0] = reinterpret_cast<unsigned*>(p + o_fb0);
  b->fbits[1] = reinterpret_cast<unsigned*>(p + o_fb1);
  b->front[0] = reinterpret_cast<int*>(p + o_f0);
  b->front[1] = reinterpret_cast<int*>(p + o_f1);
  b->cnt = reinterpret_cast<int*>(p + o_cnt);
  b->reached = reinterpret_cast<unsigned long long*>(p + o_r);
  b->queue = reinterpret_cast<int2*>(p + o_q);
  if (!h->stream) {
    if (hipStreamCreateWithFlags(&b->own_stream, hipStreamNonBlocking) != hipSuccess) {
      (void)hipFree(b->alloc);
      delete b;
      return set_error(h, SPMSPV_DEVICE_ERROR, "bfs stream");
    }
  }
  h->bfs = b;
  return SPMSPV_SUCCESS;
}

// The captured level graphs hold the matrix, arena and row-tiling pointers
// and sizes they were captured with; every change of those drops them.
void bfs_drop_graphs(spmspv_handle_t h) {
  if (!h || !h->bfs) return;
  for (auto& g : h->bfs->graph)
    for (auto& e : g)
      if (e) {
        (void)hipGraphExecDestroy(e);
        e = nullptr;
      }
  h->bfs->levels_bound = nullptr;
}
}  // namespace spmspv

extern "C" {

int spmspv_bfs_release(spmspv_handle_t h) {
  if (!h || !h->bfs) return SPMSPV_SUCCESS;
  for (auto& g : h->bfs->graph)
    for (auto& e : g)
      if (e) (void)hipGraphExecDestroy(e);
  if (h->bfs->own_stream) (void)hipStreamDestroy(h->bfs->own_stream);
  if (h->bfs->alloc) (void)hipFree(h->bfs->alloc);
  delete h->bfs;
  h->bfs = nullptr;
  return SPMSPV_SUCCESS;
}

// The level loop; with max_levels > 0 it also records, per level (the
// frontier of level L is the one reached at level L-1), the device time of
// the level and the selector features of its frontier.
static int bfs_run(spmspv_handle_t h, int src, int* d_levels, int policy, int use_graphs,
                   double stats[4], int max_levels, float* level_ms, float* level_feat) {
  if (!h) return set_error(nullptr, SPMSPV_INVALID_ARGUMENT, "null handle");
  if (src < 0 || src >= h->n || !d_levels || policy < -1 || policy >= SPMSPV_NUM_SLOTS)
    return set_error(h, SPMSPV_INVALID_ARGUMENT, "bfs: bad source, levels or policy");
  if (h->m != h->n) return set_error(h, SPMSPV_INVALID_ARGUMENT, "bfs needs a square matrix");
  if (!h->csr_row) return set_error(h, SPMSPV_MAT_FORMAT_ERR, "bfs needs CSR input");
  int rc;
  if ((rc = ensure_arena(h)) || (rc = need_csc(h))) return rc;
  if ((rc = ensure_mat_features(h)) || (rc = bfs_alloc(h))) return rc;
  BfsState* b = h->bfs;
  // the frontiers' column scans overwrite the one made for the current x
  h->prep_valid = false;
  hipStream_t s = h->stream ? h->stream : b->own_stream;
  const int smode = policy >= 0 ? 2 : h->sel_mode, sfixed = policy >= 0 ? policy : h->sel_fixed;
  // the BFS levels' own weights when set (trained on BFS levels), else the
  // SpMSpV selector's
  const float* wsel = h->have_bfs_weights ? h->bfs_weights_dev : (h->have_weights ? h->weights_dev : nullptr);
  if (use_graphs && (b->levels_bound != d_levels || b->bound_mode != smode || b->bound_fixed != sfixed ||
                     b->bound_weights != wsel)) {
    bfs_drop_graphs(h);
    b->levels_bound = d_levels;
    b->bound_mode = smode;
    b->bound_fixed = sfixed;
    b->bound_weights = wsel;
  }
  // level L's kernels are enqueued on s, which the handle's own launches
  // (prep, sort) must share
  hipStream_t saved = h->stream;
  // the handle's null stream does not hold back the BFS's own one: what was
  // queued there (a product without a count, the caller's uploads) comes first.
  // On an idle stream the event would cost 14 us of a BFS of 471 (R-MAT s22).
  if (s != saved && hipStreamQuery(saved) != hipSuccess) {
    (void)hipGetLastError();  // not ready: no error
    HIP_TRY(h, hipEventRecord(h->ev0, saved));
    HIP_TRY(h, hipStreamWaitEvent(s, h->ev0, 0));
  }
  h->stream = s;
  SelectorArgs sel{wsel, h->mat, smode, sfixed};
  const auto t0 = std::chrono::steady_clock::now();
  hipLaunchKernelGGL(k_bfs_init, dim3(std::min(4096, (h->n + 255) / 256)), dim3(256), 0, s, d_levels,
                     h->n, b->visited, b->fbits[0], b->fbits[1], b->front[0], b->cnt, b->reached, src);
  // the level words: frontier size, choice and the level counter as tag
  long long* sw = h->sig + kSigBfs;
  __atomic_store_n(sw, kSigPending, __ATOMIC_RELEASE);
  launch_prep(s, h->csc_colptr, b->front[0], h->n, 0, b->cnt, h->ptr, h->xbeg, h->split,
              h->scan_state, h->tile_mm, h->ctl, &sel, next_ep(h, 1), h->prep_samp, false,
              LevelOpen{b->cnt, 0, h->sig_dev + kSigBfs});
  hipError_t e = hipGetLastError();
  const bool trace = max_levels > 0 && level_ms && level_feat;
  // waits for the word of level `tag` (polling; the trace's events need the
  // stream drained instead)
  long long word = 0;
  bool out_of_sequence = false;
  auto level_word = [&](int tag) -> hipError_t {
    if (trace) {
      hipError_t r = hipStreamSynchronize(s);
      if (r != hipSuccess) return r;
      word = __atomic_load_n(sw, __ATOMIC_ACQUIRE);
    } else if (wait_signal(h, kSigBfs, &word) != SPMSPV_SUCCESS) {
      return hipErrorUnknown;
    }
    if ((word >> 40) != tag) out_of_sequence = true;
    return out_of_sequence ? hipErrorUnknown : hipSuccess;
  };
  if (e == hipSuccess) e = level_word(0);
  int cur = 0, nlev = 1;
  while (e == hipSuccess && (int)(word & 0xffffffff) > 0) {
    int slot = policy >= 0 ? policy : (int)((word >> 32) & 0xff);
    if (slot < 0 || slot >= SPMSPV_NUM_SLOTS) slot = SPMSPV_K_COL_LB_ATOMIC;
    // selector feature 12: log2 of the frontier's part of the edges
    if (slot == SPMSPV_K_ROW_NAIVE || slot == SPMSPV_K_ROW_LB || slot == SPMSPV_K_SPMV_LB) {
      float part;
      __atomic_load(reinterpret_cast<float*>(sw + 1) + 12, &part, __ATOMIC_ACQUIRE);
      if (part <= -std::log2((float)kTopDown)) slot = SPMSPV_K_COL_LB_ATOMIC;
    }
    const int lev = nlev - 1;  // index of the level about to run
    if (trace && lev < max_levels) {
      std::memcpy(level_feat + 16 * lev, sw + 1, sizeof(float) * 16);
      (void)hipEventRecord(h->ev0, s);
    }
    __atomic_store_n(sw, kSigPending, __ATOMIC_RELEASE);
    if (use_graphs) {
      hipGraphExec_t& ge = b->graph[slot][cur];
      if (!ge) {
        hipGraph_t g = nullptr;
        e = hipStreamBeginCapture(s, hipStreamCaptureModeThreadLocal);
        if (e != hipSuccess) break;
        enqueue_level(h, s, slot, cur, d_levels, sel);
        e = hipStreamEndCapture(s, &g);
        if (e != hipSuccess) break;
        e = hipGraphInstantiate(&ge, g, nullptr, nullptr, 0);
        (void)hipGraphDestroy(g);
        if (e != hipSuccess) {
          ge = nullptr;
          break;
        }
      }
      e = hipGraphLaunch(ge, s);
    } else {
      enqueue_level(h, s, slot, cur, d_levels, sel);
      e = hipGetLastError();
    }
    if (trace && lev < max_levels && e == hipSuccess) e = hipEventRecord(h->ev1, s);
    if (e == hipSuccess) e = level_word(nlev);
    if (trace && lev < max_levels && e == hipSuccess) {
      float ms = 0.f;
      e = hipEventElapsedTime(&ms, h->ev0, h->ev1);
      level_ms[lev] = ms;
    }
    cur ^= 1;
    ++nlev;
    if (nlev > h->n + 1) break;  // cannot happen on a correct run; bounds the loop
  }
  const double secs = std::chrono::duration<double>(std::chrono::steady_clock::now() - t0).count();
  // device epochs advance 16 per level; clear the look-back states long
  // before (ctl->epoch + offset) could wrap onto a stale word
  h->dev_levels += nlev;
  if (h->dev_levels > 200000) {
    launch_fill_i32(s, reinterpret_cast<int*>(h->sb.dstate), (long long)h->sort_words * 2, 0);
    launch_fill_i32(s, reinterpret_cast<int*>(h->sb.red_state), (long long)h->red_words * 2, 0);
    launch_fill_i32(s, reinterpret_cast<int*>(h->scan_state), (long long)h->scan_words * 2, 0);
    h->dev_levels = 0;
  }
  unsigned long long red[2] = {0, 0};
  rc = SPMSPV_SUCCESS;
  if (!out_of_sequence && e == hipSuccess) {
    __atomic_store_n(sw, kSigPending, __ATOMIC_RELEASE);
    // 256 workgroups: three atomics each on one line
    hipLaunchKernelGGL(k_reached<1024>, dim3(std::min(256, (h->n + 1023) / 1024)), dim3(1024), 0, s, d_levels,
                       h->csc_colptr, h->n, b->reached, h->sig_dev + kSigBfs);
    e = hipGetLastError();
    if (e == hipSuccess) rc = wait_signal(h, kSigBfs, &word);
    for (int k = 0; k < 2; ++k) red[k] = (unsigned long long)__atomic_load_n(sw + 1 + k, __ATOMIC_ACQUIRE);
  }
  h->stream = saved;
  if (out_of_sequence) return set_error(h, SPMSPV_DEVICE_ERROR, "bfs: a level's word arrived out of sequence");
  if (e != hipSuccess) return set_error(h, SPMSPV_DEVICE_ERROR, std::string("bfs: ") + hipGetErrorString(e));
  if (rc) return rc;
  if (stats) {
    stats[0] = nlev - 1;             // levels with a nonempty frontier
    stats[1] = (double)red[1] / 2.0; // undirected edges in the reached component
    stats[2] = secs;
    stats[3] = (double)red[0];
  }
  return SPMSPV_SUCCESS;
}

int spmspv_bfs(spmspv_handle_t h, int src, int* d_levels, int policy, int use_graphs,
               double stats[4]) {
  return bfs_run(h, src, d_levels, policy, use_graphs, stats, 0, nullptr, nullptr);
}

int spmspv_bfs_trace(spmspv_handle_t h, int src, int* d_levels, int policy, int use_graphs,
                     double stats[4], int max_levels, float* level_ms, float* level_feat) {
  if (max_levels < 1 || !level_ms || !level_feat)
    return set_error(h, SPMSPV_INVALID_ARGUMENT, "bfs trace: need max_levels >= 1 and both arrays");
  return bfs_run(h, src, d_levels, policy, use_graphs, stats, max_levels, level_ms, level_feat);
}

}  // extern "C"
