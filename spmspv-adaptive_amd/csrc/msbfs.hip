// Multi-source BFS: up to 64 level-synchronous BFSs advanced together, one
// bit per source in a 64-bit word per vertex (visited set and frontier), so
// one pass over the edges of a level serves every source. The reference has
// no BFS; its harnesses replay one frontier per SpMSpV call
// (la/test/test_application.cu:240-415). Semiring: boolean OR-AND on the
// 64-bit words, integer arithmetic only.
//
// Per level, from the current frontier (dense words front[cur], and the same
// vertices as work items: (vertex, chunk of kMsChunk column entries)):
//   push (small frontiers): a team of lanes per work item ORs
//     front[cur][u] & ~visit[v] into front[nxt][v] for every v of its chunk of
//     column u (64-bit atomics);
//   pull (large frontiers): every row v not yet reached by all sources ORs
//     front[cur][u] over its neighbours u (CSR row v), stopping once every
//     source has reached v; a lane per row tests its first kMsHead
//     neighbours and overwrites front[nxt][v], rows left open are queued as
//     (row, chunk) items for teams;
// then a commit pass folds the new bits into visit, writes the levels of the
// new (vertex, source) pairs and lists the next frontier's work items. It
// walks all vertices, or after a push from few edges only the vertices that
// the push listed. The host picks the direction from the frontier's edge
// count (pull above nnz / 14), polls one word per level for the next
// frontier's size and stops when it is empty.
//
// What bounds it: device atomics on one address take 16 ns each, so lists are
// appended to once per workgroup round (a wave per append spent 120 us of
// each pull level at R-MAT s18 on the counter), the degree sums once per
// workgroup, and a push whose level will touch more than n / 64 edges lists
// nothing. A row or column longer than a chunk is shared by several teams (one
// team walking the 30,000 neighbours of s18's largest row took 1.3 ms). The
// levels of a vertex are written by the whole wave, nsrc adjacent words at
// once. R-MAT s18 (7.9 M nonzeros), 64 sources: 2,970 -> 440 us per call.
//
// Levels are written vertex-major: levels[v * nsrc + i] is the level of v
// in the BFS from srcs[i] (-1 unreached).
#include <algorithm>
#include <chrono>

#include "handle.hpp"

using namespace spmspv;

struct MsState {
  void* alloc = nullptr;
  unsigned long long* visit = nullptr;     // n
  unsigned long long* front[2] = {nullptr, nullptr};  // n each
  int2* list[2] = {nullptr, nullptr};      // frontier work items (vertex, chunk), items_cap each
  int2* queue = nullptr;                   // items_cap: pull items (row, chunk); push: touched vertices
  unsigned long long* cnt = nullptr;       // two groups of kMsGroup words (kMsItems, ...), then
                                           // [2 * kMsGroup] reached pairs, [+ 1] their edges, [+ 2] arrivals
};

namespace {

constexpr int kMsGrid = 2048;
constexpr int kMsNT = 256;
constexpr int kMsHead = 8;      // neighbours a lane tests in the pull head pass
constexpr int kMsTeam = 16;     // lanes per work item
constexpr int kMsChunk = 256;   // neighbours per work item
constexpr int kMsUnroll = 4;    // neighbours a lane has in flight
constexpr int kMsRows = 8;      // most rows per thread and list append
// words of a counter group
constexpr int kMsItems = 0, kMsQueue = 1, kMsDeg = 2, kMsGroup = 4;
// sources of a call, passed by value
struct MsSrcs {
  int v[64];
};

// Records the new (vertex, source) pairs of the wave's vertices (nw: this
// lane's vertex's new bits, 0: none). Convergent. The nsrc levels of one
// vertex are adjacent, so the lanes write them side by side: with few such
// vertices one vertex per step, else all (vertex, source) pairs of the wave
// 64 at a time.
__device__ __forceinline__ void write_levels(int v, unsigned long long nw, int nsrc, int level,
                                             int* __restrict__ levels) {
  uint64_t any = __ballot(nw != 0ull);
  if (__popcll(any) <= nsrc) {
    while (any) {
      const int l = __builtin_ctzll(any);
      any &= any - 1;
      const int vl = __shfl(v, l, kWave);
      const unsigned long long w = __shfl(nw, l, kWave);
      if ((w >> lane()) & 1ull) levels[(long long)vl * nsrc + lane()] = level;
    }
    return;
  }
  for (int k = lane(); k < kWave * nsrc; k += kWave) {
    const int l = k / nsrc, i = k - l * nsrc;
    const int vl = __shfl(v, l, kWave);
    const unsigned long long w = __shfl(nw, l, kWave);
    if ((w >> i) & 1ull) levels[(long long)vl * nsrc + i] = level;
  }
}

// Work items of a vertex with `deg` neighbours (at least one, so that a
// frontier of vertices without neighbours is not empty).
__device__ __forceinline__ int ms_chunks(int deg) { return max(1, (deg + kMsChunk - 1) / kMsChunk); }

// No vertex visited or in a frontier, all levels -1, the counters at 0.
__global__ void k_ms_init(int n, int nsrc, unsigned long long* visit, unsigned long long* f0,
                          unsigned long long* f1, int* levels, unsigned long long* cnt) {
  const long long stride = (long long)gridDim.x * blockDim.x;
  const long long t = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  for (long long v = t; v < n; v += stride) {
    visit[v] = 0ull;
    f0[v] = 0ull;
    f1[v] = 0ull;
  }
  for (long long k = t; k < (long long)n * nsrc; k += stride) levels[k] = -1;
  if (t < 2 * kMsGroup + 3) cnt[t] = 0ull;
}

__device__ void ms_signal(const unsigned long long* c, int tag, long long* sig) {
  // the degree sum first, acknowledged before the tagged word that the host polls
  __hip_atomic_store(sig + 1, (long long)c[kMsDeg], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  __hip_atomic_store(sig, ((long long)tag << 32) | (long long)c[kMsItems], __ATOMIC_RELAXED,
                     __HIP_MEMORY_SCOPE_SYSTEM);
}

// Bits and levels of the sources; their work items are the first frontier (a
// repeated source is listed once) and the sum of their degrees gives the first
// level's direction.
__global__ __launch_bounds__(kWave) void k_ms_sources(int nsrc, MsSrcs srcs, const int* __restrict__ colptr,
                                                      unsigned long long* visit, unsigned long long* f0,
                                                      int* levels, int2* list, long long* sig) {
  const int i = threadIdx.x;
  const int s = i < nsrc ? srcs.v[i] : 0;
  int deg = 0;
  bool first = i < nsrc;
  if (i < nsrc) {
    atomicOr(visit + s, 1ull << i);
    atomicOr(f0 + s, 1ull << i);
    levels[(long long)s * nsrc + i] = 0;
    deg = colptr[s + 1] - colptr[s];
    for (int j = 0; j < i; ++j) first = first && srcs.v[j] != s;
  }
  const int nc = first ? ms_chunks(deg) : 0;
  const int end = wave_incl_sum(nc);
  for (int k = 0; k < nc; ++k) list[end - nc + k] = make_int2(s, k);
  const unsigned long long d = wave_sum((unsigned long long)deg);
  if (i == kWave - 1) {
    const unsigned long long now[kMsGroup] = {(unsigned long long)end, 0ull, d, 0ull};
    ms_signal(now, 0, sig);
  }
}

// After a level: its counters to the host, the other group cleared for the
// next level (the host has read it).
__global__ void k_ms_signal(const unsigned long long* __restrict__ c, unsigned long long* other, int tag,
                            long long* sig) {
  for (int k = 0; k < kMsGroup; ++k) other[k] = 0ull;
  ms_signal(c, tag, sig);
}

// TOUCH: a vertex whose word was 0 is listed (the commit then walks the list).
template <bool TOUCH>
__global__ __launch_bounds__(kMsNT) void k_ms_push(const int* __restrict__ colptr, const int* __restrict__ crow,
                                                   const int2* __restrict__ items, long long nitems,
                                                   const unsigned long long* __restrict__ front,
                                                   const unsigned long long* __restrict__ visit,
                                                   unsigned long long* nfront, int2* touched,
                                                   unsigned long long* tcount) {
  const int tl = threadIdx.x & (kMsTeam - 1);
  const long long team = ((long long)blockIdx.x * blockDim.x + threadIdx.x) / kMsTeam;
  const long long nteams = (long long)gridDim.x * blockDim.x / kMsTeam;
  // whole waves iterate together (the append is convergent)
  const long long wbase = team - (team % (kWave / kMsTeam));
  for (long long t0 = wbase; t0 < nitems; t0 += nteams) {
    const long long t = t0 + (team - wbase);
    int b = 0, e = 0;
    unsigned long long fu = 0ull;
    if (t < nitems) {
      const int2 it = items[t];
      fu = front[it.x];
      b = colptr[it.x] + it.y * kMsChunk;
      e = min(b + kMsChunk, colptr[it.x + 1]);
    }
    // the longest item of the wave's teams bounds the wave's trips
    int len = max(e - b, 0);
#pragma unroll
    for (int o = kMsTeam; o < kWave; o <<= 1) len = max(len, __shfl_xor(len, o));
    for (int k0 = 0; k0 < len; k0 += kMsTeam * kMsUnroll) {
      int v[kMsUnroll];
      unsigned long long add[kMsUnroll];
#pragma unroll
      for (int j = 0; j < kMsUnroll; ++j) {
        const int k = b + k0 + j * kMsTeam + tl;
        v[j] = k < e ? crow[k] : -1;
      }
#pragma unroll
      for (int j = 0; j < kMsUnroll; ++j) add[j] = v[j] >= 0 ? fu & ~visit[v[j]] : 0ull;
#pragma unroll
      for (int j = 0; j < kMsUnroll; ++j) {
        unsigned long long old = ~0ull;
        if (add[j]) old = atomicOr(nfront + v[j], add[j]);
        if (TOUCH) {
          const bool first = old == 0ull;
          const uint64_t bal = __ballot(first);
          if (bal) {
            const int leader = __builtin_ctzll(bal);
            unsigned long long base = 0;
            if (lane() == leader) base = atomicAdd(tcount, (unsigned long long)__popcll(bal));
            base = __shfl(base, leader, kWave);
            const uint64_t lt = lane() == 0 ? 0ull : (~0ull >> (kWave - lane()));
            if (first) touched[base + __popcll(bal & lt)] = make_int2(v[j], 0);
          }
        }
      }
    }
  }
}

// New bits of every vertex (TOUCH: of the listed ones): nfront & ~visit into
// visit and nfront, the levels, and the next frontier's work items, one list
// append per workgroup and `rows` (<= kMsRows) vertices per thread.
template <bool TOUCH>
__global__ __launch_bounds__(kMsNT) void k_ms_commit(const int2* __restrict__ touched, int n, int rows,
                                                     const int* __restrict__ colptr, int nsrc, int level,
                                                     unsigned long long* visit, unsigned long long* nfront,
                                                     int* levels, int2* nlist, unsigned long long* c) {
  __shared__ int s_i[kMsNT / kWave];
  __shared__ long long s_l[kMsNT / kWave];
  __shared__ unsigned long long s_base;
  const long long total = TOUCH ? (long long)c[kMsQueue] : n;
  const long long step = (long long)kMsNT * rows;
  long long deg_sum = 0;
  for (long long b0 = (long long)blockIdx.x * step; b0 < total; b0 += (long long)gridDim.x * step) {
    int vv[kMsRows], nc[kMsRows];
    int mine = 0;
#pragma unroll
    for (int k = 0; k < kMsRows; ++k) {
      nc[k] = 0;
      vv[k] = 0;
      if (k >= rows) continue;
      const long long i = b0 + (long long)k * kMsNT + threadIdx.x;
      unsigned long long nw = 0ull;
      if (i < total) {
        vv[k] = TOUCH ? touched[i].x : (int)i;
        const unsigned long long f = nfront[vv[k]], vis = visit[vv[k]];
        nw = f & ~vis;
        if (nw != f) nfront[vv[k]] = nw;
        if (nw) {
          visit[vv[k]] = vis | nw;
          const int deg = colptr[vv[k] + 1] - colptr[vv[k]];
          deg_sum += deg;
          nc[k] = ms_chunks(deg);
          mine += nc[k];
        }
      }
      write_levels(vv[k], nw, nsrc, level, levels);
    }
    int tot;
    int pos = block_excl_sum<kMsNT, int>(mine, s_i, &tot);
    if (tot == 0) continue;  // the same in every thread
    if (threadIdx.x == 0) s_base = atomicAdd(c + kMsItems, (unsigned long long)tot);
    __syncthreads();
    const unsigned long long base = s_base;
    __syncthreads();
#pragma unroll
    for (int k = 0; k < kMsRows; ++k)
      for (int q = 0; q < nc[k]; ++q) nlist[base + pos++] = make_int2(vv[k], q);
  }
  deg_sum = block_sum<kMsNT, long long>(deg_sum, s_l);
  if (threadIdx.x == 0 && deg_sum) atomicAdd(c + kMsDeg, (unsigned long long)deg_sum);
}

// Every row's word of the next frontier: the OR over its first kMsHead
// neighbours (complete, or partial and queued), 0 for a row that all sources
// have reached. The commit masks it with visit.
__global__ __launch_bounds__(kMsNT) void k_ms_pull_head(const int* __restrict__ row_ptr, const int* __restrict__ col,
                                                        int m, int rows, unsigned long long full,
                                                        const unsigned long long* __restrict__ front,
                                                        const unsigned long long* __restrict__ visit,
                                                        unsigned long long* __restrict__ nfront, int2* queue,
                                                        unsigned long long* qcount) {
  __shared__ int s_i[kMsNT / kWave];
  __shared__ unsigned long long s_base;
  const long long step = (long long)kMsNT * rows;
  for (long long b0 = (long long)blockIdx.x * step; b0 < m; b0 += (long long)gridDim.x * step) {
    int nc[kMsRows];
    int mine = 0;
#pragma unroll
    for (int k = 0; k < kMsRows; ++k) {
      nc[k] = 0;
      if (k >= rows) continue;
      const long long r = b0 + (long long)k * kMsNT + threadIdx.x;
      const unsigned long long vis = r < m ? visit[r] : full;
      int b = 0, e = 0;
      if (vis != full) {
        b = row_ptr[r];
        e = row_ptr[r + 1];
      }
      unsigned long long acc = 0ull;
      if (b < e) {
        int u[kMsHead];
#pragma unroll
        for (int j = 0; j < kMsHead; ++j) u[j] = col[min(b + j, e - 1)];
#pragma unroll
        for (int j = 0; j < kMsHead; ++j) acc |= front[u[j]];  // a repeated last neighbour changes nothing
        if (e - b > kMsHead && (acc | vis) != full) nc[k] = ms_chunks(e - b - kMsHead);
        mine += nc[k];
      }
      if (r < m) nfront[r] = acc;
    }
    int tot;
    int pos = block_excl_sum<kMsNT, int>(mine, s_i, &tot);
    if (tot == 0) continue;  // the same in every thread
    if (threadIdx.x == 0) s_base = atomicAdd(qcount, (unsigned long long)tot);
    __syncthreads();
    const unsigned long long base = s_base;
    __syncthreads();
#pragma unroll
    for (int k = 0; k < kMsRows; ++k) {
      const int r = (int)(b0 + (long long)k * kMsNT + threadIdx.x);
      for (int q = 0; q < nc[k]; ++q) queue[base + pos++] = make_int2(r, q);
    }
  }
}

// The queued (row, chunk) items: a team ORs the chunk's neighbours, kMsTeam *
// kMsUnroll per step, until every source has reached the row.
__global__ __launch_bounds__(kMsNT) void k_ms_pull_tail(const int* __restrict__ row_ptr, const int* __restrict__ col,
                                                        unsigned long long full,
                                                        const unsigned long long* __restrict__ front,
                                                        const unsigned long long* __restrict__ visit,
                                                        unsigned long long* nfront, const int2* __restrict__ queue,
                                                        const unsigned long long* __restrict__ qcount) {
  const long long nq = (long long)*qcount;
  const int tl = threadIdx.x & (kMsTeam - 1);
  const long long team = ((long long)blockIdx.x * blockDim.x + threadIdx.x) / kMsTeam;
  const long long nteams = (long long)gridDim.x * blockDim.x / kMsTeam;
  const long long wbase = team - (team % (kWave / kMsTeam));
  for (long long t0 = wbase; t0 < nq; t0 += nteams) {
    const long long t = t0 + (team - wbase);
    int r = 0, b = 0, e = 0;
    unsigned long long vis = full, acc = 0ull, had = 0ull;
    if (t < nq) {
      const int2 it = queue[t];
      r = it.x;
      b = row_ptr[r] + kMsHead + it.y * kMsChunk;
      e = min(b + kMsChunk, row_ptr[r + 1]);
      vis = visit[r];
      // other chunks of the row may add to the word meanwhile
      had = acc = __hip_atomic_load(nfront + r, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    // wave-uniform trips: until every team's chunk ends or is full
    for (int k0 = b; __ballot(k0 < e && (acc | vis) != full) != 0ull; k0 += kMsTeam * kMsUnroll) {
      int u[kMsUnroll];
      const bool go = (acc | vis) != full;
#pragma unroll
      for (int j = 0; j < kMsUnroll; ++j) {
        const int k = k0 + j * kMsTeam + tl;
        u[j] = go && k < e ? col[k] : -1;
      }
#pragma unroll
      for (int j = 0; j < kMsUnroll; ++j)
        if (u[j] >= 0) acc |= front[u[j]];
      // the team's OR, so that every lane sees when all sources reached r
#pragma unroll
      for (int o = 1; o < kMsTeam; o <<= 1) acc |= __shfl_xor(acc, o);
    }
    if (tl == 0 && t < nq && (acc & ~had)) atomicOr(nfront + r, acc);
  }
}

// The words of the listed vertices to 0.
__global__ void k_ms_clear(const int2* __restrict__ items, long long nitems, unsigned long long* front) {
  for (long long k = (long long)blockIdx.x * blockDim.x + threadIdx.x; k < nitems;
       k += (long long)gridDim.x * blockDim.x)
    if (items[k].y == 0) front[items[k].x] = 0ull;
}

// Reached (vertex, source) pairs and the edges they span: sum over v of
// popcount(visit[v]) and popcount(visit[v]) * deg(v).
__global__ __launch_bounds__(kMsNT) void k_ms_reached(int n, const unsigned long long* __restrict__ visit,
                                                      const int* __restrict__ colptr, unsigned long long* out,
                                                      long long* sig) {
  __shared__ long long s_l[kMsNT / kWave];
  long long c = 0, d = 0;
  for (long long v = (long long)blockIdx.x * blockDim.x + threadIdx.x; v < n; v += (long long)gridDim.x * blockDim.x) {
    const long long p = __popcll(visit[v]);
    c += p;
    d += p * (colptr[v + 1] - colptr[v]);
  }
  c = block_sum<kMsNT, long long>(c, s_l);
  d = block_sum<kMsNT, long long>(d, s_l);
  if (threadIdx.x == 0) count_to_host((unsigned long long)c, (unsigned long long)d, out, sig);
}

}  // namespace

namespace spmspv {
int ms_alloc(spmspv_handle_t h) {
  if (h->ms) return SPMSPV_SUCCESS;
  auto* st = new MsState();
  const size_t n = h->n;
  size_t off = 0;
  auto take = [&](size_t bytes) {
    const size_t o = off;
    off = (off + bytes + 255) / 256 * 256;
    return o;
  };
  // a work item per vertex and one more per kMsChunk of its neighbours
  const size_t items = n + (size_t)h->nnz / kMsChunk + 64;
  const size_t ov = take(n * 8), of0 = take(n * 8), of1 = take(n * 8), ol0 = take(items * 8),
               ol1 = take(items * 8), ot = take(items * 8), oc = take(64 * 8);
  if (hipMalloc(&st->alloc, off) != hipSuccess) {
    delete st;
    return set_error(h, SPMSPV_OUT_OF_MEMORY, "multi-source BFS buffers");
  }
  char* p = static_cast<char*>(st->alloc);
  st->visit = reinterpret_cast<unsigned long long*>(p + ov);
  st->front[0] = reinterpret_cast<unsigned long long*>(p + of0);
  st->front[1] = reinterpret_cast<unsigned long long*>(p + of1);
  st->list[0] = reinterpret_cast<int2*>(p + ol0);
  st->list[1] = reinterpret_cast<int2*>(p + ol1);
  st->queue = reinterpret_cast<int2*>(p + ot);
  st->cnt = reinterpret_cast<unsigned long long*>(p + oc);
  h->ms = st;
  return SPMSPV_SUCCESS;
}

void ms_release(spmspv_handle_t h) {
  if (!h || !h->ms) return;
  if (h->ms->alloc) (void)hipFree(h->ms->alloc);
  delete h->ms;
  h->ms = nullptr;
}
}  // namespace spmspv

extern "C" {

int spmspv_bfs_multi(spmspv_handle_t h, int nsrc, const int* srcs, int* d_levels, double stats[4]) {
  if (!h) return set_error(nullptr, SPMSPV_INVALID_ARGUMENT, "null handle");
  if (nsrc < 1 || nsrc > 64 || !srcs || !d_levels)
    return set_error(h, SPMSPV_INVALID_ARGUMENT, "bfs_multi: 1..64 sources and a levels array are needed");
  if (h->m != h->n) return set_error(h, SPMSPV_INVALID_ARGUMENT, "bfs_multi needs a square matrix");
  if (!h->csr_row) return set_error(h, SPMSPV_MAT_FORMAT_ERR, "bfs_multi needs CSR input");
  for (int i = 0; i < nsrc; ++i)
    if (srcs[i] < 0 || srcs[i] >= h->n) return set_error(h, SPMSPV_INVALID_ARGUMENT, "bfs_multi: source out of range");
  int rc;
  if ((rc = ensure_arena(h)) || (rc = need_csc(h)) || (rc = ms_alloc(h))) return rc;
  MsState* st = h->ms;
  hipStream_t s = h->stream;
  const int n = h->n;
  const unsigned long long full = nsrc == 64 ? ~0ull : ((1ull << nsrc) - 1ull);
  const auto t0 = std::chrono::steady_clock::now();
  MsSrcs by_value{};
  std::copy(srcs, srcs + nsrc, by_value.v);
  auto blocks = [](long long threads, int most) {
    return dim3((unsigned)std::max<long long>(1, std::min<long long>(most, (threads + kMsNT - 1) / kMsNT)));
  };
  // vertices per thread and list append: as many as leave every CU its
  // workgroups (one append per 256 to 2,048 vertices)
  const int rows = std::max(1, std::min(kMsRows, n / (kMsNT * 1024)));
  const dim3 dense = blocks(((long long)n + rows - 1) / rows, kMsGrid);
  long long* sw = h->sig + kSigMs;
  auto pending = [&]() { __atomic_store_n(sw, kSigPending, __ATOMIC_RELEASE); };
  hipLaunchKernelGGL(k_ms_init, blocks(n, kMsGrid), dim3(kMsNT), 0, s, n, nsrc, st->visit, st->front[0],
                     st->front[1], d_levels, st->cnt);
  pending();
  hipLaunchKernelGGL(k_ms_sources, dim3(1), dim3(kWave), 0, s, nsrc, by_value, h->csc_colptr, st->visit, st->front[0],
                     d_levels, st->list[0], h->sig_dev + kSigMs);
  HIP_TRY(h, hipGetLastError());
  long long word = 0;
  if ((rc = wait_signal(h, kSigMs, &word))) return rc;
  long long items = word & 0xffffffffll, prev_items = 0;
  unsigned long long fdeg = (unsigned long long)__atomic_load_n(sw + 1, __ATOMIC_ACQUIRE);
  int cur = 0, level = 1, levels_run = 0;
  while (items > 0 && level <= n) {
    const int nxt = cur ^ 1;
    // counters of this level: group `nxt`, cleared by the previous level's signal
    unsigned long long* c = st->cnt + nxt * kMsGroup;
    // the frontier's edge count decides the direction (pull above nnz / 14)
    const bool pull = fdeg * 14ull > (unsigned long long)h->nnz;
    // a push from few edges lists the vertices it touches; from more, walking
    // all vertices costs less than the list's appends (16 ns each)
    const bool touch = !pull && fdeg < (unsigned long long)n / 64;
    if (pull) {
      hipLaunchKernelGGL(k_ms_pull_head, dense, dim3(kMsNT), 0, s, h->csr_row, h->csr_col, n, rows, full,
                         st->front[cur], st->visit, st->front[nxt], st->queue, c + kMsQueue);
      hipLaunchKernelGGL(k_ms_pull_tail, dim3(kMsGrid), dim3(kMsNT), 0, s, h->csr_row, h->csr_col, full,
                         st->front[cur], st->visit, st->front[nxt], st->queue, c + kMsQueue);
    } else {
      // the next frontier's words start at 0: the frontier of two levels ago
      // leaves by its list when that is short, else by a fill
      if (prev_items > n / 8)
        launch_fill_i32(s, reinterpret_cast<int*>(st->front[nxt]), 2ll * n, 0);
      else if (prev_items > 0)
        hipLaunchKernelGGL(k_ms_clear, blocks(prev_items, kMsGrid), dim3(kMsNT), 0, s, st->list[nxt], prev_items,
                           st->front[nxt]);
      if (touch)
        hipLaunchKernelGGL(k_ms_push<true>, blocks(items * kMsTeam, kMsGrid), dim3(kMsNT), 0, s, h->csc_colptr,
                           h->csc_row, st->list[cur], items, st->front[cur], st->visit, st->front[nxt], st->queue,
                           c + kMsQueue);
      else
        hipLaunchKernelGGL(k_ms_push<false>, blocks(items * kMsTeam, kMsGrid), dim3(kMsNT), 0, s, h->csc_colptr,
                           h->csc_row, st->list[cur], items, st->front[cur], st->visit, st->front[nxt], st->queue,
                           c + kMsQueue);
    }
    if (touch)
      hipLaunchKernelGGL(k_ms_commit<true>, blocks((long long)fdeg, kMsGrid), dim3(kMsNT), 0, s, st->queue, n, 1,
                         h->csc_colptr, nsrc, level, st->visit, st->front[nxt], d_levels, st->list[nxt], c);
    else
      hipLaunchKernelGGL(k_ms_commit<false>, dense, dim3(kMsNT), 0, s, st->queue, n, rows, h->csc_colptr, nsrc, level,
                         st->visit, st->front[nxt], d_levels, st->list[nxt], c);
    pending();
    hipLaunchKernelGGL(k_ms_signal, dim3(1), dim3(1), 0, s, c, st->cnt + cur * kMsGroup, level, h->sig_dev + kSigMs);
    HIP_TRY(h, hipGetLastError());
    if ((rc = wait_signal(h, kSigMs, &word))) return rc;
    if ((word >> 32) != level) return set_error(h, SPMSPV_DEVICE_ERROR, "bfs_multi: a level's word arrived out of sequence");
    prev_items = items;
    items = word & 0xffffffffll;
    fdeg = (unsigned long long)__atomic_load_n(sw + 1, __ATOMIC_ACQUIRE);
    cur = nxt;
    ++level;
    ++levels_run;
  }
  const double secs = std::chrono::duration<double>(std::chrono::steady_clock::now() - t0).count();
  // 256 workgroups: three atomics each on one line
  pending();
  hipLaunchKernelGGL(k_ms_reached, blocks(n, 256), dim3(kMsNT), 0, s, n, st->visit, h->csc_colptr,
                     st->cnt + 2 * kMsGroup, h->sig_dev + kSigMs);
  HIP_TRY(h, hipGetLastError());
  if ((rc = wait_signal(h, kSigMs, &word))) return rc;
  unsigned long long hc[2];
  for (int k = 0; k < 2; ++k) hc[k] = (unsigned long long)__atomic_load_n(sw + 1 + k, __ATOMIC_ACQUIRE);
  if (stats) {
    stats[0] = levels_run;              // levels with a nonempty frontier
    stats[1] = (double)hc[1] / 2.0;     // undirected edges summed over the sources' components
    stats[2] = secs;
    stats[3] = (double)hc[0];           // reached (vertex, source) pairs
  }
  return SPMSPV_SUCCESS;
}

}  // extern "C"
