// A column SpMSpV in one launch for a small x: at most kFuseKeys keys whose
// products fit kFuseCap. The column scan of x (as k_prep's single tile,
// including the merge-path splits, so a call that does not fit continues with
// the usual launches), the products, their row sums and the sorted output
// with its count.
//
// Every workgroup owns a range of rows. It scans x (a few thousand column
// bounds at most) and loads the row of every product, which is cheaper than
// handing rows between workgroups, then takes the products of its rows alone:
// their rows as bits of an LDS bit array, whose prefix counts number the hit
// rows in order; each row's sum in 64-bit fixed point under that number
// (fixed_sum.hpp: exact, so the result does not depend on the order); rows and
// sums leave sorted, at the offset that a look-back over the workgroups
// gives. No sort: sorting the products in the LDS of one workgroup (three
// ranking passes on one CU) took 50 us for 10,480 products on 65,536 rows
// where this takes 20 us (calls: 55 -> 27 us; 512 products 24.6 -> 20.7); bound
// by the chain of dependent round trips (keys, column bounds, rows, values,
// look-back).
//
// In auto mode a call that fits skips the network (a size rule in front of
// it: no slot reads less than the products of x) and is reported as
// kFusedSlot, the sort-based slot, whose result (rows in order, the same on
// every run) it computes; one that does not fit runs the selector as k_prep
// does, and where an atomic column slot is chosen, gathers its products into
// acc and marks right away: every workgroup has the column bounds in LDS and
// runs the selector in one wave while the others load their first products, so
// only the compaction is left to launch. The gather as a launch of its own
// (and the launch gap) took 11 us for 49,297 products of R-MAT scale 20 (1,049
// keys, call 37.5 us -> 30.8; 115,997 products 48.8 -> 40.9; 15,999 products
// of 65,536 rows 29.0 -> 28.1). The workgroup that finishes last sets the done flag in
// ctl->kernel_choice (which shuts every gated launch queued behind), writes
// the count to ctl->ynnz, then to *count_sig and the selector word (flagged
// kSelDone, count in the bin_len field).
#include <climits>

#include "fixed_sum.hpp"
#include "kernels.hpp"
#include "selector.hpp"

namespace spmspv {

namespace {

// rows of a workgroup: at least kFuseRowsMin on up to kFuseGrid workgroups (8,
// 16, 32 and 64 of them differ by at most 1 us on 65,536 and 10^6 rows; every
// one of them reads all the products' rows), and at most what the bit array
// holds
constexpr int kFuseRowsMin = 8192, kFuseGrid = 32, kFuseRows = 131072;

// Workgroups at least when the launch may gather: 32 of them took 36.3 us for
// the 49,297 products above, 64 to 256 of them 32.4 to 32.9 us; 115,997
// products 42.7, 43.9, 42.4 and 44.8 us with 64, 96, 128 and 256 of them (the
// gather's loads still behind the selector). Up to kFuseGather products per
// workgroup it is faster than the gather launch: 466 k products 51.2 -> 42.5,
// 400 k of 3,000 keys 94.0 -> 81.7 us.
constexpr int kGatherGrid = 128;
constexpr int kNaiveAtomicSlot = 0, kLbAtomicSlot = 2;  // SPMSPV_K_COL_NAIVE_ATOMIC, SPMSPV_K_COL_LB_ATOMIC

// One workgroup of 1,024 threads per CU (the sums of kFuseCap rows and the
// bit array fill its LDS); KPT keys and IPT products per thread.
template <int NT, int KPT, int IPT>
__global__ __launch_bounds__(NT) void k_col_fused(const int* __restrict__ colptr, const int* __restrict__ crow,
                                                  const float* __restrict__ cval, const int* __restrict__ xkey,
                                                  const float* __restrict__ xval, int ncols, int xnnz, int m,
                                                  int rows, int nranges, int* __restrict__ ptr, int* __restrict__ xbeg,
                                                  int* __restrict__ split, Ctl* ctl, SelectorArgs sel,
                                                  int* __restrict__ ykey, float* __restrict__ yval,
                                                  long long* count_sig, int cap, unsigned long long* state, Ep ep,
                                                  float* acc, unsigned char* marks) {
  constexpr int NW = NT / kWave, CAP = NT * IPT, KEYS = NT * KPT;
  static_assert(CAP < (1 << 14), "fixed-point sums of a row's products; 16-bit prefix counts");
  static_assert(KEYS < 65536, "16-bit x entries");
  constexpr int WORDS = kFuseRows / 32, WPT = WORDS / NT;
  // the column scan and the product -> x entry map (or, when the products do
  // not fit, the selector's weights), then the sums
  struct Scan {
    int ptr[KEYS + 4];
    int beg[KEYS];
    union {
      unsigned short seg[CAP];
      float w[kNWeights];
    };
  };
  struct Sums {
    unsigned long long q[CAP];
    unsigned e[CAP];
  };
  union Raw {
    Scan scan;
    Sums sums;
  };
  __shared__ __align__(16) Raw s;
  __shared__ unsigned s_bits[WORDS];
  __shared__ unsigned short s_pfx[WORDS];
  __shared__ long long s_l[NW];
  __shared__ int s_i[NW], s_mn[NW];
  __shared__ unsigned long long s_pre;
  __shared__ MatFeat s_mf;
  __shared__ Ctl s_ctl;  // the selector's outputs
  const bool first = blockIdx.x == 0;
  // the selector's weights and matrix features, loaded beside the column
  // scan (stored to LDS only when the products do not fit)
  constexpr int kWPT = (kNWeights + NT - 1) / NT;
  constexpr int kMF = sizeof(MatFeat) / sizeof(double);
  float wr[kWPT];
  double mfr = 0.0;
  if ((first || acc) && sel.mode != 2 && sel.mat) {
    if (sel.weights) {
#pragma unroll
      for (int i = 0; i < kWPT; ++i) {
        const int idx = threadIdx.x + i * NT;
        wr[i] = idx < kNWeights ? sel.weights[idx] : 0.f;
      }
    }
    if (threadIdx.x < kMF) mfr = reinterpret_cast<const double*>(sel.mat)[threadIdx.x];
  }
  // ---- column scan of x
  const int base = threadIdx.x * KPT;
  int c[KPT], beg[KPT], len[KPT];
#pragma unroll
  for (int j = 0; j < KPT; ++j) c[j] = xnnz > 0 ? xkey[base + j < xnnz ? base + j : xnnz - 1] : 0;
#pragma unroll
  for (int j = 0; j < KPT; ++j) {
    const int ok = (base + j < xnnz && (unsigned)c[j] < (unsigned)ncols) ? 1 : 0;
    const int ci = c[j] & -ok;
    beg[j] = colptr[ci];
    len[j] = colptr[ci + ok];
    c[j] = ok;
  }
#pragma unroll
  for (int k = 0; k < WPT; ++k) s_bits[k * NT + threadIdx.x] = 0u;
  long long tsum = 0;
  int mx = 0, mn = INT_MAX;
#pragma unroll
  for (int j = 0; j < KPT; ++j) {
    len[j] = c[j] ? len[j] - beg[j] : 0;
    beg[j] = c[j] ? beg[j] : 0;
    if (c[j]) {
      mx = max(mx, len[j]);
      mn = min(mn, len[j]);
    }
    tsum += len[j];
  }
  // sum, longest and shortest column over the workgroup with one barrier
  long long bl = 0, run;
  {
    long long inc = tsum;
#pragma unroll
    for (int o = 1; o < kWave; o <<= 1) {
      const long long u = __shfl_up(inc, o);
      if (lane() >= o) inc += u;
      mx = max(mx, __shfl_xor(mx, o));
      mn = min(mn, __shfl_xor(mn, o));
    }
    const int w = threadIdx.x / kWave;
    if (lane() == kWave - 1) {
      s_l[w] = inc;
      s_i[w] = mx;
      s_mn[w] = mn;
    }
    __syncthreads();
    run = inc - tsum;
#pragma unroll
    for (int k = 0; k < NW; ++k) {
      const long long u = s_l[k];
      if (k < w) run += u;
      bl += u;
      mx = max(mx, s_i[k]);
      mn = min(mn, s_mn[k]);
    }
  }
#pragma unroll
  for (int j = 0; j < KPT; ++j) {
    const int i = base + j;
    if (i < xnnz) {
      s.scan.ptr[i] = (int)run;
      s.scan.beg[i] = beg[j];
      if (first) {
        ptr[i] = (int)run;
        xbeg[i] = beg[j];
        if (split) {
          const long long Mi = i + run;
          const long long Mn = Mi + len[j] + 1;
          for (long long d = (Mi / kLbTile + 1) * kLbTile; d <= Mn; d += kLbTile) split[d / kLbTile] = i + 1;
        }
      }
      run += len[j];
    }
  }
  if (threadIdx.x == 0) {
    s.scan.ptr[xnnz] = (int)bl;
    if (first) {
      ptr[xnnz] = (int)bl;
      ctl->bin_len = bl;
      ctl->max_len = xnnz > 0 ? mx : 0;
      ctl->min_len = mn;
      ctl->xnnz = xnnz;
      const long long nt = ((long long)xnnz + bl + kLbTile - 1) / kLbTile;
      ctl->n_tiles = nt;
      if (split) {
        split[0] = 0;
        split[nt] = xnnz;
      }
    }
  }
  const bool fuse = bl <= CAP && bl <= cap && ykey != nullptr && yval != nullptr;
  if (!fuse) {
    const bool small = acc && bl <= (long long)gridDim.x * kFuseGather;
    if (!first && !small) return;
    const bool net = sel.mode != 2 && sel.mat;
    __syncthreads();  // the scan is complete
    if (net) {
      if (sel.weights) {
#pragma unroll
        for (int i = 0; i < kWPT; ++i) {
          const int idx = threadIdx.x + i * NT;
          if (idx < kNWeights) s.scan.w[wlds_index(idx)] = wr[i];
        }
      }
      if (threadIdx.x < kMF) reinterpret_cast<double*>(&s_mf)[threadIdx.x] = mfr;
      __syncthreads();
    }
    // Wave 0 runs the selector, as the last tile of k_prep does. The other
    // waves take an equal share of the products, a few per thread and round;
    // the first round is loaded beside the selector and dropped when another
    // slot is chosen.
    constexpr int GPT = 2, GNT = NT - kWave;
    const int n = small ? (int)bl : 0, step = (int)gridDim.x * GNT;
    int p0 = threadIdx.x < kWave ? n : (int)blockIdx.x * GNT + (int)threadIdx.x - kWave;
    int r[GPT];
    float v[GPT];
    const auto load = [&]() {
      int e[GPT];
#pragma unroll
      for (int j = 0; j < GPT; ++j) {
        const int p = min(p0 + j * step, n - 1);
        int lo = 0, hi = xnnz;  // ptr[lo] <= p < ptr[hi]
        while (hi - lo > 1) {
          const int mid = (lo + hi) >> 1;
          if (s.scan.ptr[mid] <= p) lo = mid;
          else hi = mid;
        }
        e[j] = lo;
        r[j] = s.scan.beg[lo] + (p - s.scan.ptr[lo]);
      }
#pragma unroll
      for (int j = 0; j < GPT; ++j) {
        v[j] = cval[r[j]] * xval[e[j]];
        r[j] = crow[r[j]];
      }
    };
    if (p0 < n) load();
    int choice = sel.mode == 2 ? sel.fixed : -1;
    if (net) {
      SelectorArgs sl = sel;
      if (sel.weights) sl.weights = s.scan.w;
      sl.mat = &s_mf;
      select_in_wave(&s_ctl, sl, (double)xnnz, (double)bl, (double)(xnnz > 0 ? mx : 0));
      __syncthreads();
      choice = s_ctl.kernel_choice;
      if (first && threadIdx.x < kF) ctl->feat[threadIdx.x] = s_ctl.feat[threadIdx.x];
    }
    const bool gather = small && (choice == kNaiveAtomicSlot || choice == kLbAtomicSlot);
    if (first && threadIdx.x == 0) {
      if (choice >= 0) ctl->kernel_choice = choice | (gather ? kSelGathered : 0);
      if (sel.stash) *sel.stash = sel_word(bl, gather ? choice | kSelGathered : choice);
    }
    if (!gather) return;
    while (p0 < n) {
#pragma unroll
      for (int j = 0; j < GPT; ++j) {
        if (p0 + j * step < n) {
          atomic_add_f32(acc + r[j], v[j]);
          marks[r[j]] = 1;
        }
      }
      p0 += GPT * step;
      if (p0 < n) load();
    }
    return;
  }
  if ((int)blockIdx.x >= nranges) return;  // only there for a gather
  __syncthreads();  // the scan is complete
  // products per thread for this call (<= IPT)
  const int ie = (int)((bl + NT - 1) / NT);
  // ---- product -> x entry map, merge-path style: thread t fills products
  // t*ie .. t*ie+ie-1 from one search and a forward walk (x entries with
  // empty columns are stepped over)
  {
    const int p0 = threadIdx.x * ie;
    if (p0 < bl) {
      int lo = 0, hi = xnnz;  // ptr[lo] <= p0 < ptr[hi]
      while (hi - lo > 1) {
        const int mid = (lo + hi) >> 1;
        if (s.scan.ptr[mid] <= p0) lo = mid;
        else hi = mid;
      }
      int e = lo, nxt = s.scan.ptr[lo + 1];
#pragma unroll
      for (int k = 0; k < IPT; ++k) {
        const int p = p0 + k;
        if (k < ie && p < bl) {
          while (nxt <= p) nxt = s.scan.ptr[++e + 1];
          s.scan.seg[p] = (unsigned short)e;
        }
      }
    }
  }
  __syncthreads();
  // ---- rows of all products, the values of this workgroup's
  const int lo_row = (int)blockIdx.x * rows;
  const unsigned nrows = (unsigned)min(rows, m - lo_row);
  int pos[IPT], row[IPT];
  float val[IPT];
  bool mine[IPT];
#pragma unroll
  for (int j = 0; j < IPT; ++j) {
    const int p = j * NT + threadIdx.x;
    const bool ok = j < ie && p < bl;
    const int e = ok ? s.scan.seg[p] : 0;
    pos[j] = ok ? s.scan.beg[e] + (p - s.scan.ptr[e]) : 0;
    val[j] = ok ? xval[e] : 0.f;
    row[j] = ok ? crow[pos[j]] : -1;
  }
#pragma unroll
  for (int j = 0; j < IPT; ++j) {
    row[j] -= lo_row;
    mine[j] = j < ie && (unsigned)row[j] < nrows && j * NT + (int)threadIdx.x < bl;
    if (mine[j]) {
      val[j] *= cval[pos[j]];
      atomicOr(&s_bits[row[j] >> 5], 1u << (row[j] & 31));
    }
  }
  __syncthreads();
  // ---- hit rows numbered in order
  unsigned wb[WPT];
  int cnt = 0;
#pragma unroll
  for (int k = 0; k < WPT; ++k) {
    wb[k] = s_bits[threadIdx.x * WPT + k];
    cnt += __popc(wb[k]);
  }
  int tot;
  int at = block_excl_sum<NT, int>(cnt, s_i, &tot);
  // this workgroup's count goes out before its sums: the others' look-back
  // finds it
  const unsigned epoch = ep_of(ctl, ep);
  if (threadIdx.x == 0) st_relaxed(&state[blockIdx.x], pack_state(first ? 2 : 1, epoch, (unsigned long long)tot));
  const int at0 = at;
#pragma unroll
  for (int k = 0; k < WPT; ++k) {
    s_pfx[threadIdx.x * WPT + k] = (unsigned short)at;
    at += __popc(wb[k]);
  }
  for (int u = threadIdx.x; u < tot; u += NT) {
    s.sums.q[u] = 0ull;
    s.sums.e[u] = 0u;
  }
  __syncthreads();
  // ---- exact row sums; a row with an Inf or NaN among its products (exponent
  // 0xFF, known to all once the maxima are in) collects which of the two
  // infinities and NaN it holds, which is all that its sum depends on
  int num[IPT];
#pragma unroll
  for (int j = 0; j < IPT; ++j) {
    num[j] = 0;
    if (mine[j]) {
      const int wd = row[j] >> 5;
      num[j] = s_pfx[wd] + __popc(s_bits[wd] & ((1u << (row[j] & 31)) - 1u));
      atomicMax(&s.sums.e[num[j]], prod_ef(val[j]));
    }
  }
  __syncthreads();
#pragma unroll
  for (int j = 0; j < IPT; ++j) {
    if (mine[j]) {
      const unsigned E = s.sums.e[num[j]];
      if (E == 0xFFu) atomicOr(&s.sums.q[num[j]], (unsigned long long)special_kind(val[j]));
      else atomicAdd(&s.sums.q[num[j]], (unsigned long long)prod_fixed(val[j], E));
    }
  }
  __syncthreads();
  const long long pre = (long long)tile_prefix(state, blockIdx.x, epoch, (unsigned long long)tot, &s_pre);
  // ---- sorted output, device-coherent (visible once acknowledged)
  for (int u = threadIdx.x; u < tot; u += NT) {
    const float v = s.sums.e[u] == 0xFFu ? special_value((unsigned)s.sums.q[u])
                                         : fixed_value((long long)s.sums.q[u], s.sums.e[u]);
    __hip_atomic_store(yval + pre + u, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
  {
    long long o = pre + at0;
#pragma unroll
    for (int k = 0; k < WPT; ++k) {
      unsigned b = wb[k];
      while (b) {
        const int r = ((int)(threadIdx.x * WPT + k) << 5) + __ffs(b) - 1;
        b &= b - 1;
        __hip_atomic_store(ykey + o, lo_row + r, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        ++o;
      }
    }
  }
  // ---- the last workgroup publishes: one 64-bit atomic per workgroup, an
  // arrival in the high half and, from the last row range, the count in the
  // low half (as k_compact)
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  __syncthreads();
  if (threadIdx.x == 0) {
    const unsigned long long count = (unsigned long long)(pre + tot);
    auto* word = reinterpret_cast<unsigned long long*>(&ctl->done[kSlotCount]);
    const unsigned long long in = (1ull << 32) | ((int)blockIdx.x == nranges - 1 ? count : 0ull);
    const unsigned long long now =
        __hip_atomic_fetch_add(word, in, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) + in;
    if ((int)(now >> 32) == nranges) {
      __hip_atomic_store(word, 0ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      const long long total = (long long)(unsigned)now;
      const int choice = sel.mode == 2 ? sel.fixed : kFusedSlot;
      ctl->ynnz = (int)total;
      ctl->sort_small = 1;
      ctl->kernel_choice = choice | kSelDone;
      // the outputs are device-coherent and acknowledged: no L2 write-back
      // before the words
      if (count_sig) *count_sig = total;
      if (sel.stash) *sel.stash = sel_word(total, choice | kSelDone);
    }
  }
}

}  // namespace

bool launch_col_fused(hipStream_t s, const int* colptr, const int* crow, const float* cval, const int* xkey,
                      const float* xval, int ncols, int xnnz, int m, int* ptr, int* xbeg, int* split, Ctl* ctl,
                      const SelectorArgs& sel, int* ykey, float* yval, long long* count_sig, int cap,
                      unsigned long long* state, Ep ep, float* acc, unsigned char* marks) {
  if (xnnz > kFuseKeys || m > kFuseRowsMax) return false;
  const int grid = std::max(std::min(kFuseGrid, (m + kFuseRowsMin - 1) / kFuseRowsMin), (m + kFuseRows - 1) / kFuseRows);
  const int rows = (m + grid - 1) / grid, ranges = (m + rows - 1) / rows;
  hipLaunchKernelGGL((k_col_fused<kFuseNT, kFuseKeys / kFuseNT, kFuseCap / kFuseNT>), dim3(acc ? std::max(ranges, kGatherGrid) : ranges),
                     dim3(kFuseNT), 0, s, colptr, crow, cval, xkey, xval, ncols, xnnz, m, rows, ranges, ptr, xbeg, split, ctl,
                     sel, ykey, yval, count_sig, cap, state, ep, acc, marks);
  return true;
}

}  // namespace spmspv
