// CSR5-style SpMV / masked SpMSpV for 64-lane wavefronts (the spmv_type 1
// path of K5/K7; the reference's csr5_spmv_cuda.h:440-582 and
// csr5_spmspv.h:449-610 with CSR5Preprocess, spmspv.h:1425-1582, built for
// 32-lane warps). The format is re-derived for wave64:
//   * a tile is 64 lanes x S items (S = sigma in {8, 16, 24, 32}); lane l
//     owns the tile's items l*S .. l*S+S-1 in CSR order, stored in groups
//     of four (item i of lane l at tile*64*S + (i/4)*256 + l*4 + i%4) so
//     that every four item steps are one 16-byte load per lane, 1 KB per
//     wave side by side;
//   * the descriptor is one 32-bit word per lane: bit i marks a row start
//     at item i (bit 0 of lane 0 always marks the tile start). Marker
//     offsets (the reference's y_offset) come from a DPP prefix sum of the
//     popcounts and the cross-lane segmented sum (its seg_offset) from a
//     DPP segmented scan, so neither is stored;
//   * tile_info[t] = index, in the list of non-empty rows, of the row that
//     holds the tile's first item, with bit 31 set when that item continues
//     a row from the previous tile. The k-th marker of tile t is non-empty
//     row rows_ne[base + k], which replaces the reference's per-tile
//     empty_offset arrays; empty rows are written from their own list;
//   * the copy's columns are renumbered by nonzero count and every row's
//     items stored in that order, so that the densest columns come first.
// One wave per tile, no barrier inside the tile loop; each wave walks tiles
// w, w + waves, ... with the next tile's loads in flight (column indices
// and values two tiles ahead, x gathered one tile ahead). The only LDS use
// is a copy of the first x entries (the densest columns), made by each block
// at its start: one block per CU then serves most gathers from LDS.
#include <algorithm>
#include <climits>

#include "handle.hpp"
#include "ranking.hpp"

namespace spmspv {

namespace {

// columns (after renumbering, the ones with the most nonzeros) whose x
// entries the tile kernel keeps in LDS: all 160 KB of a CU's LDS, shared by
// one block per CU that holds as many waves as the registers allow. At R-MAT
// s20 they take 72 % of the nonzeros, and the distinct cache lines per
// wave-wide gather fall to under a third.
constexpr int kCsr5Hot = 40960;
// threads per block of the tile kernel: 256 without the LDS copy; with it,
// all the waves a CU can hold at the register use of each width (168
// registers at S = 24: 3 waves per SIMD; 241 at S = 32: 2; <= 128 below: 4)
constexpr int csr5_nt(int S, int HOT) { return HOT == 0 ? 256 : S >= 32 ? 512 : S >= 24 ? 768 : 1024; }
static_assert(kCsr5Hot * 4 <= 160 * 1024, "LDS of one CU");

// ---- preprocessing --------------------------------------------------------
constexpr int kScanPart = 2048;

__global__ __launch_bounds__(256) void k_nonempty_part(const int* __restrict__ row_ptr, int m,
                                                       int* __restrict__ sums) {
  __shared__ int lds[4];
  const long long base = (long long)blockIdx.x * kScanPart;
  int v = 0;
#pragma unroll
  for (int k = 0; k < kScanPart / 256; ++k) {
    const long long r = base + k * 256 + threadIdx.x;
    if (r < m) v += row_ptr[r + 1] > row_ptr[r];
  }
  v = block_sum<256>(v, lds);
  if (threadIdx.x == 0) sums[blockIdx.x] = v;
}

// exclusive scan of the part sums in one workgroup; sums[nparts] = total
__global__ __launch_bounds__(256) void k_scan_parts(int* sums, int nparts) {
  __shared__ int lds[4];
  int run = 0;
  for (int c = 0; c < nparts; c += 256) {
    const int i = c + threadIdx.x;
    const int v = i < nparts ? sums[i] : 0;
    int tot;
    const int ex = block_excl_sum<256>(v, lds, &tot);
    if (i < nparts) sums[i] = run + ex;
    run += tot;
  }
  if (threadIdx.x == 0) sums[nparts] = run;
}

// rank[r] = non-empty rows before r; rows_ne / rows_empty lists (ascending)
__global__ __launch_bounds__(256) void k_rank_rows(const int* __restrict__ row_ptr, int m,
                                                   const int* __restrict__ sums, int* __restrict__ rank,
                                                   int* __restrict__ rows_ne, int* __restrict__ rows_empty) {
  __shared__ int lds[4];
  constexpr int PT = kScanPart / 256;
  const long long base = (long long)blockIdx.x * kScanPart + (long long)threadIdx.x * PT;
  int f[PT];
  int loc = 0;
#pragma unroll
  for (int k = 0; k < PT; ++k) {
    const long long r = base + k;
    f[k] = r < m ? (row_ptr[r + 1] > row_ptr[r]) : 0;
    loc += f[k];
  }
  int tot;
  int run = sums[blockIdx.x] + block_excl_sum<256>(loc, lds, &tot);
#pragma unroll
  for (int k = 0; k < PT; ++k) {
    const long long r = base + k;
    if (r < m) {
      rank[r] = run;
      if (f[k]) rows_ne[run] = (int)r;
      else rows_empty[r - run] = (int)r;
    }
    run += f[k];
  }
}

// tile_info and the tile-start marker of every tile
__global__ void k_tile_info(const int* __restrict__ row_ptr, const int* __restrict__ rank, int m,
                            int nnz, int T, int ntiles, int n_ne, unsigned* __restrict__ tinfo,
                            unsigned* __restrict__ flags) {
  const int t = blockIdx.x * blockDim.x + threadIdx.x;
  if (t > ntiles) return;
  const long long j0 = (long long)t * T;
  if (j0 >= nnz) {
    tinfo[t] = (unsigned)n_ne;  // past the data: a "real start" sentinel
    return;
  }
  // the row holding item j0: first r with row_ptr[r + 1] > j0
  int lo = 0, hi = m - 1;
  while (lo < hi) {
    const int mid = (lo + hi) >> 1;
    if (row_ptr[mid + 1] > j0) hi = mid;
    else lo = mid + 1;
  }
  const bool cont = row_ptr[lo] < j0;
  tinfo[t] = (unsigned)rank[lo] | (cont ? 0x80000000u : 0u);
  flags[(size_t)t * kWave] |= 1u;  // only this thread touches lane 0 here
}

// row-start markers (one-time preprocessing, atomics are fine)
__global__ void k_row_markers(const int* __restrict__ row_ptr, int m, int T, int S,
                              unsigned* __restrict__ flags) {
  for (long long r = (long long)blockIdx.x * blockDim.x + threadIdx.x; r < m;
       r += (long long)gridDim.x * blockDim.x) {
    const int j = row_ptr[r];
    if (row_ptr[r + 1] <= j) continue;
    const int t = j / T, o = j % T;
    atomicOr(flags + (size_t)t * kWave + o / S, 1u << (o % S));
  }
}

// The copy of a matrix whose columns keep their order.
__global__ void k_csr5_transpose(const int* __restrict__ col, const float* __restrict__ val, int nnz,
                                 int T, int S, long long total, int* __restrict__ ccol,
                                 float* __restrict__ cval) {
  for (long long q = (long long)blockIdx.x * blockDim.x + threadIdx.x; q < total;
       q += (long long)gridDim.x * blockDim.x) {
    // position o of a tile holds item i of lane l with o = (i / 4) * 256 +
    // l * 4 + i % 4: each lane's items come in 16-byte groups of four, one
    // vector load per group, a wave's load 1 KB side by side
    const long long t = q / T;
    const int o = (int)(q - t * T);
    const int g = o >> 8, r = o & 255;
    const int l = r >> 2, i = g * 4 + (r & 3);
    const long long src = t * T + (long long)l * S + i;
    const bool ok = src < nnz;
    ccol[q] = ok ? col[src] : 0;
    cval[q] = ok ? val[src] : 0.f;
  }
}

// ---- SpMV / masked SpMSpV ---------------------------------------------------
// HOT > 0: the first `hot` (<= HOT) entries of x, the columns with the most
// nonzeros once the columns are renumbered, are copied into LDS at kernel
// start and gathered from there; the other lanes of a gather read global x.
template <int S, bool MASKED, bool HITS, int HOT>
__global__ __launch_bounds__(csr5_nt(S, HOT)) void k_csr5(const int* __restrict__ ccol,
                                              const float* __restrict__ cval,
                                              const unsigned* __restrict__ flags,
                                              const unsigned* __restrict__ tinfo,
                                              const float* __restrict__ x,
                                              int nnz, int ntiles,
                                              float* __restrict__ y, unsigned char* __restrict__ marks,
                                              float* __restrict__ carry_val,
                                              int* __restrict__ carry_row,
                                              int* __restrict__ carry_hit, int hot, int xn,
                                              float* __restrict__ clr, Gate g) {
  if (gate_shut(g)) return;
  if (clr) {
    // a buffer the caller wants all +0.0 (xn floats, 16-byte aligned)
    const int n4 = xn >> 2, gt = (int)(gridDim.x * blockDim.x);
    for (int i = (int)(blockIdx.x * blockDim.x + threadIdx.x); i < n4; i += gt)
      reinterpret_cast<float4*>(clr)[i] = make_float4(0.f, 0.f, 0.f, 0.f);
    const int i = (n4 << 2) + (int)(blockIdx.x * blockDim.x + threadIdx.x);
    if (i < xn) clr[i] = 0.f;
  }
  constexpr int T = kWave * S;
  const int lanes = lane();
  const int waves = gridDim.x * (blockDim.x / kWave);
  __shared__ float sx[HOT > 0 ? HOT : 1];
  // x through a buffer descriptor: one 32-bit offset per gather, and an
  // offset past x reads 0 instead of faulting
  const __amdgpu_buffer_rsrc_t xr =
      __builtin_amdgcn_make_buffer_rsrc((void*)x, (short)0, xn * 4, 0x00020000);
  if (HOT > 0) {
    // every wave of the block takes part (before any of them may leave)
    constexpr int NT = csr5_nt(S, HOT);
    constexpr int PT = HOT > 0 ? (HOT + NT - 1) / NT : 1;
    float v[PT];
#pragma unroll
    for (int k = 0; k < PT; ++k) {
      const int c = k * NT + (int)threadIdx.x;
      v[k] = x[c < hot ? c : 0];
    }
#pragma unroll
    for (int k = 0; k < PT; ++k) {
      const int c = k * NT + (int)threadIdx.x;
      if (HOT % NT == 0 || c < HOT) sx[c] = v[k];
    }
    __syncthreads();
  }
  // wave-uniform, so that per-tile words come through scalar loads
  int t = __builtin_amdgcn_readfirstlane(blockIdx.x * (blockDim.x / kWave) + threadIdx.x / kWave);
  if (t >= ntiles) return;

  int cN[S];  // stage 2: columns / values loading
  float vN[S];
  float vG[S], xG[S];  // stage 1: values and gathered x
  // hot items: their product (masked) is formed as soon as LDS answers and
  // kept in vG; bit i of hG marks item i hot, bit i of bG its support bit
  unsigned hG = 0u, bG = 0u;
  unsigned fG;  // the tile's marker word

  static_assert(S % 4 == 0, "items come in groups of four per lane");
  typedef int i4v __attribute__((ext_vector_type(4)));
  typedef float f4v __attribute__((ext_vector_type(4)));
  auto load_cv = [&](int tt) {
    // group g of this lane: items 4g .. 4g+3, one 16-byte load each
    const i4v* __restrict__ ct = reinterpret_cast<const i4v*>(ccol + (size_t)tt * T) + lanes;
    const f4v* __restrict__ vt = reinterpret_cast<const f4v*>(cval + (size_t)tt * T) + lanes;
#pragma unroll
    for (int g4 = 0; g4 < S / 4; ++g4) {
      const i4v c = __builtin_nontemporal_load(ct + g4 * kWave);
      const f4v v = __builtin_nontemporal_load(vt + g4 * kWave);
      cN[4 * g4] = c.x;
      cN[4 * g4 + 1] = c.y;
      cN[4 * g4 + 2] = c.z;
      cN[4 * g4 + 3] = c.w;
      vN[4 * g4] = v.x;
      vN[4 * g4 + 1] = v.y;
      vN[4 * g4 + 2] = v.z;
      vN[4 * g4 + 3] = v.w;
    }
  };
  auto gather = [&](int tt) {
    // real moves rather than renames (see the row-merge kernel): the stage
    // registers keep their roles and no in-flight load is copied. They come
    // first so that vN is free before the gathers' registers are taken (its
    // loads are a tile old; the column loads issued beside them are waited
    // for by the gathers anyway)
#pragma unroll
    for (int i = 0; i < S; ++i) asm volatile("v_mov_b32 %0, %1" : "=v"(vG[i]) : "v"(vN[i]));
    unsigned hm = 0u;
    if (HOT > 0) {
#pragma unroll
      for (int i = 0; i < S; ++i) hm |= ((unsigned)cN[i] < (unsigned)hot ? 1u : 0u) << i;
    }
    float xL[HOT > 0 ? S : 1];
#pragma unroll
    for (int i = 0; i < S; ++i) {
      if (HOT > 0) {
        // both reads unconditional: the hot lanes give the global read an
        // offset past the end of x (the buffer read returns 0 without a
        // memory access), the others read LDS word 0 (a broadcast)
        const unsigned c = (unsigned)cN[i];
        const bool hc = (hm >> i) & 1u;
        xG[i] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(xr, hc ? 0xFFFFFFF0u : c * 4u, 0, 0));
        xL[i] = sx[hc ? c : 0u];
      } else {
        xG[i] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(xr, (unsigned)cN[i] * 4u, 0, 0));
      }
    }
    fG = flags[(size_t)tt * kWave + lanes];
    if (HOT > 0) {
      // LDS answers within a few hundred cycles: the hot products are formed
      // here, so that xL dies at once and only two mask words live on
      unsigned bm = 0u;
#pragma unroll
      for (int i = 0; i < S; ++i) {
        const bool hc = (hm >> i) & 1u;
        const bool xb = __builtin_bit_cast(unsigned, xL[i]) != 0u;
        float p = vG[i] * xL[i];
        if (MASKED) p = xb ? p : 0.f;
        vG[i] = hc ? p : vG[i];
        bm |= (hc && xb ? 1u : 0u) << i;
      }
      hG = hm;
      bG = bm;
    }
  };

  load_cv(t);
  gather(t);
  load_cv(min(t + waves, ntiles - 1));

  for (; t < ntiles; t += waves) {
    const unsigned f = fG;
    const unsigned hh = hG, hb = bG;
    const unsigned ti = tinfo[t];
    const unsigned tn = tinfo[t + 1];
    const int base = (int)(ti & 0x7fffffffu);
    const int lim = nnz - t * T;  // items of this tile that exist (>= T except the last)

    // markers before this lane (DPP inclusive prefix of the popcounts)
    const int cnt = __popc(f);
    int incl = cnt;
    incl += dpp_i32<kDppRowShr1, 0xf>(0, incl);
    incl += dpp_i32<kDppRowShr2, 0xf>(0, incl);
    incl += dpp_i32<kDppRowShr4, 0xf>(0, incl);
    incl += dpp_i32<kDppRowShr8, 0xf>(0, incl);
    incl += dpp_i32<kDppRowBcast15, 0xa>(0, incl);
    incl += dpp_i32<kDppRowBcast31, 0xc>(0, incl);
    const int excl = incl - cnt;
    const int total = __shfl(incl, kWave - 1, kWave);

    // walk this lane's items; a segment that ends at a marker inside the
    // lane is a finished row. Products are formed on the way, so that the
    // stage-1 registers are free before the next tile is gathered into them.
    float s = 0.f, head_s = 0.f;
    int h = 0, head_h = 0, j = 0;
    bool head = true;
#pragma unroll
    for (int i = 0; i < S; ++i) {
      if ((f >> i) & 1u) {
        if (head) {
          head_s = s;
          head_h = h;
          head = false;
        } else {
          const unsigned k = (unsigned)(base + excl + j - 1);
          y[k] = s;
          if (HITS && h) marks[k] = 1;
        }
        s = 0.f;
        h = 0;
        ++j;
      }
      const bool ok = lanes * S + i < lim;
      bool b = __builtin_bit_cast(unsigned, xG[i]) != 0u;
      float q = vG[i] * xG[i];
      if (MASKED) q = b ? q : 0.f;
      if (HOT > 0 && ((hh >> i) & 1u)) {  // a select, not a branch
        b = (hb >> i) & 1u;
        q = vG[i];
      }
      s += ok ? q : 0.f;
      if (HITS) h |= (ok && b) ? 1 : 0;
    }
    __builtin_amdgcn_sched_barrier(0);
    gather(min(t + waves, ntiles - 1));
    __builtin_amdgcn_sched_barrier(0);
    load_cv(min(t + 2 * waves, ntiles - 1));
    __builtin_amdgcn_sched_barrier(0);

    // the segment open at the lane's end runs into the next lanes
    int fl = cnt > 0 ? 1 : 0;
    float sv = s;
    int hv = h;
    wave_seg_scan(fl, sv, hv);  // inclusive: segment open after this lane
    const float cin = dpp_f32<kDppWaveShr1, 0xf>(0.f, sv);
    const int hin = dpp_i32<kDppWaveShr1, 0xf>(0, hv);
    if (cnt > 0 && excl > 0) {
      // the head segment closes the row of the marker before this lane
      const unsigned k = (unsigned)(base + excl - 1);
      y[k] = cin + head_s;
      if (HITS && (hin | head_h)) marks[k] = 1;
    }
    if (lanes == kWave - 1) {
      // the tile's open segment: complete when the next tile starts a row
      const int k = base + total - 1;
      if (!(tn & 0x80000000u)) {
        y[(unsigned)k] = sv;
        if (HITS && hv) marks[k] = 1;
        carry_row[t] = -1;
      } else {
        carry_row[t] = k;
        carry_val[t] = sv;
        carry_hit[t] = hv;
      }
    }
  }
}

// rows that run through several tiles: their tail parts, added in tile order
__global__ void k_csr5_fixup(const float* __restrict__ carry_val, const int* __restrict__ carry_row,
                             const int* __restrict__ carry_hit, int ntiles, float* y,
                             unsigned char* marks, Gate g) {
  if (gate_shut(g)) return;
  for (int t = blockIdx.x * blockDim.x + threadIdx.x; t < ntiles; t += gridDim.x * blockDim.x) {
    int r, h;
    float s;
    if (!carry_run<int>(carry_val, carry_row, carry_hit, t, ntiles, r, s, h)) continue;
    y[r] += s;
    if (marks && h) marks[r] = 1;
  }
}

// dense y from the non-empty-row results: y[r] = y_ne[rank[r]] or 0, the rows
// that run through several tiles with their tail parts added in tile order
// (by the first fix_blocks workgroups, the others leave those rows alone; one
// launch where a fix-up in front of this one cost 5 us)
__global__ void k_csr5_expand(const int* __restrict__ row_ptr, const int* __restrict__ rank,
                              const int* __restrict__ rows_ne, int m, int T, const float* __restrict__ y_ne,
                              const float* __restrict__ carry_val, const int* __restrict__ carry_row, int ntiles,
                              int fix_blocks, float* __restrict__ y, Gate g) {
  if (gate_shut(g)) return;
  if ((int)blockIdx.x < fix_blocks) {
    for (int t = blockIdx.x * blockDim.x + threadIdx.x; t < ntiles; t += fix_blocks * blockDim.x) {
      int k, h;
      float s;
      if (carry_run<int>(carry_val, carry_row, nullptr, t, ntiles, k, s, h)) y[rows_ne[k]] = y_ne[k] + s;
    }
    return;
  }
  for (long long r = (long long)(blockIdx.x - fix_blocks) * blockDim.x + threadIdx.x; r < m;
       r += (long long)(gridDim.x - fix_blocks) * blockDim.x) {
    const int b = row_ptr[r], e = row_ptr[r + 1];
    const float v = e > b ? y_ne[rank[r]] : 0.f;
    if (e <= b || b / T == (e - 1) / T) y[r] = v;
  }
}

}  // namespace

namespace {

// ---- column order (most nonzeros first) -------------------------------------
// Sort key of column c: nnz - count(c), so an ascending stable sort puts the
// densest columns first and keeps equal counts in index order; the column
// index rides along as the value's bits.
__global__ void k_col_keys_from_ptr(const int* __restrict__ colptr, int n, long long nnz,
                                    unsigned* __restrict__ keys, float* __restrict__ vals) {
  for (long long c = (long long)blockIdx.x * blockDim.x + threadIdx.x; c < n;
       c += (long long)gridDim.x * blockDim.x) {
    keys[c] = (unsigned)(nnz - (colptr[c + 1] - colptr[c]));
    vals[c] = __int_as_float((int)c);
  }
}
__global__ void k_col_count(const int* __restrict__ col, int nnz, int n, unsigned* cnt) {
  for (long long j = (long long)blockIdx.x * blockDim.x + threadIdx.x; j < nnz;
       j += (long long)gridDim.x * blockDim.x) {
    const int c = col[j];
    if ((unsigned)c < (unsigned)n) atomicAdd(cnt + c, 1u);
  }
}
__global__ void k_col_keys_from_count(const unsigned* __restrict__ cnt, int n, long long nnz,
                                      unsigned* __restrict__ keys, float* __restrict__ vals) {
  for (long long c = (long long)blockIdx.x * blockDim.x + threadIdx.x; c < n;
       c += (long long)gridDim.x * blockDim.x) {
    keys[c] = (unsigned)(nnz - (long long)cnt[c]);
    vals[c] = __int_as_float((int)c);
  }
}
__global__ void k_set_count(long long* p, long long v) { *p = v; }
__global__ void k_set_int(int* p, int v) { *p = v; }
__global__ void k_invert_order(const float* __restrict__ vals, int n, int* __restrict__ cperm) {
  for (long long q = (long long)blockIdx.x * blockDim.x + threadIdx.x; q < n;
       q += (long long)gridDim.x * blockDim.x)
    cperm[__float_as_int(vals[q])] = (int)q;
}

}  // namespace

bool launch_column_order(hipStream_t s, const ColumnOrderArgs& a, const int* col, int nnz, int n,
                         int* cperm) {
  if (n <= 0 || n > a.sb_cap || nnz >= 0x7ffffffe) return false;
  const int grid = std::max(1, std::min(8192, (n + 255) / 256));
  if (a.csc_colptr) {
    hipLaunchKernelGGL(k_col_keys_from_ptr, dim3(grid), dim3(256), 0, s, a.csc_colptr, n,
                       (long long)nnz, a.sb.keyA, a.sb.valA);
  } else {
    launch_fill_i32(s, reinterpret_cast<int*>(a.sb.keyB), n, 0);
    hipLaunchKernelGGL(k_col_count, dim3(std::max(1, std::min(8192, (nnz + 255) / 256))), dim3(256), 0, s,
                       col, nnz, n, a.sb.keyB);
    hipLaunchKernelGGL(k_col_keys_from_count, dim3(grid), dim3(256), 0, s, a.sb.keyB, n, (long long)nnz,
                       a.sb.keyA, a.sb.valA);
  }
  hipLaunchKernelGGL(k_set_count, dim3(1), dim3(1), 0, s, a.n_dev, (long long)n);
  const int fb = launch_radix_sort(s, a.sb, nnz + 1, a.n_dev, a.ctl, n, n, false, a.ep);
  hipLaunchKernelGGL(k_invert_order, dim3(grid), dim3(256), 0, s, fb ? a.sb.valB : a.sb.valA, n, cperm);
  return hipGetLastError() == hipSuccess;
}

// ---- items of every row in the order of their new columns --------------------
// Rows of up to kOrderWin nonzeros: one workgroup takes the rows that start in
// its window of kOrderWin CSR positions, which are consecutive positions and at
// most kOrderCap of them, sorts them in LDS by (row, new column) and writes
// them to their places in the tiles. A longer row (it can only be the last one
// of a window) is left to a sort of all such rows' items through memory.
// Two stable sorts of every item through memory, by new column, then by row,
// took 1,740 us at R-MAT s19 (15.9 M nonzeros), this 450 us: 302 in LDS, which
// the ranking's ballots and LDS round trips bound, 150 for the 15 % of the
// items in long rows. Two workgroups of 512 threads share a CU's LDS (10 bytes
// per item and the counters) and overlap each other's barriers; one of 1,024
// with twice the window took 435 us in LDS, four of 256 (two thirds of the
// window, more long rows) 20 us more in all.
constexpr int kOrderNT = 512, kOrderIPT = 12, kOrderCap = kOrderNT * kOrderIPT, kOrderWin = kOrderCap / 2;

// where CSR position p lies in the copy (the layout in k_csr5_transpose)
__device__ __forceinline__ long long csr5_place(long long p, int T, int S) {
  const long long t = p / T;
  const int o = (int)(p - t * T);
  const int l = o / S, i = o - l * S;
  return t * T + (i >> 2) * (4 * kWave) + l * 4 + (i & 3);
}

// Rows of more than kOrderWin nonzeros: their number (high word of *count) and
// nonzeros (low word), and each one's row and first item among them.
__global__ void k_long_rows(const int* __restrict__ row_ptr, int m, unsigned long long* count,
                            int* __restrict__ long_row, int* __restrict__ long_off) {
  for (long long r0 = (long long)blockIdx.x * blockDim.x; r0 < m; r0 += (long long)gridDim.x * blockDim.x) {
    const long long r = r0 + threadIdx.x;
    const int len = r < m ? row_ptr[r + 1] - row_ptr[r] : 0;
    const unsigned long long mine = len > kOrderWin ? (1ull << 32) + (unsigned)len : 0ull;
    if (!__ballot(mine != 0ull)) continue;
    // one atomic per wave: rows and nonzeros of the wave at once
    const unsigned long long inc = wave_incl_sum(mine);
    unsigned long long base = 0;
    if (lane() == kWave - 1) base = atomicAdd(count, inc);
    base = __shfl(base, kWave - 1, kWave) + inc - mine;
    if (mine) {
      long_row[base >> 32] = (int)r;
      long_off[base >> 32] = (int)(unsigned)base;
    }
  }
}

// their items: key = new column, v = index of the row among them, w = value
__global__ void k_long_items(const int* __restrict__ row_ptr, const int* __restrict__ col,
                             const float* __restrict__ val, const int* __restrict__ cperm,
                             const int* __restrict__ long_row, const int* __restrict__ long_off, int items,
                             SortSet s) {
  for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < items; i += gridDim.x * blockDim.x) {
    const int li = (int)s.v[i];
    const int j = row_ptr[long_row[li]] + (i - long_off[li]);
    s.k[i] = (unsigned)cperm[col[j]];
    s.w[i] = __float_as_uint(val[j]);
  }
}

// sorted (key = row index, v = new column, w = value) to their places
__global__ void k_long_place(const int* __restrict__ row_ptr, const int* __restrict__ long_row,
                             const int* __restrict__ long_off, int items, SortSet s, int T, int S,
                             int* __restrict__ ccol, float* __restrict__ cval) {
  for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < items; i += gridDim.x * blockDim.x) {
    const int li = (int)s.k[i];
    const long long q = csr5_place((long long)row_ptr[long_row[li]] + (i - long_off[li]), T, S);
    ccol[q] = (int)s.v[i];
    cval[q] = __uint_as_float(s.w[i]);
  }
}

template <int NT, int IPT>
__global__ __launch_bounds__(NT) void k_order_rows(const int* __restrict__ row_ptr, const int* __restrict__ col,
                                                   const float* __restrict__ val, const int* __restrict__ cperm,
                                                   const int* __restrict__ rows_ne, const int* __restrict__ ne_before,
                                                   int m, int nnz, int nbits, int T, int S, long long total,
                                                   int* __restrict__ ccol, float* __restrict__ cval) {
  constexpr int CAP = NT * IPT, WIN = CAP / 2, NW = NT / kWave;
  __shared__ unsigned s_k[CAP];
  __shared__ float s_v[CAP];
  __shared__ unsigned short s_r[CAP];
  __shared__ unsigned s_cnt[NW * 256];
  __shared__ unsigned s_dstart[256];
  __shared__ unsigned s_t[NW];
  __shared__ int s_i[NW];
  if (blockIdx.x == gridDim.x - 1) {  // positions past the data, to the end of the last tile
    for (long long p = nnz + (long long)threadIdx.x; p < total; p += NT) {
      const long long q = csr5_place(p, T, S);
      ccol[q] = 0;
      cval[q] = 0.f;
    }
  }
  const long long w0 = (long long)blockIdx.x * WIN;
  const int w1 = (int)min(w0 + WIN, (long long)nnz);
  // the rows that start in [w0, w1): r0 .. rl, CSR positions [j0, j1)
  int r0 = block_last_le<NT>(row_ptr, 0, m, (int)w0, s_i);
  if (row_ptr[r0] < w0) ++r0;
  const int j0 = row_ptr[r0];
  if (j0 >= w1) return;
  const int rl = block_last_le<NT>(row_ptr, r0, m, w1 - 1, s_i);
  const int bl = row_ptr[rl], el = row_ptr[rl + 1];
  const bool is_long = el - bl > WIN;
  const int cnt = (is_long ? bl : el) - j0;
  if (cnt <= 0) return;
  // items per thread (<= IPT): every wave gets its share
  const int ie = (cnt + NT - 1) / NT;
  for (int i = threadIdx.x; i < cnt; i += NT) s_r[i] = 0;
  __syncthreads();
  const int n1 = ne_before[rl] + (is_long ? 0 : 1);
  for (int i = ne_before[r0] + (int)threadIdx.x; i < n1; i += NT) s_r[row_ptr[rows_ne[i]] - j0] = 1;
  __syncthreads();
  // row of every item, counted among the window's rows with nonzeros (only
  // these are walked: there may be any number of empty rows between them)
  int nrows;
  {
    const int i0 = threadIdx.x * ie;
    int heads = 0;
    for (int k = 0; k < ie; ++k) heads += i0 + k < cnt ? s_r[i0 + k] : 0;
    int run = block_excl_sum<NT, int>(heads, s_i, &nrows) - 1;
    for (int k = 0; k < ie; ++k) {
      if (i0 + k < cnt) {
        run += s_r[i0 + k];
        s_r[i0 + k] = (unsigned short)run;
      }
    }
  }
  __syncthreads();
  const int w = threadIdx.x / kWave;
  const int p0 = w * kWave * ie + lane();
  unsigned key[IPT], row[IPT], dig[IPT];
  float v[IPT];
  bool valid[IPT];
  int rank[IPT];
#pragma unroll
  for (int j = 0; j < IPT; ++j) {
    const int p = p0 + j * kWave;
    valid[j] = j < ie && p < cnt;
    key[j] = valid[j] ? (unsigned)col[j0 + p] : 0u;
    v[j] = valid[j] ? val[j0 + p] : 0.f;
    row[j] = valid[j] ? s_r[p] : 0u;
  }
#pragma unroll
  for (int j = 0; j < IPT; ++j) key[j] = valid[j] ? (unsigned)cperm[key[j]] : 0u;
  // stable LDS radix sort by (row, new column), digits of equal width
  const int bits = nbits + (nrows > 1 ? 32 - __builtin_clz(nrows - 1) : 0);
  const int passes = max(1, (bits + 7) / 8), per = (bits + passes - 1) / passes;
  for (int ps = 0; ps < passes; ++ps) {
    const int shift = ps * per, db = min(per, bits - shift);
    const unsigned mask = (1u << db) - 1u;
#pragma unroll
    for (int j = 0; j < IPT; ++j)
      dig[j] = valid[j] ? (unsigned)((((unsigned long long)row[j] << nbits) | key[j]) >> shift) & mask : 0u;
    wave_rank_digits<IPT>(dig, valid, s_cnt + w * 256, rank, ie, db);
    __syncthreads();
    unsigned tot = 0;
    if (threadIdx.x < 256) tot = digit_wave_offsets<NW>(s_cnt);
    unsigned dtot;
    const unsigned dex = block_excl_sum<NT, unsigned>(tot, s_t, &dtot);
    if (threadIdx.x < 256) s_dstart[threadIdx.x] = dex;
    __syncthreads();
#pragma unroll
    for (int j = 0; j < IPT; ++j) {
      if (valid[j]) {
        const unsigned q = s_dstart[dig[j]] + s_cnt[w * 256 + dig[j]] + rank[j];
        s_k[q] = key[j];
        s_v[q] = v[j];
        s_r[q] = (unsigned short)row[j];
      }
    }
    __syncthreads();
    if (ps + 1 < passes) {
#pragma unroll
      for (int j = 0; j < IPT; ++j) {
        const int p = p0 + j * kWave;
        if (valid[j]) {
          key[j] = s_k[p];
          v[j] = s_v[p];
          row[j] = s_r[p];
        }
      }
      __syncthreads();
    }
  }
  for (int i = threadIdx.x; i < cnt; i += NT) {
    const long long q = csr5_place((long long)j0 + i, T, S);
    ccol[q] = (int)s_k[i];
    cval[q] = s_v[i];
  }
}

// Every row's items in the order of their new columns, at their places in
// ccol / cval. nlong rows of more than kOrderWin nonzeros hold `items` of them.
static void launch_order_rows(hipStream_t s, const ColumnOrderArgs& a, const int* row_ptr, const int* col,
                              const float* val, int m, int n, int nnz, int T, int S, long long total,
                              const int* cperm, const int* rows_ne, const int* ne_before, int nlong, int items,
                              const int* long_row, const int* long_off, int* ccol, float* cval) {
  int nbits = 1;
  while (nbits < 31 && (1 << nbits) < n) ++nbits;
  if (nlong > 0) {
    // two sorts, by new column, then by row; all passes write two sets of
    // arrays in turn, the last one the set that is not the copy's own arrays
    const int grid = std::max(1, std::min(8192, (items + 255) / 256));
    const SortSet tmp{a.sb.keyA, reinterpret_cast<unsigned*>(a.sb.valA), reinterpret_cast<unsigned*>(a.sb.valB)};
    const SortSet own{a.sb.keyB, reinterpret_cast<unsigned*>(ccol), reinterpret_cast<unsigned*>(cval)};
    const int p1 = radix_passes(n), p2 = nlong > 1 ? radix_passes(nlong) : 0;
    const SortSet sets[2] = {(p1 + p2) & 1 ? tmp : own, (p1 + p2) & 1 ? own : tmp};
    // the first pass reads sets[1] and writes sets[0]
    launch_expand_rows(s, long_off, nlong, items, reinterpret_cast<int*>(sets[1].v));
    hipLaunchKernelGGL(k_long_items, dim3(grid), dim3(256), 0, s, row_ptr, col, val, cperm, long_row, long_off, items,
                       sets[1]);
    hipLaunchKernelGGL(k_set_count, dim3(1), dim3(1), 0, s, a.n_dev, (long long)items);
    const Ep e1{a.ep.v + 4u, -1}, e2{a.ep.v + 8u, -1};
    const int f1 = launch_radix_sets(s, a.sb, sets[1], sets[0], sets[1], n, a.n_dev, a.ctl, items, items, false, e1,
                                     Gate{}, 0);
    const auto by_row = [](const SortSet& q) { return SortSet{q.v, q.k, q.w}; };
    SortSet done = by_row(sets[f1]);
    if (nlong > 1) {
      const SortSet o0 = sets[f1 ^ 1], o1 = done;
      const int f2 = launch_radix_sets(s, a.sb, done, o0, o1, nlong, a.n_dev, a.ctl, items, items, false, e2, Gate{}, 0);
      done = f2 ? o1 : o0;
    }
    hipLaunchKernelGGL(k_long_place, dim3(grid), dim3(256), 0, s, row_ptr, long_row, long_off, items, done, T, S, ccol,
                       cval);
  }
  hipLaunchKernelGGL((k_order_rows<kOrderNT, kOrderIPT>), dim3((nnz - 1) / kOrderWin + 1), dim3(kOrderNT), 0, s,
                     row_ptr, col, val, cperm, rows_ne, ne_before, m, nnz, nbits, T, S, total, ccol, cval);
}

int csr5_sigma_of(int sigma, int m, long long nnz) {
  int s = sigma;
  if (s <= 0) {
    // nonzeros per row -> sigma, the reference's auto rule (spmspv.h:1397-1411)
    const long long per = m > 0 ? nnz / m : 0;
    if (per <= 4) s = 4;
    else if (per <= 32) s = (int)per;
    else if (per <= 256) s = 32;
    else s = 6;
  }
  // the instantiated widths
  if (s <= 8) return 8;
  if (s <= 16) return 16;
  if (s <= 24) return 24;
  return 32;
}

size_t csr5_bytes(int m, int n, long long nnz, int S) {
  const long long T = (long long)kWave * S;
  const long long ntiles = (nnz + T - 1) / T;
  auto up = [](size_t v) { return (v + 255) & ~size_t(255); };
  size_t b = 0;
  b += up(sizeof(int) * (size_t)std::max<long long>(ntiles * T, 1)) * 2;  // ccol, cval
  b += up(sizeof(unsigned) * (size_t)(ntiles + 1) * kWave);              // flags
  b += up(sizeof(unsigned) * (size_t)(ntiles + 2));                      // tinfo
  b += up(sizeof(int) * (size_t)m) * 4;                                  // rank, rows_ne, rows_empty, y_ne
  b += up(sizeof(int) * (size_t)(m / kScanPart + 2));                    // part sums
  b += up(sizeof(float) * (size_t)(ntiles + 1)) * 3;                     // carries
  b += up(sizeof(int) * (size_t)std::max(n, 1));                         // column order
  b += up(sizeof(unsigned long long));                                   // rows over kOrderWin: counts,
  b += up(sizeof(int) * (size_t)(nnz / kOrderWin + 2)) * 2;              // rows, first items
  return b;
}

hipError_t csr5_build(hipStream_t s, const int* row_ptr, const int* col, const float* val, int m,
                      int n, int nnz, int S, void* mem, int* h_pin, const ColumnOrderArgs* order,
                      Csr5* out) {
  const int T = kWave * S;
  const int ntiles = (int)(((long long)nnz + T - 1) / T);
  auto up = [](size_t v) { return (v + 255) & ~size_t(255); };
  char* p = static_cast<char*>(mem);
  Csr5 c{};
  c.S = S;
  c.row_ptr = row_ptr;
  c.ntiles = ntiles;
  c.ccol = reinterpret_cast<int*>(p);
  p += up(sizeof(int) * (size_t)std::max<long long>((long long)ntiles * T, 1));
  c.cval = reinterpret_cast<float*>(p);
  p += up(sizeof(int) * (size_t)std::max<long long>((long long)ntiles * T, 1));
  c.flags = reinterpret_cast<unsigned*>(p);
  p += up(sizeof(unsigned) * (size_t)(ntiles + 1) * kWave);
  c.tinfo = reinterpret_cast<unsigned*>(p);
  p += up(sizeof(unsigned) * (size_t)(ntiles + 2));
  int* rank = reinterpret_cast<int*>(p);
  c.rank = rank;
  p += up(sizeof(int) * (size_t)m);
  c.y_ne = reinterpret_cast<float*>(p);
  p += up(sizeof(float) * (size_t)m);
  c.rows_ne = reinterpret_cast<int*>(p);
  p += up(sizeof(int) * (size_t)m);
  c.rows_empty = reinterpret_cast<int*>(p);
  p += up(sizeof(int) * (size_t)m);
  int* sums = reinterpret_cast<int*>(p);
  p += up(sizeof(int) * (size_t)(m / kScanPart + 2));
  c.carry_val = reinterpret_cast<float*>(p);
  p += up(sizeof(float) * (size_t)(ntiles + 1));
  c.carry_row = reinterpret_cast<int*>(p);
  p += up(sizeof(float) * (size_t)(ntiles + 1));
  c.carry_hit = reinterpret_cast<int*>(p);
  p += up(sizeof(float) * (size_t)(ntiles + 1));
  int* cperm = reinterpret_cast<int*>(p);
  p += up(sizeof(int) * (size_t)std::max(n, 1));
  c.n = n;
  unsigned long long* long_count = reinterpret_cast<unsigned long long*>(p);
  p += up(sizeof(unsigned long long));
  int* long_row = reinterpret_cast<int*>(p);
  p += up(sizeof(int) * (size_t)(nnz / kOrderWin + 2));
  int* long_off = reinterpret_cast<int*>(p);
  // the order needs the sort buffers to hold a key per column
  if (order && nnz <= order->sb_cap && launch_column_order(s, *order, col, nnz, n, cperm)) {
    c.cperm = cperm;
    hipLaunchKernelGGL(k_set_count, dim3(1), dim3(1), 0, s, reinterpret_cast<long long*>(long_count), 0ll);
    hipLaunchKernelGGL(k_long_rows, dim3(std::max(1, std::min(2048, (m + 255) / 256))), dim3(256), 0, s, row_ptr, m,
                       long_count, long_row, long_off);
  }

  const int parts = (m + kScanPart - 1) / kScanPart;
  if (parts > 0) {
    hipLaunchKernelGGL(k_nonempty_part, dim3(parts), dim3(256), 0, s, row_ptr, m, sums);
    hipLaunchKernelGGL(k_scan_parts, dim3(1), dim3(256), 0, s, sums, parts);
    hipLaunchKernelGGL(k_rank_rows, dim3(parts), dim3(256), 0, s, row_ptr, m, sums, rank, c.rows_ne,
                       c.rows_empty);
  }
  launch_fill_i32(s, reinterpret_cast<int*>(c.flags), (long long)(ntiles + 1) * kWave, 0);
  h_pin[2] = h_pin[3] = 0;
  hipError_t e = hipMemcpyAsync(h_pin, sums + parts, sizeof(int), hipMemcpyDeviceToHost, s);
  if (e == hipSuccess && c.cperm)
    e = hipMemcpyAsync(h_pin + 2, long_count, sizeof(*long_count), hipMemcpyDeviceToHost, s);
  if (e != hipSuccess) return e;
  if ((e = hipStreamSynchronize(s)) != hipSuccess) return e;
  c.n_ne = parts > 0 ? h_pin[0] : 0;
  c.n_empty = m - c.n_ne;
  if (ntiles > 0) {
    hipLaunchKernelGGL(k_tile_info, dim3((ntiles + 1 + 255) / 256), dim3(256), 0, s, row_ptr, rank, m,
                       nnz, T, ntiles, c.n_ne, c.tinfo, c.flags);
    hipLaunchKernelGGL(k_row_markers, dim3(std::min(8192, (m + 255) / 256)), dim3(256), 0, s, row_ptr,
                       m, T, S, c.flags);
    const long long total = (long long)ntiles * T;
    if (c.cperm) {
      const int items = h_pin[2], nlong = h_pin[3];  // low and high word of the count
      if (nlong > 0) {
        // the rows' first items are searched as a row pointer is
        hipLaunchKernelGGL(k_set_int, dim3(1), dim3(1), 0, s, long_off + nlong, items);
      }
      launch_order_rows(s, *order, row_ptr, col, val, m, n, nnz, T, S, total, cperm, c.rows_ne, rank, nlong, items,
                        long_row, long_off, c.ccol, c.cval);
    } else {
      hipLaunchKernelGGL(k_csr5_transpose, dim3((unsigned)std::min<long long>(8192, (total + 255) / 256)),
                         dim3(256), 0, s, col, val, nnz, T, S, total, c.ccol, c.cval);
    }
  }
  *out = c;
  return hipGetLastError();
}

void launch_csr5(hipStream_t s, const Csr5& c, bool masked, bool hits, const float* x,
                 int m, int nnz, float* y, bool y_dense_rows,
                 unsigned char* marks, float** vals_out, const int** keymap_out, int* n_out,
                 hipEvent_t ev_begin, hipEvent_t ev_end, Gate g, float* clear) {
  const bool compressed = c.n_empty > 0;
  float* yk = compressed ? c.y_ne : y;  // results indexed by non-empty row
  *vals_out = yk;
  *keymap_out = compressed ? c.rows_ne : nullptr;
  *n_out = compressed ? c.n_ne : m;
  if (m <= 0 || c.ntiles == 0) {
    // no tile kernel: the buffer is cleared by a fill (gated alike)
    if (clear && c.n > 0) launch_fill_f32(s, clear, c.n, 0.f, g);
    if (m > 0 && y_dense_rows) launch_fill_f32(s, y, m, 0.f, g);
    return;
  }
  // the LDS copy holds the hot columns once they come first (column order),
  // or the whole of x when it fits
  const bool lds_hot = c.n >= 1 && (c.cperm != nullptr || c.n <= kCsr5Hot);
#define SPMSPV_CSR5(SS, MK, HT, HOTN)                                                            \
  {                                                                                              \
    const void* fn = (const void*)k_csr5<SS, MK, HT, HOTN>;                                  \
    constexpr int nt = csr5_nt(SS, HOTN), wpb = nt / kWave;                                      \
    const int waves = std::max(wpb, std::min(c.ntiles, resident_blocks(fn, nt) * wpb));          \
    hipLaunchKernelGGL((k_csr5<SS, MK, HT, HOTN>), dim3((waves + wpb - 1) / wpb), dim3(nt), 0, \
                       s,                                                                        \
                       c.ccol, c.cval, c.flags, c.tinfo, x, nnz, c.ntiles, yk, marks,            \
                       c.carry_val, c.carry_row, c.carry_hit, std::min(c.n, HOTN), c.n, clear, g); \
  }
#define SPMSPV_CSR5_H(SS, MK, HT)                \
  if (lds_hot) SPMSPV_CSR5(SS, MK, HT, kCsr5Hot) \
  else SPMSPV_CSR5(SS, MK, HT, 0)
#define SPMSPV_CSR5_S(SS)                               \
  if (masked && hits) SPMSPV_CSR5_H(SS, true, true)     \
  else if (masked) SPMSPV_CSR5_H(SS, true, false)       \
  else if (hits) SPMSPV_CSR5_H(SS, false, true)         \
  else SPMSPV_CSR5_H(SS, false, false)
  if (ev_begin) (void)hipEventRecord(ev_begin, s);
  if (c.S == 8) {
    SPMSPV_CSR5_S(8)
  } else if (c.S == 16) {
    SPMSPV_CSR5_S(16)
  } else if (c.S == 24) {
    SPMSPV_CSR5_S(24)
  } else {
    SPMSPV_CSR5_S(32)
  }
#undef SPMSPV_CSR5_S
#undef SPMSPV_CSR5_H
#undef SPMSPV_CSR5
  if (ev_end) (void)hipEventRecord(ev_end, s);
  const int fix = std::min(1024, (c.ntiles + 255) / 256);
  const bool expand = compressed && y_dense_rows;
  // with hits, the compaction reads the fixed non-empty-row results
  const bool fused = expand && !hits;
  if (!fused)
    hipLaunchKernelGGL(k_csr5_fixup, dim3(fix), dim3(256), 0, s, c.carry_val, c.carry_row, c.carry_hit, c.ntiles, yk,
                       hits ? marks : nullptr, g);
  if (expand) {
    const int fix_blocks = fused ? fix : 0;
    // already fixed: no row is left out
    const int T = fused ? kWave * c.S : INT_MAX;
    hipLaunchKernelGGL(k_csr5_expand, dim3(fix_blocks + std::min(8192, (m + 255) / 256)), dim3(256), 0, s, c.row_ptr,
                       c.rank, c.rows_ne, m, T, c.y_ne, c.carry_val, c.carry_row, c.ntiles, fix_blocks, y, g);
  }
}

}  // namespace spmspv
