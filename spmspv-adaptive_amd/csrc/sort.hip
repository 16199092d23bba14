// In-house LSD radix sort of (uint32 key, 32-bit value) pairs and the
// segmented reduce-by-key that follows it: the sort half of the reference's
// CSC sort kernels (thrust::sort_by_key + thrust::reduce_by_key,
// la/include/spmspv/csc-spmspv/detail/device/csc_sort_spmspv.cuh:339-437,
// 1030-1152), written for wave64:
//  * keys are ranked inside a tile with a wave ballot per bit of the digit (at
//    most 8; peers hold the same digit) and per-wave digit counters in LDS
//    (stable);
//  * each pass counts digits per tile, turns the counts into positions (the
//    scatter's workgroups sum them; for many tiles one small look-back scan
//    over 256 x tiles entries) and scatters, so no tile waits on a chain of
//    earlier tiles;
//  * tiles are re-ordered in LDS before the store so that runs of equal
//    digits leave as contiguous, coalesced writes;
//  * n <= one tile takes a single-workgroup path that sorts all passes in
//    LDS and reduces in the same launch.
// The reduce is deterministic: fixed-order segmented scans inside a tile
// and a fixed-order carry fix-up across tiles.
#include "kernels.hpp"
#include "ranking.hpp"
#include "selector.hpp"

namespace spmspv {

// -------------------------------------------------------- segmented scan
// Exclusive segmented sum over the threads of a block: the combine of
// (f1,v1) then (f2,v2) is (f1|f2, f2 ? v2 : v1 + v2). Returns for each
// thread the combined value of all earlier threads back to the nearest one
// with f set (inclusive). Also returns the block-inclusive value of the last
// thread in *last_incl (valid in all threads).
template <int NT, typename V>
__device__ __forceinline__ V block_seg_excl(bool f, V v, int* s_f, V* s_v, V* last_incl) {
  constexpr int NW = NT / kWave;
  const int w = threadIdx.x / kWave;
  int fi = f ? 1 : 0;
  V vi = v;
#pragma unroll
  for (int o = 1; o < kWave; o <<= 1) {
    const int fo = __shfl_up(fi, o, kWave);
    const V vo = __shfl_up(vi, o, kWave);
    if (lane() >= o) {
      if (!fi) vi = vo + vi;
      fi |= fo;
    }
  }
  if (lane() == kWave - 1) {
    s_f[w] = fi;
    s_v[w] = vi;
  }
  __syncthreads();
  V pv = V(0);
  for (int k = 0; k < w; ++k) pv = s_f[k] ? s_v[k] : pv + s_v[k];
  V tv = V(0);
  for (int k = 0; k < NW; ++k) tv = s_f[k] ? s_v[k] : tv + s_v[k];
  const V incl = fi ? vi : pv + vi;
  V ex = __shfl_up(incl, 1, kWave);
  if (lane() == 0) ex = pv;
  __syncthreads();
  *last_incl = tv;
  return ex;
}

// ---------------------------------------------------------- tile reduce
// Reduces the sorted keys s_k[0..cnt) / values s_v of one tile. `prev_key`
// is the key just before the tile (ignored when global_start). get_prefix
// (called by all threads with the tile's head count) returns the number of
// heads of all earlier tiles. Segment ends whose head lies in an earlier
// tile go to carry_val/carry_idx[tile] for the fix-up kernel.
template <int NT, int IPT, typename PrefixFn>
__device__ __forceinline__ long long tile_reduce(const unsigned* s_k, const float* s_v, int cnt,
                                                 unsigned prev_key, bool global_start,
                                                 PrefixFn get_prefix, int* ykey, float* yval,
                                                 float* carry_val, int* carry_idx, long long tile,
                                                 int* s_i, int* s_f, float* s_fv, int ipt = IPT) {
  // thread t reduces sorted items t*ipt .. t*ipt+ipt-1 (ipt <= IPT)
  const int i0 = threadIdx.x * ipt;
  bool head[IPT];
  int nh = 0;
  float tail = 0.f;
#pragma unroll
  for (int j = 0; j < IPT; ++j) {
    const int i = i0 + j;
    head[j] = false;
    if (j < ipt && i < cnt) {
      const unsigned pk = (i == 0) ? prev_key : s_k[i - 1];
      head[j] = (i == 0 && global_start) || s_k[i] != pk;
      if (head[j]) tail = s_v[i];
      else tail += s_v[i];
    }
    nh += head[j] ? 1 : 0;
  }
  int htot;
  const int hex = block_excl_sum<NT, int>(nh, s_i, &htot);
  const long long gpre = get_prefix(htot);
  float last_incl;
  const float cin = block_seg_excl<NT, float>(nh > 0, tail, s_f, s_fv, &last_incl);
  float acc = cin;
  int hc = hex;
#pragma unroll
  for (int j = 0; j < IPT; ++j) {
    const int i = i0 + j;
    if (j >= ipt || i >= cnt) break;
    if (head[j]) {
      ++hc;
      acc = s_v[i];
      ykey[gpre + hc - 1] = (int)s_k[i];
    } else {
      acc += s_v[i];
    }
    const bool end = (i == cnt - 1) || (s_k[i + 1] != s_k[i]);
    if (end) {
      if (hc > 0) {
        yval[gpre + hc - 1] = acc;
      } else {
        carry_val[tile] = acc;
        carry_idx[tile] = (int)(gpre - 1);
      }
    }
  }
  if (threadIdx.x == 0 && carry_idx && (cnt == 0 || head[0])) carry_idx[tile] = -1;
  return gpre + htot;
}

// ------------------------------------------------------------ one pass
// A pass is three launches (two where the counts are summed in the scatter),
// with no look-back chain between tiles:
//   k_digit_count  per-tile digit counts, digit-major: cnt[d * ntiles + t];
//   k_digit_scan   exclusive scan of that array in place, so that
//                  cnt[d * ntiles + t] becomes the global position of the
//                  first item of digit d in tile t (stable: digit, then tile);
//   k_sort_scatter ranks the tile again and writes every item there.
// (With every tile resident at once, a per-digit decoupled look-back
// spends most of the pass waiting for the prefix to crawl along the tile
// chain; the scan of 256 x ntiles counts costs a few microseconds.)
// Smaller sorts have no scan: the counts are 16 bits wide and tile-major,
// cnt[t << bits | d], k_digit_count also adds them up per kChunk tiles
// (chunk, a buffer for each pass: cleared by the next pass, or by the first
// pass of the next sort), and every scatter workgroup sums the chunks and the
// tiles of its own chunk itself while its keys are on their way. The
// scan is 6 us and a launch gap per pass whatever the size; the sums cost what
// is read for them, tiles * (chunks + half a chunk) rows. The whole slot (3
// passes of 7 bits): 391 k products 93.9 -> 82.6 us, 1.53 M 114.9 -> 102.9,
// 2.93 M 137.1 -> 128.7; (8 + 7 + 7): 0.81 M 111.0 -> 99.0, 3.02 M 152.5 ->
// 142.3, 3.44 M (its 8-bit pass over the line) 166.5 -> 163.9. Nothing more was
// gained above the line (5.6 M: 227.0 without it, 226.1 with the scan).
constexpr long long kDirectReads = 20 << 20;
constexpr int kChunkWords = kChunkRows * 64;  // 64-bit words (4 digits) of a pass's buffer
__host__ __device__ inline bool counts_direct(long long ntiles, int bits) {
  return ntiles <= kChunkRows * kChunk && (ntiles * (ntiles / kChunk + kChunk / 2)) << bits <= kDirectReads;
}
static_assert(kChunk * kSortTile < 65536, "16-bit digit counts of a chunk");
// digits of a row of those counts (whole 8-byte words)
__host__ __device__ inline int direct_row(int bits) { return bits < 2 ? 4 : 1 << bits; }

// Keys of tile t in the wave-major layout of wave_rank.
template <int NT, int IPT>
__device__ __forceinline__ void load_tile_keys(const unsigned* __restrict__ kin, long long n,
                                               long long base, unsigned (&key)[IPT],
                                               bool (&valid)[IPT]) {
  const int w = threadIdx.x / kWave;
#pragma unroll
  for (int j = 0; j < IPT; ++j) {
    const long long gi = base + (long long)w * kWave * IPT + j * kWave + lane();
    valid[j] = gi < n;
    key[j] = kin[valid[j] ? gi : n - 1];
  }
}

template <int NT, int IPT>
__global__ __launch_bounds__(NT) void k_digit_count(const unsigned* __restrict__ kin,
                                                    const long long* __restrict__ n_dev, int shift, int bits,
                                                    unsigned* __restrict__ cnt,
                                                    unsigned long long* __restrict__ chunk, int pass, int small_cap,
                                                    long long n_cap, Gate g) {
  if (gate_shut(g)) return;
  constexpr int TILE = NT * IPT;
  constexpr int NW = NT / kWave;
  static_assert(NT == 256, "one thread per digit");
  const unsigned mask = (1u << bits) - 1u;
  __shared__ unsigned s_cnt[NW * 256];
  const long long n = *n_dev;
  if (n <= small_cap || n > n_cap) return;
  const unsigned ntiles = (unsigned)((n + TILE - 1) / TILE);
  const int w = threadIdx.x / kWave;
  if (chunk) {
    const int first = pass == 0 ? 1 : pass - 1, last = pass == 0 ? 4 : pass;
    for (int i = first * kChunkWords + blockIdx.x * NT + threadIdx.x; i < last * kChunkWords; i += gridDim.x * NT)
      chunk[i] = 0ull;
  }
  // tiles are independent: any grid covers them. Only counts are needed
  // here (no ranks): LDS atomics into a private histogram per wave. Lanes that
  // add to one LDS word take turns, so where many lanes hold the first lane's
  // digit (power-law column indices), those lanes add once between them (52 ->
  // 20 us for 15.9 M such keys; the same grouping of every digit by ballots
  // costs 7.4 -> 10.7 us for 1.4 M even ones)
  for (unsigned t = blockIdx.x; t < ntiles; t += gridDim.x) {
    unsigned key[IPT];
    bool valid[IPT];
    load_tile_keys<NT, IPT>(kin, n, (long long)t * TILE, key, valid);
#pragma unroll
    for (int q = 0; q < NW; ++q) s_cnt[q * 256 + threadIdx.x] = 0u;
    __syncthreads();
#pragma unroll
    for (int j = 0; j < IPT; ++j)
    {
      const unsigned d = (key[j] >> shift) & mask;
      const uint64_t same = __ballot(valid[j] && d == (unsigned)__builtin_amdgcn_readfirstlane((int)d));
      const bool many = __popcll(same) > 4;
      const bool in_same = (same >> lane()) & 1ull;
      if (many && same && __builtin_ctzll(same) == lane())
        atomicAdd(&s_cnt[w * 256 + d], (unsigned)__popcll(same));
      if (valid[j] && !(many && in_same)) atomicAdd(&s_cnt[w * 256 + d], 1u);
    }
    __syncthreads();
    unsigned tot = 0;
#pragma unroll
    for (int q = 0; q < NW; ++q) tot += s_cnt[q * 256 + threadIdx.x];
    if (chunk && counts_direct(ntiles, bits)) {
      const int row = direct_row(bits);
      if ((int)threadIdx.x < row) reinterpret_cast<unsigned short*>(cnt)[t * row + threadIdx.x] = (unsigned short)tot;
      s_cnt[threadIdx.x] = tot;
      __syncthreads();
      if ((int)threadIdx.x < row / 4) {
        unsigned long long four = 0ull;
#pragma unroll
        for (int k = 0; k < 4; ++k) four |= (unsigned long long)s_cnt[threadIdx.x * 4 + k] << (16 * k);
        if (four) atomicAdd(chunk + (size_t)pass * kChunkWords + t / kChunk * (row / 4) + threadIdx.x, four);
      }
    } else if (threadIdx.x <= mask) {
      cnt[(size_t)threadIdx.x * ntiles + t] = tot;
    }
    __syncthreads();
  }
}

// In-place exclusive scan of cnt[0 .. 2^bits * ntiles) (ntiles from n and the
// sort tile), ordered tiles of NT * IPT entries with decoupled look-back.
template <int NT, int IPT>
__global__ __launch_bounds__(NT) void k_digit_scan(unsigned* __restrict__ cnt,
                                                   const long long* __restrict__ n_dev, int sort_tile,
                                                   int bits, bool chunks, int small_cap, long long n_cap,
                                                   unsigned long long* state, Ctl* ctl,
                                                   Ep epa, Gate g) {
  if (gate_shut(g)) return;
  __shared__ unsigned long long s_pre;
  __shared__ unsigned s_t[NT / kWave];
  const long long n = *n_dev;
  if (n <= small_cap || n > n_cap) return;
  if (chunks && counts_direct((n + sort_tile - 1) / sort_tile, bits)) return;
  const long long E = ((n + sort_tile - 1) / sort_tile) << bits;
  const unsigned nb = (unsigned)((E + NT * IPT - 1) / (NT * IPT));
  const unsigned t = blockIdx.x;
  if (t >= nb) return;
  const unsigned epoch = ep_of(ctl, epa);
  const long long base = (long long)t * NT * IPT + (long long)threadIdx.x * IPT;
  unsigned v[IPT];
  unsigned sum = 0;
#pragma unroll
  for (int j = 0; j < IPT; ++j) {
    const long long i = base + j;
    v[j] = cnt[i < E ? i : E - 1];
    v[j] = i < E ? v[j] : 0u;
    sum += v[j];
  }
  unsigned btot;
  const unsigned bex = block_excl_sum<NT, unsigned>(sum, s_t, &btot);
  const unsigned long long pre = tile_prefix(state, t, epoch, (unsigned long long)btot, &s_pre);
  unsigned run = (unsigned)pre + bex;
#pragma unroll
  for (int j = 0; j < IPT; ++j) {
    const long long i = base + j;
    if (i < E) cnt[i] = run;
    run += v[j];
  }
}

// Global start of digit threadIdx.x in tile t from the 16-bit counts, by the
// whole workgroup: 8-byte loads of 4 digits (16-byte ones take the registers
// of a wave per SIMD), the rows (every chunk's, then those of the earlier
// tiles of t's chunk) split over the groups of lanes that cover a row. s_a,
// s_b: NW * 256 words each; the caller syncs before it uses them again.
template <int NT>
__device__ __forceinline__ unsigned direct_start(const unsigned* cnt, const unsigned long long* chunk, unsigned t,
                                                 unsigned ntiles, int bits, unsigned* s_a, unsigned* s_b,
                                                 unsigned* s_t) {
  constexpr int NW = NT / kWave, U = 4;
  const int row = direct_row(bits), lpr = row / 4;
  const unsigned grp = NT / lpr;
  const int c = threadIdx.x % lpr;
  const unsigned mine = t / kChunk, nch = (ntiles + kChunk - 1) / kChunk, rows = nch + t % kChunk;
  const uint2* pc = reinterpret_cast<const uint2*>(chunk) + c;
  const uint2* pt = reinterpret_cast<const uint2*>(cnt) + (size_t)mine * kChunk * lpr + c;
  unsigned before[4], all[4];
#pragma unroll
  for (int k = 0; k < 4; ++k) before[k] = all[k] = 0u;
  for (unsigned u0 = threadIdx.x / lpr; u0 < rows; u0 += grp * U) {
    uint2 v[U];
#pragma unroll
    for (int j = 0; j < U; ++j) {
      const unsigned u = min(u0 + j * grp, rows - 1);
      v[j] = *(u < nch ? pc + (size_t)u * lpr : pt + (size_t)(u - nch) * lpr);
    }
#pragma unroll
    for (int j = 0; j < U; ++j) {
      const unsigned u = u0 + j * grp;
      const unsigned mb = u < mine || (u >= nch && u < rows) ? ~0u : 0u, ma = u < nch ? ~0u : 0u;
      const unsigned w[2] = {v[j].x, v[j].y};
#pragma unroll
      for (int k = 0; k < 2; ++k) {
        before[2 * k] += w[k] & mb & 0xFFFFu;
        before[2 * k + 1] += (w[k] & mb) >> 16;
        all[2 * k] += w[k] & ma & 0xFFFFu;
        all[2 * k + 1] += (w[k] & ma) >> 16;
      }
    }
  }
  // the groups of a wave, then the waves
  for (int o = lpr; o < kWave; o <<= 1) {
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      before[k] += __shfl_xor(before[k], o);
      all[k] += __shfl_xor(all[k], o);
    }
  }
  if (lane() < lpr) {
    const int w = threadIdx.x / kWave;
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      s_a[w * 256 + c * 4 + k] = before[k];
      s_b[w * 256 + c * 4 + k] = all[k];
    }
  }
  __syncthreads();
  unsigned b = 0u, a = 0u;  // items of the digit before the tile, and in all tiles
  if ((int)threadIdx.x < row) {
#pragma unroll
    for (int w = 0; w < NW; ++w) {
      b += s_a[w * 256 + threadIdx.x];
      a += s_b[w * 256 + threadIdx.x];
    }
  }
  unsigned tot;
  return block_excl_sum<NT, unsigned>(a, s_t, &tot) + b;
}

// Sorts of many items with two payloads stream through HBM: twice the tile, so
// that a run of equal digits fills its lines (15.9 M items of R-MAT scale 19,
// 382 MB: 97 -> 86.5 us per pass; a copy would take 81). The second payload goes
// through the first one's LDS, which leaves two workgroups per CU; 512 x 16 took
// 88, 1,024 x 6 and x 8 105 us. Their counts do not fit 16 bits per 16 tiles, so
// the positions come from the scan. ToCSC with the narrow / wide tile, us:
// R-MAT 0.88 M nonzeros 59 / 75, 1.82 M 73 / 87, 4.41 M 158 / 166, 5.34 M 182 /
// 186, 6.26 M 198 / 198, 7.61 M 218 / 218, 15.5 M 432 / 408; even columns 2.10 M
// 89 / 109, 4.88 M 162 / 165, 5.88 M 180 / 180, 6.88 M 195 / 200, 8.39 M 219 /
// 223, 12.6 M 346 / 330, 16.8 M 504 / 442; banded 4.46 M 153 / 158, 6.29 M 206 /
// 203, 7.34 M 229 / 225.
constexpr int kWideNT = 512;
constexpr long long kWideItems = 6 << 20;

// PAY: payload words per item (0: keys only). Four waves per SIMD (three with
// two payloads, as LDS allows): five spill the payloads (R-MAT scale 22, 1 %:
// 105.5 -> 110.7 us).
template <int NT, int IPT, int PAY>
__global__ __launch_bounds__(NT, NT == 256 && PAY > 1 ? 3 : 4) void k_sort_scatter(SortSet in, SortSet out, const long long* __restrict__ n_dev,
                                                     int shift, int bits, const unsigned* __restrict__ pos0,
                                                     const unsigned long long* __restrict__ chunk, int small_cap, long long n_cap, Gate g) {
  if (gate_shut(g)) return;
  constexpr int TILE = NT * IPT;
  constexpr int NW = NT / kWave;
  constexpr bool WIDE = NT > 256;  // the second payload goes through the first one's LDS
  static_assert(NT >= 256, "one thread per digit");
  __shared__ unsigned s_k[TILE];
  __shared__ unsigned s_v[PAY > 0 ? TILE : 1];
  __shared__ unsigned s_w[PAY > 1 && !WIDE ? TILE : 1];
  __shared__ unsigned s_cnt[NW * 256];
  __shared__ unsigned s_dstart[256];
  __shared__ unsigned s_gbase[256];
  __shared__ unsigned s_t[NW];
  const unsigned mask = (1u << bits) - 1u;
  const long long n = *n_dev;
  if (n <= small_cap || n > n_cap) return;
  const unsigned ntiles = (unsigned)((n + TILE - 1) / TILE);
  const int w = threadIdx.x / kWave;
  const unsigned d = threadIdx.x;
  // tiles are independent: any grid covers them
  for (unsigned t = blockIdx.x; t < ntiles; t += gridDim.x) {
    const long long base = (long long)t * TILE;
    // this tile's global start of digit d, from the scan (issued with the keys)
    const bool direct = chunk && counts_direct(ntiles, bits);
    unsigned gb = direct ? 0u : pos0[(size_t)(d & mask) * ntiles + t];
    unsigned key[IPT], pv[IPT], pw[IPT];
    bool valid[IPT];
    int rank[IPT];
    unsigned dig[IPT];
    load_tile_keys<NT, IPT>(in.k, n, base, key, valid);
#pragma unroll
    for (int j = 0; j < IPT; ++j) {
      const long long gi = base + (long long)w * kWave * IPT + j * kWave + lane();
      if (PAY > 0) pv[j] = in.v[valid[j] ? gi : n - 1];
      if (PAY > 1) pw[j] = in.w[valid[j] ? gi : n - 1];
    }
    if (NT == 256 && direct) {
      gb = direct_start<256>(pos0, chunk, t, ntiles, bits, s_cnt, s_k, s_t);
      __syncthreads();
    }
    wave_rank<IPT>(key, valid, shift, s_cnt + w * 256, rank, dig, IPT, bits);
    __syncthreads();
    const unsigned tot = NT == 256 || d < 256 ? digit_wave_offsets<NW>(s_cnt) : 0u;
    unsigned dtot;
    const unsigned dst = block_excl_sum<NT, unsigned>(tot, s_t, &dtot);
    if (NT == 256 || d < 256) {
      s_dstart[d] = dst;
      s_gbase[d] = gb;
    }
    __syncthreads();
#pragma unroll
    for (int j = 0; j < IPT; ++j) {
      if (valid[j]) {
        const unsigned p = s_dstart[dig[j]] + s_cnt[w * 256 + dig[j]] + rank[j];
        s_k[p] = key[j];
        if (PAY > 0) s_v[p] = pv[j];
        if (PAY > 1 && !WIDE) s_w[p] = pw[j];
        if (PAY > 1 && WIDE) rank[j] = (int)p;
      }
    }
    __syncthreads();
    const int cnt = (int)min((long long)TILE, n - base);
    for (int i = threadIdx.x; i < cnt; i += NT) {
      const unsigned k = s_k[i];
      const unsigned dd = (k >> shift) & mask;
      const unsigned q = s_gbase[dd] + (i - s_dstart[dd]);
      out.k[q] = k;
      if (PAY > 0) out.v[q] = s_v[i];
      if (PAY > 1 && !WIDE) out.w[q] = s_w[i];
    }
    if (PAY > 1 && WIDE) {
      __syncthreads();
#pragma unroll
      for (int j = 0; j < IPT; ++j)
        if (valid[j]) s_v[rank[j]] = pw[j];
      __syncthreads();
      for (int i = threadIdx.x; i < cnt; i += NT) {
        const unsigned dd = (s_k[i] >> shift) & mask;
        out.w[s_gbase[dd] + (i - s_dstart[dd])] = s_v[i];
      }
    }
    __syncthreads();
  }
}

// --------------------------------------------------- single-workgroup path
// n <= TILE: all passes in LDS. mode 0: reduce and write (ykey, yval,
// ctl->ynnz). mode 1: write the sorted items to `out`.
template <int NT, int IPT, int PAY>
__global__ __launch_bounds__(NT) void k_sort_small(SortSet in, const long long* __restrict__ n_dev, int passes,
                                                   int mode, Ctl* ctl, int* ykey, float* yval, SortSet out,
                                                   int cap, long long* sig, Gate g) {
  if (gate_shut(g)) return;
  constexpr int TILE = NT * IPT;
  constexpr int NW = NT / kWave;
  __shared__ unsigned s_k[TILE];
  __shared__ float s_v[TILE];
  __shared__ unsigned s_w[PAY > 1 ? TILE : 1];
  __shared__ unsigned s_cnt[NW * 256];
  __shared__ unsigned s_dstart[256];
  __shared__ unsigned s_t[NW];
  __shared__ int s_i[NW];
  __shared__ int s_f[NW];
  __shared__ float s_fv[NW];
  const long long n = *n_dev;
  if (n > TILE || n > cap) return;
  const int w = threadIdx.x / kWave;
  // items per thread for this n (<= IPT): every wave ranks its share
  const int ie = (int)((n + NT - 1) / NT);
  unsigned key[IPT], pw[IPT];
  float val[IPT];
  bool valid[IPT];
  int rank[IPT];
  unsigned dig[IPT];
#pragma unroll
  for (int j = 0; j < IPT; ++j) {
    const int gi = w * kWave * ie + j * kWave + lane();
    valid[j] = j < ie && gi < n;
    key[j] = valid[j] ? in.k[gi] : 0u;
    val[j] = PAY > 0 && valid[j] ? __uint_as_float(in.v[gi]) : 0.f;
    if (PAY > 1) pw[j] = valid[j] ? in.w[gi] : 0u;
  }
  for (int p = 0; p < passes; ++p) {
    wave_rank<IPT>(key, valid, 8 * p, s_cnt + w * 256, rank, dig, ie);
    __syncthreads();
    const unsigned tot = digit_wave_offsets<NW>(s_cnt);
    unsigned dtot;
    const unsigned dex = block_excl_sum<NT, unsigned>(tot, s_t, &dtot);
    s_dstart[threadIdx.x] = dex;
    __syncthreads();
#pragma unroll
    for (int j = 0; j < IPT; ++j) {
      if (valid[j]) {
        const unsigned pos = s_dstart[dig[j]] + s_cnt[w * 256 + dig[j]] + rank[j];
        s_k[pos] = key[j];
        s_v[pos] = val[j];
        if (PAY > 1) s_w[pos] = pw[j];
      }
    }
    __syncthreads();
    if (p + 1 < passes) {
#pragma unroll
      for (int j = 0; j < IPT; ++j) {
        const int gi = w * kWave * ie + j * kWave + lane();
        if (valid[j]) {
          key[j] = s_k[gi];
          val[j] = s_v[gi];
          if (PAY > 1) pw[j] = s_w[gi];
        }
      }
      __syncthreads();
    }
  }
  const int cnt = (int)n;
  if (mode == 1) {
    for (int i = threadIdx.x; i < cnt; i += NT) {
      out.k[i] = s_k[i];
      if (PAY > 0) out.v[i] = __float_as_uint(s_v[i]);
      if (PAY > 1) out.w[i] = s_w[i];
    }
    return;
  }
  auto no_prefix = [](int) -> long long { return 0; };
  const long long tot = tile_reduce<NT, IPT>(s_k, s_v, cnt, 0u, true, no_prefix, ykey, yval,
                                             nullptr, nullptr, 0, s_i, s_f, s_fv, ie);
  if (threadIdx.x == 0) {
    ctl->ynnz = (int)tot;
    ctl->sort_small = 1;
  }
  if (sig) {  // the result first, then its count
    __threadfence_system();
    __syncthreads();
    if (threadIdx.x == 0) *sig = tot;
  }
}

// ------------------------------------------------------- reduce by key
template <int NT, int IPT>
__global__ __launch_bounds__(NT) void k_reduce(const unsigned* __restrict__ keys,
                                               const float* __restrict__ vals,
                                               const long long* __restrict__ n_dev, Ctl* ctl,
                                               int* ykey, float* yval, float* carry_val,
                                               int* carry_idx, unsigned long long* state, Ep epa,
                                               int small_cap, long long n_cap, Gate g) {
  if (gate_shut(g)) return;
  constexpr int TILE = NT * IPT;
  constexpr int NW = NT / kWave;
  __shared__ unsigned s_k[TILE];
  __shared__ float s_v[TILE];
  __shared__ int s_i[NW];
  __shared__ int s_f[NW];
  __shared__ float s_fv[NW];
  __shared__ unsigned long long s_pre;
  const long long n = *n_dev;
  if (n <= small_cap || n > n_cap) return;
  const unsigned ntiles = (unsigned)((n + TILE - 1) / TILE);
  const unsigned t = blockIdx.x;
  if (t >= ntiles) return;
  const unsigned epoch = ep_of(ctl, epa);
  {
    const long long base = (long long)t * TILE;
    const int cnt = (int)min((long long)TILE, n - base);
    {
      // all of a thread's loads at once (clamped), then into LDS
      unsigned kk[IPT];
      float vv[IPT];
#pragma unroll
      for (int j = 0; j < IPT; ++j) {
        const int i = threadIdx.x + j * NT;
        const long long gi = base + (i < cnt ? i : 0);
        kk[j] = keys[gi];
        vv[j] = vals[gi];
      }
#pragma unroll
      for (int j = 0; j < IPT; ++j) {
        const int i = threadIdx.x + j * NT;
        if (i < cnt) {
          s_k[i] = kk[j];
          s_v[i] = vv[j];
        }
      }
    }
    const unsigned prev = base > 0 ? keys[base - 1] : 0u;
    __syncthreads();
    auto prefix = [&](int htot) -> long long {
      return (long long)tile_prefix(state, t, epoch, (unsigned long long)htot, &s_pre);
    };
    const long long end = tile_reduce<NT, IPT>(s_k, s_v, cnt, prev, base == 0, prefix, ykey, yval,
                                               carry_val, carry_idx, t, s_i, s_f, s_fv);
    if (t == ntiles - 1 && threadIdx.x == 0) {
      ctl->ynnz = (int)end;
      ctl->sort_small = 0;
    }
  }
}

__global__ void k_carry_fixup(const float* __restrict__ carry_val, const int* __restrict__ carry_idx,
                              const long long* __restrict__ n_dev, int tile, int small_cap, long long n_cap,
                              float* yval, Ctl* ctl, long long* sig, Gate g) {
  if (gate_shut(g)) return;
  const long long n = *n_dev;
  if (n <= small_cap || n > n_cap) return;
  const long long ntiles = (n + tile - 1) / tile;
  for (long long t = (long long)blockIdx.x * blockDim.x + threadIdx.x; t < ntiles;
       t += (long long)gridDim.x * blockDim.x) {
    int idx, h;
    float s;
    if (!carry_run<long long>(carry_val, carry_idx, nullptr, t, ntiles, idx, s, h)) continue;
    __hip_atomic_store(yval + idx, yval[idx] + s, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
  if (sig) {
    // the results before this launch are visible to it; its own stores are
    // device-coherent and acknowledged before the workgroup's arrival: the
    // last one sends the count (as k_compact does)
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    if (threadIdx.x == 0) {
      unsigned* arrived = &ctl->done[kSlotSort];
      if (__hip_atomic_fetch_add(arrived, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == gridDim.x - 1) {
        __hip_atomic_store(arrived, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        *sig = ctl->ynnz;
      }
    }
  }
}

static int key_bits(int range) {
  int bits = 1;
  while (bits < 32 && (1u << bits) < (unsigned)range) ++bits;
  return bits;
}
static int key_passes(int range) { return (key_bits(range) + 7) / 8; }
int radix_passes(int range) { return key_passes(range); }

// Grid for a launch over n items in tiles of `tile`: exact when the host
// knows n (n_hint >= 0), else the bound n_cap.
static int tiles_grid(long long n_hint, long long n_cap, int tile) {
  const long long n = n_hint >= 0 ? n_hint : n_cap;
  return (int)std::max<long long>(1, (n + tile - 1) / tile);
}

// One counted pass (count, scan, scatter) over *n_dev items; tiles beyond
// the device-side count exit at once. small_cap: passes do nothing when
// n <= small_cap (the single-workgroup path handled them).
static void launch_digit_pass(hipStream_t s, const SortBufs& b, const SortSet& in, const SortSet& out, int shift,
                              int bits, int pass, bool chunks, const long long* n_dev, Ctl* ctl, long long n_hint,
                              long long n_cap, int small_cap, Ep e, Gate g) {
  if (in.w && n_hint >= kWideItems) {
    constexpr int tile = kWideNT * kSortIPT;
    const int tiles = tiles_grid(n_hint, n_cap, tile), pgrid = std::min(tiles, 2048);
    const int sgrid = (int)std::max<long long>(1, (((long long)tiles << bits) + kDScanTile - 1) / kDScanTile);
    hipLaunchKernelGGL((k_digit_count<kSortNT, tile / kSortNT>), dim3(pgrid), dim3(kSortNT), 0, s, in.k, n_dev, shift,
                       bits, b.dcount, nullptr, pass, small_cap, n_cap, g);
    hipLaunchKernelGGL((k_digit_scan<kDScanNT, kDScanIPT>), dim3(sgrid), dim3(kDScanNT), 0, s, b.dcount, n_dev, tile,
                       bits, false, small_cap, n_cap, b.dstate, ctl, e, g);
    hipLaunchKernelGGL((k_sort_scatter<kWideNT, kSortIPT, 2>), dim3(pgrid), dim3(kWideNT), 0, s, in, out, n_dev, shift,
                       bits, b.dcount, nullptr, small_cap, n_cap, g);
    return;
  }
  const int tiles = tiles_grid(n_hint, n_cap, kSortTile);
  const int pgrid = std::min(tiles, 2048);  // count / scatter loop over their tiles
  const int sgrid = (int)std::max<long long>(1, (((long long)tiles << bits) + kDScanTile - 1) / kDScanTile);
  hipLaunchKernelGGL((k_digit_count<kSortNT, kSortIPT>), dim3(pgrid), dim3(kSortNT), 0, s, in.k, n_dev,
                     shift, bits, b.dcount, chunks ? b.dchunk : nullptr, pass, small_cap, n_cap, g);
  if (!chunks || !counts_direct(tiles, bits))
    hipLaunchKernelGGL((k_digit_scan<kDScanNT, kDScanIPT>), dim3(sgrid), dim3(kDScanNT), 0, s, b.dcount,
                       n_dev, kSortTile, bits, chunks, small_cap, n_cap, b.dstate, ctl, e, g);
#define SPMSPV_SCATTER(PAY)                                                                                  \
  hipLaunchKernelGGL((k_sort_scatter<kSortNT, kSortIPT, PAY>), dim3(pgrid), dim3(kSortNT), 0, s, in, out, n_dev, \
                     shift, bits, b.dcount, chunks ? b.dchunk + pass * kChunkWords : nullptr, small_cap, n_cap, g)
  if (in.w) SPMSPV_SCATTER(2);
  else if (in.v) SPMSPV_SCATTER(1);
  else SPMSPV_SCATTER(0);
#undef SPMSPV_SCATTER
}

// The digits of a key of key_bits(range) bits are as equal as they can be:
// 20 bits are 7 + 7 + 6, not 8 + 8 + 4, and 22 are 8 + 7 + 7 (fewer ballots per item and counts per
// tile, longer runs of equal digits to store).
int launch_radix_sets(hipStream_t s, const SortBufs& b, const SortSet& in, const SortSet& out0, const SortSet& out1,
                      int range, const long long* n_dev, Ctl* ctl, long long n_hint, long long n_cap,
                      bool skip_small, Ep ep, Gate g, int small_cap) {
  const int total = key_bits(range), passes = key_passes(range);
  const int last = (passes & 1) ? 0 : 1;
  const SortSet outs[2] = {out0, out1};
  const bool small_known = n_hint >= 0 && n_hint <= small_cap;
  const bool big_known = n_hint > small_cap;
  if (!big_known && !skip_small) {
#define SPMSPV_SMALL(PAY)                                                                                \
  hipLaunchKernelGGL((k_sort_small<kSortNT, kSortIPT, PAY>), dim3(1), dim3(kSortNT), 0, s, in, n_dev, passes, 1, \
                     ctl, nullptr, nullptr, outs[last], small_cap, nullptr, g)
    if (in.w) SPMSPV_SMALL(2);
    else if (in.v) SPMSPV_SMALL(1);
    else SPMSPV_SMALL(0);
#undef SPMSPV_SMALL
  }
  if (small_known) return last;
  for (int p = 0, shift = 0, bits; p < passes; ++p, shift += bits) {
    const Ep e{ep.v + (unsigned)p, ep.dev < 0 ? -1 : ep.dev + p};
    bits = (total - shift + passes - p - 1) / (passes - p);
    launch_digit_pass(s, b, p == 0 ? in : outs[(p - 1) & 1], outs[p & 1], shift, bits, p, passes > 1, n_dev, ctl, n_hint, n_cap,
                      small_cap, e, g);
  }
  return last;
}

static SortSet set_a(const SortBufs& b) { return {b.keyA, reinterpret_cast<unsigned*>(b.valA), nullptr}; }
static SortSet set_b(const SortBufs& b) { return {b.keyB, reinterpret_cast<unsigned*>(b.valB), nullptr}; }

int launch_radix_sort(hipStream_t s, const SortBufs& b, int range, const long long* n_dev, Ctl* ctl,
                      long long n_hint, long long n_cap, bool skip_small, Ep ep, Gate g, int small_cap) {
  const int last = launch_radix_sets(s, b, set_a(b), set_b(b), set_a(b), range, n_dev, ctl, n_hint, n_cap, skip_small,
                                     ep, g, small_cap);
  return last == 0 ? 1 : 0;
}

void launch_sort_reduce(hipStream_t s, const SortBufs& b, int m, Ctl* ctl, int* ykey, float* yval,
                        long long binlen_hint, long long n_cap, Ep ep, Gate g, int small_cap, long long* sig,
                        bool skip_small) {
  const long long* n_dev = &ctl->bin_len;
  const int passes = key_passes(m);
  const bool small_known = binlen_hint >= 0 && binlen_hint <= small_cap;
  if (binlen_hint <= small_cap && !skip_small) {
    hipLaunchKernelGGL((k_sort_small<kSortNT, kSortIPT, 1>), dim3(1), dim3(kSortNT), 0, s, set_a(b), n_dev, passes, 0,
                       ctl, ykey, yval, SortSet{}, small_cap, sig, g);
  }
  if (small_known) return;
  const int fb = launch_radix_sort(s, b, m, n_dev, ctl, binlen_hint, n_cap, true, ep, g, small_cap);
  const unsigned* kf = fb ? b.keyB : b.keyA;
  const float* vf = fb ? b.valB : b.valA;
  const Ep er{ep.v + 4u, ep.dev < 0 ? -1 : ep.dev + 4};
  hipLaunchKernelGGL((k_reduce<kRedNT, kRedIPT>), dim3(tiles_grid(binlen_hint, n_cap, kRedTile)),
                     dim3(kRedNT), 0, s, kf, vf, n_dev, ctl, ykey, yval, b.carry_val, b.carry_idx,
                     b.red_state, er, small_cap, n_cap, g);
  const int fgrid = std::min(2048, std::max(1, tiles_grid(binlen_hint, n_cap, kRedTile) / 256 + 1));
  hipLaunchKernelGGL(k_carry_fixup, dim3(fgrid), dim3(256), 0, s, b.carry_val, b.carry_idx, n_dev,
                     kRedTile, small_cap, n_cap, yval, ctl, sig, g);
}

}  // namespace spmspv
