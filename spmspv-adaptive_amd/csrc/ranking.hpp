// Stable ranking of items by a digit of up to 8 bits inside a wave, by
// ballots: the inner step of every radix sort here.
#pragma once

#include "common.hpp"

namespace spmspv {

// ---------------------------------------------------------------- ranking
// Items of a tile are laid out per wave: wave w owns positions
// [w*64*IPT, (w+1)*64*IPT); item j of lane l sits at w*64*IPT + j*64 + l
// (IPT may be a run-time nj <= IPT: slots j >= nj hold no item). On return
// cnt (this wave's 256 counters) holds the per-digit counts of the wave's
// chunk and rank[j] the stable rank of item j among equal digits inside
// the chunk.
// A digit is `bits` (<= 8) wide, one ballot per bit.
// The ranking is bound by these instructions and their branches: the lane's bit
// spread over a word makes a ballot's agreement one three-input operation per
// half, the first six bits are looked at without a branch (a narrower digit's
// high bits are 0 in every lane, which changes nothing), and a lane without an
// item takes part instead of being masked out. R-MAT scale 19's rows ordered in
// LDS: 331 -> 302 us; a pass over 3.3 M pairs 24.4 -> 21.1. All peers first, then
// the counters: 342 us (registers).
__device__ __forceinline__ uint64_t digit_peers(unsigned d, bool valid, int bits) {
  const uint64_t all = __ballot(valid);
  unsigned lo = (unsigned)all, hi = (unsigned)(all >> 32);
#pragma unroll
  for (int b = 0; b < 8; ++b) {
    if (b >= 6 && b >= bits) break;
    int mine = (int)(d << (31 - b)) >> 31;  // the bit in all 32 places
    asm volatile("" : "+v"(mine));          // (one instruction serves the ballot too)
    const uint64_t bb = __ballot(mine != 0);
    lo &= ~((unsigned)bb ^ (unsigned)mine);
    hi &= ~((unsigned)(bb >> 32) ^ (unsigned)mine);
  }
  return ((uint64_t)hi << 32) | lo;
}

template <int IPT>
__device__ __forceinline__ void wave_rank_digits(const unsigned (&dig)[IPT], const bool (&valid)[IPT], unsigned* cnt,
                                                 int (&rank)[IPT], int nj = IPT, int bits = 8) {
  for (int k = lane(); k < 256; k += kWave) cnt[k] = 0u;
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  const uint64_t lt = lane() == 0 ? 0ull : (~0ull >> (kWave - lane()));
#pragma unroll
  for (int j = 0; j < IPT; ++j) {
    rank[j] = 0;
    if (j >= nj) continue;  // slots past the tile's fill (wave-uniform): no items
    const unsigned d = dig[j];
    const uint64_t peers = digit_peers(d, valid[j], bits);
    // (a lane without an item reads a counter for nothing and is nobody's peer)
    const unsigned base = cnt[d];
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
    rank[j] = (int)base + __popcll(peers & lt);
    if ((peers >> lane()) == 1ull) cnt[d] = base + (unsigned)__popcll(peers);
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
  }
}

// The same on the digit (key >> shift) & (2^bits - 1) of each item, returned
// in dig (0 where there is no item).
template <int IPT>
__device__ __forceinline__ void wave_rank(const unsigned (&key)[IPT], const bool (&valid)[IPT],
                                          int shift, unsigned* cnt, int (&rank)[IPT],
                                          unsigned (&dig)[IPT], int nj = IPT, int bits = 8) {
  const unsigned mask = (1u << bits) - 1u;
#pragma unroll
  for (int j = 0; j < IPT; ++j) dig[j] = j < nj && valid[j] ? ((key[j] >> shift) & mask) : 0u;
  wave_rank_digits<IPT>(dig, valid, cnt, rank, nj, bits);
}

// Converts the per-wave counts into exclusive-over-waves offsets (in place)
// and returns, for digit d = threadIdx.x (NT == 256), the tile total.
template <int NW>
__device__ __forceinline__ unsigned digit_wave_offsets(unsigned* s_cnt) {
  const int d = threadIdx.x;
  unsigned tot = 0;
#pragma unroll
  for (int w = 0; w < NW; ++w) {
    const unsigned c = s_cnt[w * 256 + d];
    s_cnt[w * 256 + d] = tot;
    tot += c;
  }
  return tot;
}

}  // namespace spmspv
