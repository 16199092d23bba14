// Launch interface of the gfx950 kernels. All launches go to the given
// stream and never allocate; sizes that only the device knows (bin_len,
// tile counts) are read by the kernels from the control block.
#pragma once

#include <vector>

#include <hip/hip_runtime.h>

#include "common.hpp"

namespace spmspv {

// Tile geometry (one place, so the arena sizing in the handle agrees).
// Tile of the column scan: a chain of round trips (keys, column bounds, look-
// back), so the tiles are small while the look-back stays short. 105 k keys of
// R-MAT scale 20: 15.1 us with 8 keys per thread, 12.8 with 4, 12.3 with 2; the
// eight levels of a BFS on scale 22 (up to 10^6 keys) 125, 113 and 116 us.
constexpr int kPrepNT = 256, kPrepIPT = 4, kPrepTile = kPrepNT * kPrepIPT;
// The wide tile: the scans of many vectors in one launch, which fill the chip as
// they are (48 vectors of R-MAT scale 20: 29 us with 8 keys per thread, 38 with
// 4), and the no-allocation call, whose fixed scratch holds words per tile.
constexpr int kWideIPT = 8, kWideTile = kPrepNT * kWideIPT;
// odd items per thread: a lane walking VT consecutive LDS words then hits
// a different bank than its neighbours (stride 7 is coprime with 32 banks)
constexpr int kLbNT = 256, kLbVT = 7, kLbTile = kLbNT * kLbVT;
constexpr int kCmpNT = 256;  // bit-array words per compaction tile (8,192 rows, 8 per thread)
constexpr int kSortNT = 256, kSortIPT = 12, kSortTile = kSortNT * kSortIPT;
constexpr int kChunk = 16, kChunkRows = 100;  // tiles of a chunk of the digit counts, chunks at most
constexpr int kDScanNT = 256, kDScanIPT = 8, kDScanTile = kDScanNT * kDScanIPT;
constexpr int kRedNT = 256, kRedIPT = 7, kRedTile = kRedNT * kRedIPT;
constexpr int kRowNT = 256, kRowVT = 7, kRowTile = kRowNT * kRowVT;
// row-merge items per thread the autotuner may pick (odd: conflict-free)
constexpr int kRowVTMin = 5;
constexpr int kSmallSortCap = kSortTile;  // single-workgroup LDS sort + reduce
constexpr int kPersistGrid = 1024;        // workgroups of a persistent launch

// Ticket slots in Ctl (one per persistent kernel kind).
enum Slot { kSlotPrep = 0, kSlotCompact, kSlotHist, kSlotSort, kSlotReduce, kSlotMat, kSlotBfs,
            kSlotBatch, kSlotBucket, kSlotSelect,
            // done[10..11] as one 64-bit word: the compaction's arrivals
            // (high half) and result count (low half)
            kSlotCount = 10 };
constexpr int kSelMaxGrid = 512;  // workgroups of the features-only selector launch

struct MatFeat {  // device-resident matrix features (computeMatFeture_serial)
  double max_row, min_row, avg_row, range, std_row, equality, gini, std_trunc;
  double m, n, nnz;
};

// Device-side switch for work queued before the host knows whether it is
// wanted: a launch whose gate has a word does nothing unless *word == want
// (read as the kernel starts; an earlier launch on the stream wrote it).
struct Gate {
  const int* word = nullptr;
  int want = 0;
};
__device__ __forceinline__ bool gate_shut(const Gate& g) {
  return g.word != nullptr && *g.word != g.want;
}

// --- column path ---------------------------------------------------------
// Column-length gather + exclusive scan + (bin_len, max, min) + merge-path
// splits for the load-balanced gather; when `mlp` is non-null the last
// workgroup also builds the selector features and runs the MLP.
struct SelectorArgs {
  const float* weights;  // NWEIGHTS floats or null
  const MatFeat* mat;
  int mode;              // 0 mlp, 1 tree, 2 fixed
  int fixed;
  long long* stash;      // when set: the selector word of this x (sel_word) is stored here
  // features-only launch for a large x: the selector word may carry the
  // sampled estimate of bin_len (flagged kSelEstimated) instead of the sum
  int estimate;
  // switching-aware choice: with penalty > 0 and prev >= 0, a slot of the
  // previous call's family (column 0-3, row SpMSpV 4-5, SpMV 6-7) whose
  // logit is within penalty of the top one is kept instead of a switch
  int prev;
  float penalty;
  // tuned size rule behind the network: a load-balanced column or row slot
  // (2, 3, 5, 7) becomes the bucket slot (8) when bin_lo <= bin_len <= bin_hi
  // (off by default: bin_hi < bin_lo)
  long long bin_lo = 0, bin_hi = -1;
};
// BFS (bfs.hip): the column scan of a frontier also sends the level's word and
// opens the level: cnt the counters, nxt the frontier's index, sig the words.
struct LevelOpen {
  int* cnt = nullptr;
  int nxt = 0;
  long long* sig = nullptr;
};
// The end of a count in two words over the whole grid: every workgroup's
// thread 0 adds its parts into out[0], out[1] and arrives in out[2] (all 0
// before the launch); the last one sends both words to the host, sig[1] and
// sig[2], then 1 in sig[0]: a polled word where a copy and a stream wait cost
// more (BFS of R-MAT scale 22 457 -> 448 us, 64 sources of scale 18 428 -> 406).
__device__ inline void count_to_host(unsigned long long c, unsigned long long d, unsigned long long* out,
                                     long long* sig) {
  atomicAdd(out, c);
  atomicAdd(out + 1, d);
  // the sums are in place before the arrival
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  if (atomicAdd(out + 2, 1ull) != gridDim.x - 1) return;
  sig[1] = (long long)__hip_atomic_load(out, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  sig[2] = (long long)__hip_atomic_load(out + 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  __hip_atomic_store(sig, 1ll, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}
__host__ __device__ inline int slot_family(int k) { return k < 4 ? 0 : (k < 6 ? 1 : 2); }
// The selector's x inputs for a large x (xnnz > kSampleMin) come from
// kSampleKeys evenly spaced keys (positions floor(i * xnnz / kSampleKeys)):
// bin_len is their column lengths' sum scaled by xnnz / kSampleKeys, and
// max_len their longest column. Every launch that runs the selector uses
// this definition, so training and dispatch see the same features.
constexpr int kSampleMin = 1 << 16, kSampleKeys = 1024;
// {bin_len, kernel choice} in one 64-bit word, so that a single store
// publishes both (no ordering fence); never negative, choice 0xff = none.
// Flag kSelEstimated in the choice byte: bin_len is the sampled estimate.
constexpr int kSelEstimated = 0x40;
// Flag kSelDone: the launch that selected also computed the result (the
// single-launch small-x column path); the bin_len field holds y_nnz. Set
// in ctl->kernel_choice too, where it shuts every gated launch.
constexpr int kSelDone = 0x80;
// Flag kSelGathered: the launch that selected an atomic column slot also did
// its gather (the products are in acc, the rows in marks); the compaction is
// left. Set in ctl->kernel_choice too: a launch gated on the slot alone
// stays shut, a compaction gated on slot and flag runs.
constexpr int kSelGathered = 0x20;
__host__ __device__ inline long long sel_word(long long bin_len, int choice) {
  return (bin_len << 8) | (long long)(choice & 0xff);
}
__host__ __device__ inline long long sel_word_binlen(long long w) { return w >> 8; }
__host__ __device__ inline int sel_word_choice(long long w) {
  const int c = (int)(w & 0xff);
  return c == 0xff ? -1 : (c & 0x1f);
}
__host__ __device__ inline bool sel_word_done(long long w) {
  const int c = (int)(w & 0xff);
  return c != 0xff && (c & kSelDone) != 0;
}
__host__ __device__ inline bool sel_word_gathered(long long w) {
  const int c = (int)(w & 0xff);
  return c != 0xff && (c & kSelGathered) != 0;
}
__host__ __device__ inline bool sel_word_estimated(long long w) {
  const int c = (int)(w & 0xff);
  return c != 0xff && (c & kSelEstimated) != 0;
}
// samp (2 * kSampleKeys / kPrepNT long longs, or null): the first tiles'
// partials of a large x's sampled selector inputs, so that the sampling
// overlaps the scan instead of following the last tile's look-back.
void launch_prep(hipStream_t s, const int* colptr, const int* xkey, int ncols, int xnnz,
                 const int* xnnz_dev, int* ptr, int* xbeg, int* split, unsigned long long* state,
                 int* tile_mm, Ctl* ctl, const SelectorArgs* sel, Ep ep, long long* samp = nullptr,
                 bool wide = false, const LevelOpen& open = {});
// The vectors of a batch: one launch selects for all of them, one scans many
// that need it. Vector v has keys xkey[key0 .. key0 + xnnz), tiles
// [tile0, tile0 + ntiles) of kWideTile keys (at least one) and, once its
// slot is known, its scan from scan0 (xnnz + 1 places) and splits from split0.
struct BatchVec {
  int key0, xnnz, tile0, ntiles;
  int scan0, split0;
};
// Per vector: ctls[v].{bin_len, max_len, xnnz, n_tiles} and the selector word
// (exact bin_len and choice) in stash[v]. tile_vec[t]: vector of tile t;
// tsum / tmax: per tile; arrive[v]: 0 before and after.
void launch_batch_select(hipStream_t s, const int* colptr, const int* xkey, int ncols, int ntiles, const int* tile_vec,
                         const BatchVec* vec, long long* tsum, int* tmax, unsigned* arrive, Ctl* ctls,
                         const SelectorArgs& sel, long long* stash);
// ptr and xbeg (at scan0) and split (at split0) as launch_prep, for the tiles
// listed: list[i] = tile.
void launch_batch_scan(hipStream_t s, const int* colptr, const int* xkey, int ncols, int nlist, const int* list,
                       const int* tile_vec, const BatchVec* vec, const long long* tsum, int* ptr, int* xbeg,
                       int* split);
// Features-only selector: ctl->{bin_len, max_len, min_len, xnnz} of x and,
// with sel.mat set, the selector's choice (and the selector word in
// sel.stash). part: 5 * kSelMaxGrid partials. No column scan. With enc set
// (already all +0.0), x's support encoding is scattered into it as well.
void launch_select_feat(hipStream_t s, const int* colptr, const int* xkey, const float* xval,
                        int ncols, int xnnz, long long* part, Ctl* ctl, const SelectorArgs& sel,
                        float* enc, const int* enc_perm = nullptr);
// mode 0: FP32 atomics into acc + marks; mode 1: (row, a*x) at the product
// index; mode 2: the row keys alone (boolean, cval and xval unread).
void launch_naive_col(hipStream_t s, int mode, const int* colptr, const int* crow, const float* cval,
                      const int* xkey, const float* xval, const int* ptr, int ncols, int xnnz,
                      const int* xnnz_dev, int team, float* acc, unsigned char* marks, int* bkey,
                      float* bval, Gate g = {});
// modes as launch_naive_col.
void launch_lb_gather(hipStream_t s, int mode, const int* ptr, const int* xbeg, const float* xval,
                      const int* split, const int* crow, const float* cval, const Ctl* ctl,
                      int xnnz, const int* xnnz_dev, float* acc, unsigned char* marks, int* bkey,
                      float* bval, long long tiles_hint, Gate g = {});
// Two-layer load balance: tiles of exactly kLbTile products; starts holds
// ceil(bin_len / kLbTile) + 1 ints. mode 0: atomics into acc + marks,
// mode 1: bins at the product index.
void launch_tl_gather(hipStream_t s, int mode, const int* ptr, const int* xbeg, const float* xval, int xnnz,
                      int* starts, const int* crow, const float* cval, const Ctl* ctl, float* acc,
                      unsigned char* marks, int* bkey, float* bval, long long tiles_hint, Gate g = {});
// hits (bit array, or mark bytes when marks != null) -> sorted (key, val);
// clears the hits (and acc entries when reset_acc) so the accumulator
// returns to all-zero. With keymap, hit k is reported as key keymap[k]
// (keymap ascending keeps the keys sorted). With sig (may be host-mapped),
// the result count is also written to *sig once every workgroup's stores
// are visible, as launch_signal_int after this launch would.
// clr (nullable): nclr 64-bit words at a stride of kBinCurStride set to 0 (the
// bucket slot's cursors, once its accumulate kernel has read them).
void launch_compact(hipStream_t s, unsigned* bitmap, unsigned char* marks, int m, float* acc,
                    int reset_acc, int* ykey, float* yval, unsigned long long* state, Ctl* ctl,
                    Ep ep, const int* keymap = nullptr, Gate g = {}, long long* sig = nullptr,
                    unsigned long long* clr = nullptr, int nclr = 0);
// bitmap of (v != 0) over a dense vector (whole words, no atomics)
void launch_bitmap_from_dense(hipStream_t s, const float* v, int n, unsigned* bits);
void launch_fill_f32(hipStream_t s, float* p, long long n, float v, Gate g = {});
// ctl->epoch advanced, for the launches of a captured call (Ep{0, 0 .. 15})
void launch_next_epoch(hipStream_t s, Ctl* ctl, unsigned long long* const (&state)[3], const size_t (&words)[3]);
// *dst = *src once every earlier launch on s has finished (dst may be host-mapped)
void launch_signal_int(hipStream_t s, const int* src, long long* dst, Gate g = {});
void launch_fill_i32(hipStream_t s, int* p, long long n, int v);
// dense[key[i]] = val[i]; with `encode`, a zero value is stored as -0.0
// (the support encoding: +0.0 outside the support, nonzero bits inside).
// With perm, entry k lands at dense[perm[k]].
void launch_scatter(hipStream_t s, const int* key, const float* val, int nnz, const int* nnz_dev,
                    int len, float* dense, bool encode = false, Gate g = {}, const int* perm = nullptr);
// enc[c] = bit c of bits ? (x[c] == 0 ? -0.0 : x[c]) : +0.0, or x[c] without
// bits (at enc[perm[c]] with perm)
void launch_encode_x(hipStream_t s, const float* x, const unsigned* bits, int n, float* enc,
                     const int* perm = nullptr);
void launch_set_bits(hipStream_t s, const int* key, int nnz, const int* nnz_dev, int len,
                     unsigned* bits);
void launch_clear_keys(hipStream_t s, const int* key, int nnz, float* dense, unsigned* bits);

// Single-launch small-x column path (smallx.hip): x of at most kFuseKeys keys
// whose products (bin_len) fit kFuseCap, on at most kFuseRowsMax rows. It also
// writes the column scan (ptr, xbeg, split, ctl) like launch_prep, so a
// call that does not fit goes on with the usual launches (gated on
// ctl->kernel_choice, which gets kSelDone when the launch finished the
// call). In auto mode (sel.mode != 2) a call that fits is reported as
// kFusedSlot, the sort-based slot whose result it computes. With acc set, a
// call that does not fit and whose slot is an atomic one is gathered into acc
// and marks (kSelGathered), up to kFuseGather products per workgroup. Returns
// false (nothing launched) when xnnz or m is larger.
constexpr int kFuseNT = 1024, kFuseKeys = 4096, kFuseCap = kFuseNT * 11;
constexpr int kFuseRowsMax = 1 << 26;  // 512 workgroups of kFuseRows: two rounds of one per CU
constexpr int kFusedSlot = 1;  // SPMSPV_K_COL_NAIVE_SORT
constexpr int kFuseGather = 4096;
// cap (<= kFuseCap): largest bin_len that takes the single launch (the
// autotuner may lower it). state: a look-back word per workgroup.
bool launch_col_fused(hipStream_t s, const int* colptr, const int* crow, const float* cval, const int* xkey,
                      const float* xval, int ncols, int xnnz, int m, int* ptr, int* xbeg, int* split, Ctl* ctl,
                      const SelectorArgs& sel, int* ykey, float* yval, long long* count_sig, int cap,
                      unsigned long long* state, Ep ep, float* acc = nullptr, unsigned char* marks = nullptr);

// --- sort path -----------------------------------------------------------
// Sorts (bkey, bval)[bin_len] by key (< m) with an LSD radix sort
// (onesweep), then reduces equal keys into (ykey, yval) and ctl->ynnz.
// bin_len <= kSmallSortCap takes a single-workgroup LDS path.
struct SortBufs {
  unsigned* keyA;
  float* valA;
  unsigned* keyB;
  float* valB;
  unsigned* dcount;     // 256 per sort tile: per-tile digit counts, then their scan
  unsigned long long* dchunk;     // 4 * kChunkRows * 64: digit counts per kChunk tiles, 0 between sorts but for the last pass's
  unsigned long long* dstate;     // look-back words of the digit-count scan
  unsigned long long* red_state;  // per reduce tile
  float* carry_val;
  int* carry_idx;
};
// Items of a sort: keys and up to two payload words (null: absent).
struct SortSet {
  unsigned* k = nullptr;
  unsigned* v = nullptr;
  unsigned* w = nullptr;
};
// n_hint: item count when the host knows it (exact grids), else -1 and the
// grids cover n_cap; with more items than n_cap nothing is sorted. ep: first of the 5 epochs the sort + reduce use.
// small_cap (<= kSmallSortCap): largest item count that takes the
// single-workgroup path (the autotuner may lower it); skip_small: nothing is
// done for that many. sig: the result count goes there once the results are
// visible (and nothing when nothing is sorted).
void launch_sort_reduce(hipStream_t s, const SortBufs& b, int m, Ctl* ctl, int* ykey, float* yval,
                        long long binlen_hint, long long n_cap, Ep ep, Gate g = {},
                        int small_cap = kSmallSortCap, long long* sig = nullptr, bool skip_small = false);
// Sorts in[*n_dev] by key < range, stable, its passes writing out0 and out1 in
// turn (`in` may be out1, and is not written otherwise); returns which of the
// two holds the result. With ep.dev >= 0 (captured graphs) the passes use
// device epochs ep.dev + pass, otherwise ep.v + pass (4 at most). b gives the
// digit counts' buffers.
int launch_radix_sets(hipStream_t s, const SortBufs& b, const SortSet& in, const SortSet& out0, const SortSet& out1,
                      int range, const long long* n_dev, Ctl* ctl, long long n_hint, long long n_cap,
                      bool skip_small, Ep ep, Gate g = {}, int small_cap = kSmallSortCap);
int radix_passes(int range);  // of a sort by keys < range
// Sorts (keyA, valA)[*n_dev] by key < range; returns 0 if the result is in
// A, 1 if in B. With valA and valB null it sorts the keys alone.
int launch_radix_sort(hipStream_t s, const SortBufs& b, int range, const long long* n_dev, Ctl* ctl,
                      long long n_hint, long long n_cap, bool skip_small, Ep ep, Gate g = {},
                      int small_cap = kSmallSortCap);

// Bucket slot: row bins, ranges of consecutive rows with about equal
// numbers of the matrix's nonzeros (about nnz / 2^bucket_bits each) and at
// most 2^kBinRowBits rows, at most kBinMax of them. Bin b owns the product
// slots [base[b], base[b+1]) of bkey/bval (nnz capacity): the nonzeros of
// its rows, an upper bound on its products. bin_layout computes the layout
// on the host from the row pointer (returns the bin count, or -1 when more
// than kBinMax bins would be needed). Per call the products are scattered
// into their bins and summed per bin in LDS windows into acc (marks set);
// the caller's compaction gives the sorted result and clears acc, marks
// and the cursors (two bins' per 128-byte line; its clr argument). Needs k_prep's
// scan and splits.
constexpr int kBinRowBits = 12, kBinMax = 6144, kBinChunk = 16384, kBinCurStride = 16, kBinTbl = 2048;
struct BinLayout {
  std::vector<int> start;  // first row of each bin, then m
  std::vector<int> base;   // first product slot of each bin, then nnz
  std::vector<int> tbl;    // bin of the first row of each block of 2^tbl_shift rows
  int tbl_shift = 0;
  int max_rows = 1;        // rows of the largest bin
};
struct BinWs {
  unsigned long long* cursor;  // kBinMax / 2 * kBinCurStride: products reserved in bins 2i (low half) and 2i + 1
  int* base;         // kBinMax + 1
  int* start;        // kBinMax + 1
  int* tbl;          // kBinTbl
  int ntbl = 1, tbl_shift = 0;
  int max_rows = 1;
};
int bin_layout(const std::vector<int>& row_ptr, int m, int bucket_bits, BinLayout* out);
// cnt[crow[i]] += 1 for every nonzero (nonzeros per row of a CSC matrix)
void launch_row_counts(hipStream_t s, const int* crow, long long nnz, int* cnt);
void launch_bucket(hipStream_t s, const int* ptr, const int* xbeg, const float* xval, const int* split,
                   const int* crow, const float* cval, const Ctl* ctl, int xnnz, const BinWs& ws, int nbins,
                   unsigned* bkey, float* bval, float* acc, unsigned char* marks, long long tiles_hint,
                   long long binlen_hint, long long binlen_cap, Gate g = {});

// --- row path ------------------------------------------------------------
// --- CSR5 for wave64 (spmv_type 1) ----------------------------------------
struct Csr5 {
  int S = 0;            // items per lane (sigma)
  int n = 0;            // columns
  // new index of every column (most nonzeros first: the gathers of the hot
  // columns then share cache lines), or null when the columns keep their
  // order; ccol holds the new indices and x must be given in that order
  int* cperm = nullptr;
  const int* row_ptr = nullptr;  // the CSR it was built from
  int ntiles = 0;       // tiles of 64 * S items
  int n_ne = 0, n_empty = 0;
  int* ccol = nullptr;  // transposed column indices, ntiles * 64 * S
  float* cval = nullptr;
  unsigned* flags = nullptr;  // one row-start marker word per lane and tile
  unsigned* tinfo = nullptr;  // first non-empty row index | continuation bit
  int* rows_ne = nullptr;     // non-empty rows, ascending
  int* rows_empty = nullptr;  // empty rows, ascending
  int* rank = nullptr;        // rank[r] = non-empty rows before r
  float* y_ne = nullptr;      // per non-empty row results when some rows are empty
  float* carry_val = nullptr;
  int* carry_row = nullptr;
  int* carry_hit = nullptr;
};
// sigma (<= 0: from nonzeros per row) rounded up to an instantiated width
int csr5_sigma_of(int sigma, int m, long long nnz);
size_t csr5_bytes(int m, int n, long long nnz, int S);
// What the column ordering of a CSR5 build may use: the sort buffers (n <=
// their capacity), the control block, a device count word, fresh epochs,
// and the CSC column pointer when there is one (else columns are counted).
struct ColumnOrderArgs {
  SortBufs sb;
  long long sb_cap;
  Ctl* ctl;
  long long* n_dev;
  Ep ep;  // 12 consecutive epochs
  const int* csc_colptr;
};
// cperm[c] = rank of column c by nonzero count (descending, ties by index).
// Returns false (no order) when the sort buffers cannot hold n keys.
bool launch_column_order(hipStream_t s, const ColumnOrderArgs& a, const int* col, int nnz, int n,
                         int* cperm);
// Builds the CSR5 copy of a CSR into `mem` (csr5_bytes); with `order`, the
// columns are renumbered by nonzero count and every row's items put in that
// order (the caller's CSR is untouched); synchronises s.
hipError_t csr5_build(hipStream_t s, const int* row_ptr, const int* col, const float* val, int m,
                      int n, int nnz, int S, void* mem, int* h_pin, const ColumnOrderArgs* order,
                      Csr5* out);
// x as for launch_row_merge (the support encoding with masked or hits, else
// plain), indexed by the copy's column order.
// Without empty rows the results go to y (one mark byte per row with hits).
// With empty rows they go to the non-empty-row space: vals_out = y_ne,
// marks indexed by non-empty row, keymap_out = rows_ne (for the
// compaction), and y is filled only when y_dense_rows (a dense output).
// n_out = entries of that space (m or n_ne).
// ev_begin / ev_end (nullable) are recorded around the tile kernel alone.
// clear (nullable, c.n floats, 16-byte aligned, not x) is set to +0.0 by the
// tile kernel as it runs.
void launch_csr5(hipStream_t s, const Csr5& c, bool masked, bool hits, const float* x,
                 int m, int nnz, float* y, bool y_dense_rows,
                 unsigned char* marks, float** vals_out, const int** keymap_out, int* n_out,
                 hipEvent_t ev_begin = nullptr, hipEvent_t ev_end = nullptr, Gate g = {},
                 float* clear = nullptr);

// Workgroups of `block` threads of `kernel` resident on the whole device
// at once (occupancy x CUs), cached per kernel.
int resident_blocks(const void* kernel, int block);
void launch_row_split(hipStream_t s, const int* row_ptr, int m, int nnz, int* split, int ntiles,
                      int tile);
// vt in {5, 7, 11}: merged items per thread (tile = 256 * vt).
// With masked or hits, x must be the support-encoded vector
// (launch_encode_x / launch_scatter with encode); without either it is plain
// dense x.
void launch_row_merge(hipStream_t s, bool masked, bool hits, const int* row_ptr, const int* col,
                      const float* val, const float* x, int m, int nnz,
                      const int* split, int ntiles, int vt, float* y, unsigned* ybits,
                      float* carry_val, int* carry_row, int* carry_hit,
                      hipEvent_t ev_begin = nullptr, hipEvent_t ev_end = nullptr, Gate g = {});
// val == nullptr and x == nullptr: the boolean form (hit bits into ybits
// only).
void launch_row_naive(hipStream_t s, bool masked, bool hits, const int* row_ptr, const int* col,
                      const float* val, const float* x, const unsigned* xbits, int m, int team,
                      float* y, unsigned* ybits);

// --- CSC construction ----------------------------------------------------
// rowid[j] = row of nonzero j
void launch_expand_rows(hipStream_t s, const int* row_ptr, int m, int nnz, int* rowid);
hipError_t launch_csr_to_csc_sorted(hipStream_t s, const int* row_ptr, const int* col, const float* val,
                              int m, int n, int nnz, int* colptr, int* crow, float* cval,
                              const SortBufs& b, long long* n_dev, Ctl* ctl, Ep ep);

// --- features ------------------------------------------------------------
void launch_mat_features(hipStream_t s, const int* row_ptr, int m, int n, int nnz, int* hist,
                         double* partials, MatFeat* out, Ctl* ctl);

}  // namespace spmspv
