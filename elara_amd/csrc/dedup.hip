// Batch dedup and duplicate-id gradient reduction in a fixed order, optionally fused with row-sparse Adam
// (HBM-bound; no MFMA).
//
// Replaces the step before Adam on every batch: torch.unique(ids, return_inverse=True) (srm2/train.py:352) and
// aten.embedding_dense_backward (srm2/train.py:429), and gives config C3 its fused form (dedup, fixed-order
// segment sum, Adam on each unique row).
//
// Sort.  Stable LSD radix sort of (id, occurrence index) pairs, 8-bit digits, ceil(key_bits / 8) passes (or one
// pass fewer with 9- or 10-bit digits), keys held as uint32 when key_bits <= 32, in tiles of 4096 keys.  A pass is
// per-tile digit histograms, above kSortFoldTiles tiles a launch of a wave per digit scanning that digit's per-tile
// counts, and a scatter in which each key's rank among equal digits of its tile comes from wave ballots (peer mask
// of the digit bits), a per-wave running count in LDS and a scan over the tile's waves, so equal keys keep their
// occurrence order.
//
// Segments.  Sorted position i starts a segment when its key differs from position i-1; per-block head counts, then
// a launch in which each block adds up the counts of the blocks before it (or, above kFoldMaxBlocks blocks, a
// one-block scan launch in between), gives every position its unique index (the inverse), every unique id its
// first position, and lays out the partial chunks of the long segments.
//
// Summation order: ATen's, as torch.ops.aten.embedding_dense_backward computes it on this GPU
// (aten/src/ATen/native/cuda/Embedding.cu embedding_dense_backward_cuda and EmbeddingBackwardKernel.cu, PyTorch
// 2.10 / 2.11; third-party code the reference calls, restated here).  Every id's sum is ((0 + G1) + G2) + ..., G
// the left-to-right sum of one group of that id's occurrences, taken in ascending occurrence index:
//   n <= 3072 indices (embedding_backward_feature_kernel): a group is the id's occurrences inside one window of
//       16 consecutive indices (the kernel's blockDim.y in ATen's ROCm build; 32 in its CUDA build);
//   n >  3072 (embedding_backward_cuda_kernel on a stable sort): groups are the id's occurrences cut into runs of
//       NROWS_PER_THREAD = 10 from its first.
// ATen starts every group sum from zero as well; the total never is -0 (it starts at +0 and a rounded sum is -0
// only when both terms are), so starting a group from its first gradient gives the same bits.  Long (Zipf-hot)
// segments are cut into chunks of 6 groups summed in parallel by different waves (partial sums per group, added in
// order by the segment's own wave).
#include "elr_dir_dev.h"
#include "elr_scan.h"
#include "elr_seg_dev.h"

namespace elr {

// A sort tile is 4,096 keys: 1,024 threads with 4 keys each below kSortBig keys, where a tile's chain of ranking rounds
// and LDS passes is what a launch takes (a pass of 426k keys, the digit counts summed as below: 18 us of histogram and
// scatter, against 25 in three launches with 256 threads of 16 keys), and 256 threads with 16 keys each from there, where
// several tiles per CU hide it (scatters of 3.4M keys: 26 us against 36).
constexpr int kSortTile = 4096;
constexpr int kSortThreadsSmall = 1024;
constexpr int kSortThreadsBig = 256;
constexpr int64_t kSortBig = int64_t(1) << 20;
inline int64_t sort_tiles(int64_t n) { return (n + kSortTile - 1) / kSortTile; }
// Up to this many tiles every scatter block adds up the tiles' digit counts itself; above, a launch of a wave per digit
// scans them (k_radix_hist_scan).  At 104 tiles the scans' launches (4.2 us each) cost more than the sums: a batch of
// 426k ids sorted twice 312 against 303 us, and at 26 tiles 99 against 92 us for the whole duplicate-id update.
constexpr int64_t kSortFoldTiles = 128;
static_assert(kSortFoldTiles * kSortTile <= kSortBig, "the scatters that sum the counts have 1,024 threads");
// Rounds of a segment tile (k_seg_count, k_seg_apply): 8 from 2^20 positions, 4 below, so that a small batch still
// spreads over the chip (k_seg_count and k_seg_apply of 426k positions: 15 us against 20 with 16 rounds; of 3.4M: 33 with 8
// rounds, 34 with 16).
constexpr int kSegItemsBig = 8;
constexpr int kSegItemsSmall = 4;
constexpr int64_t kSegBig = int64_t(1) << 20;
inline int seg_items_for(int64_t n) { return n >= kSegBig ? kSegItemsBig : kSegItemsSmall; }
// LDS of a CU, and what a block's small shared arrays (scans, counters) take beside its large ones, at most.
constexpr size_t kLdsBytes = 160 * 1024, kLdsSlack = 1024;
constexpr int kRadixMaxBits = 10;   // passes take digits of 8, 9 or 10 bits (sort_plan)
constexpr int kRadixMaxBins = 1 << kRadixMaxBits;
constexpr int64_t kAtenSmall = 3072;                      // ATen's windowed path up to this many indices
constexpr int kAtenWinShift = 4;                          // its window: 16 indices
constexpr int64_t kWinHot = 64;                           // windowed segments longer than this are hot (SegFinalSub)
constexpr int kSegParts = 8;                              // run sums a final-kernel wave loads together
constexpr int kSegBlock = 256;

template <int RB, typename Key>
__device__ __forceinline__ uint32_t digit_of(Key k, int shift) {
  return (uint32_t)((k >> shift) & (Key)((1u << RB) - 1));
}

// Passes and digit width of a sort of key_bits-bit keys: one pass fewer than 8-bit digits need when digits of at
// most max_bits bits then suffice (27-bit keys: 3 passes of 9 bits instead of 4 of 8), else 8-bit digits.
inline void sort_plan(int key_bits, int max_bits, int& passes, int& rb) {
  const int p8 = (key_bits + 7) / 8;
  if (p8 > 1) {
    const int w = (key_bits + p8 - 2) / (p8 - 1);
    if (w <= max_bits) {
      passes = p8 - 1;
      rb = w < 8 ? 8 : w;
      return;
    }
  }
  passes = p8;
  rb = 8;
}

// The key of a caller's id.  An id outside [0, lim) takes the key lim, which the sort's digits cover and no valid id
// has (key_lim): digits that cover fewer bits than the whole id would otherwise sort it between the occurrences of a
// valid id, whose segment it would split in two, and a 32-bit key would cut it to a valid id.  lim == 0: every id is
// its own key (elr_unique, elr_dedup_plan: the caller's ids lie in [0, 2^key_bits)).
template <typename Key>
__device__ __forceinline__ Key key_of(int64_t id, uint64_t lim) {
  return lim && (uint64_t)id >= lim ? (Key)lim : (Key)id;
}

// Per-tile histogram of RB-bit digits: digit-major (hist[d * ntile + tile]) for k_radix_hist_scan, tile-major
// (hist[tile * BINS + d]) when the scatter adds the counts up itself (fold).
template <typename Src, typename Key, int RB, int NT>
__global__ __launch_bounds__(NT) void k_radix_hist(const Src* __restrict__ src, int64_t n, uint64_t lim, int shift,
                                                   int32_t* __restrict__ hist, int64_t ntile, int fold) {
  constexpr int BINS = 1 << RB, ITEMS = kSortTile / NT;
  constexpr bool FIRST = std::is_same_v<Src, int64_t>;   // the caller's ids
  __shared__ int h[BINS];
  const int t = threadIdx.x;
  const int64_t base = (int64_t)blockIdx.x * kSortTile;
  Key kk[ITEMS];
#pragma unroll
  for (int r = 0; r < ITEMS; ++r) {
    const int64_t pos = base + r * NT + t;
    const Src x = pos < n ? src[pos] : (Src)0;
    kk[r] = FIRST ? key_of<Key>((int64_t)x, lim) : (Key)x;
  }
  for (int b = t; b < BINS; b += NT) h[b] = 0;
  __syncthreads();
#pragma unroll
  for (int r = 0; r < ITEMS; ++r)
    if (base + r * NT + t < n) atomicAdd(&h[digit_of<RB>(kk[r], shift)], 1);
  __syncthreads();
  for (int b = t; b < BINS; b += NT)
    hist[fold ? (int64_t)blockIdx.x * BINS + b : (int64_t)b * ntile + blockIdx.x] = h[b];
}

// One wave per digit: exclusive scan of that digit's per-tile counts (in place) and the digit's total.  The wave
// loads up to 512 counts (8 per lane) before it scans them, so a few hundred tiles cost one round of loads; no
// block barrier.
constexpr int kHistScanThreads = 256;
__global__ __launch_bounds__(kHistScanThreads) void k_radix_hist_scan(int32_t* __restrict__ hist, int64_t ntile,
                                                                      int nbins, int32_t* __restrict__ dtot) {
  constexpr int kWaves = kHistScanThreads / 64, kPer = 8;
  const int lane = threadIdx.x & 63;
  const int d = blockIdx.x * kWaves + (threadIdx.x >> 6);
  if (d >= nbins) return;
  int32_t* h = hist + (int64_t)d * ntile;
  int carry = 0;   // n < 2^31
  for (int64_t g0 = 0; g0 < ntile; g0 += 64 * kPer) {
    int x[kPer];
#pragma unroll
    for (int k = 0; k < kPer; ++k) {
      const int64_t b = g0 + k * 64 + lane;
      x[k] = b < ntile ? h[b] : 0;
    }
#pragma unroll
    for (int k = 0; k < kPer; ++k) {
      const int64_t b = g0 + k * 64 + lane;
      const int inc = wave_incl_scan<int>(x[k]);
      if (b < ntile) h[b] = carry + inc - x[k];
      carry += __shfl(inc, 63, 64);
    }
  }
  if (lane == 0) dtot[d] = carry;
}

// One block: exclusive scan of per-block counts in place (grids above kFoldMaxBlocks; see k_seg_apply).
__global__ __launch_bounds__(kScanBlock) void k_scan_blocks(int64_t* __restrict__ bsum, int64_t n) {
  scan_channels_block(bsum, n, 1, nullptr);
}

// The lanes of this wave (of those for which valid holds) whose RB-bit digit d equals this lane's.
__device__ __forceinline__ uint64_t digit_peers(uint32_t d, bool valid, int rb) {
  uint64_t m = __ballot(valid);
#pragma unroll
  for (int b = 0; b < rb; ++b) {
    const bool bit = (d >> b) & 1u;
    const uint64_t bal = __ballot(bit);
    m &= bit ? bal : ~bal;
  }
  return m;
}

// Exclusive prefix over values held BPT per thread of an NT-thread block (in thread order): put(j, prefix of x[j]).
template <int NT, int BPT, class Put>
__device__ __forceinline__ void bins_excl_scan(const int (&x)[BPT], Put&& put) {
  int v[1] = {0}, e[1], tot[1];
#pragma unroll
  for (int j = 0; j < BPT; ++j) v[0] += x[j];
  block_excl_scan<NT, 1>(v, e, tot);
#pragma unroll
  for (int j = 0; j < BPT; ++j) {
    put(j, e[0]);
    e[0] += x[j];
  }
}

// Stable scatter of one pass.  FIRST: the source keys are the caller's int64 ids and the values are their
// positions.  Wave w of the block takes the tile's w-th part, 64 consecutive positions per round, so an item's
// rank among the tile's items of its digit is: items of that digit in earlier waves' parts, plus those of its
// own wave's earlier rounds (a per-wave running count in LDS, which only that wave touches, in program order), plus
// its peers in the same round below its lane (ballots).  The waves run their rounds without block barriers; one
// scan over the waves' counts per digit at the end gives the first term.  The tile is then sorted by digit in LDS
// and written out run by run, so consecutive threads write consecutive addresses of one digit's bucket instead of
// 64 scattered ones.  A digit's first position for this tile: the exclusive scan of the digit totals plus the
// earlier tiles' counts, both from the scan launch (offs, dtot) or, with fold, summed here from the tile-major
// histograms.
// (256-thread blocks of 32-bit keys: four waves per SIMD, which their LDS allows, asked of the register allocator too; the
// first pass otherwise takes 129 registers and three waves, 32 us against 27 at 3.4M keys)
template <typename Src, typename Key, bool FIRST, int RB, int NT>
__global__ __launch_bounds__(NT, NT == kSortThreadsBig && sizeof(Key) == 4 ? 4 : 1) void k_radix_scatter(const Src* __restrict__ src_keys,
                                                                const int32_t* __restrict__ src_vals, int64_t n,
                                                                uint64_t lim, int shift, const int32_t* __restrict__ offs,
                                                                const int32_t* __restrict__ dtot, int ntile, int fold,
                                                                Key* __restrict__ dst_keys,
                                                                int32_t* __restrict__ dst_vals) {
  constexpr int TILE = kSortTile, ITEMS = TILE / NT, NW = NT / 64;
  constexpr int BINS = 1 << RB;
  constexpr int G = NT > BINS ? NT / BINS : 1;      // groups of threads that share the tiles' counts (fold)
  constexpr int BPT = BINS > NT ? BINS / NT : 1;    // digits per thread, digit t * BPT + j
  __shared__ int bo[BINS];            // global position of this tile's first item of digit d (n < 2^31)
  __shared__ int lbase[BINS];         // position of digit d's first item in the tile sorted by digit
  __shared__ uint16_t wc[NW][BINS];   // per wave: running count of digit d, then the count in earlier waves
  __shared__ Key lk[TILE];
  __shared__ int32_t lv[TILE];
  static_assert(sizeof(bo) + sizeof(lbase) + sizeof(wc) + sizeof(lk) + sizeof(lv) + kLdsSlack <= kLdsBytes / 2,
                "two blocks per CU");
  const int t = threadIdx.x, w = t >> 6, lane = t & 63;
  const int64_t tile0 = (int64_t)blockIdx.x * TILE, base = tile0 + (int64_t)w * (ITEMS * 64);
  // the tile's items first, so that their loads overlap the digit bases' loads and scan (the ids become keys after it: a
  // use before it would wait for them)
  Src in[ITEMS];
  int32_t vv[ITEMS];
#pragma unroll
  for (int r = 0; r < ITEMS; ++r) {
    const int64_t pos = base + (int64_t)r * 64 + lane;
    const bool valid = pos < n;
    in[r] = valid ? src_keys[pos] : (Src)0;
    vv[r] = valid ? (FIRST ? (int32_t)pos : src_vals[pos]) : 0;
  }
  const bool own = t * BPT < BINS;   // this thread's digits
  int first[BPT], total[BPT];        // their items in earlier tiles and in all tiles
#pragma unroll
  for (int j = 0; j < BPT; ++j) first[j] = total[j] = 0;
  if (NT == kSortThreadsSmall && fold) {
    const int d = t & (BINS - 1), g = t / BINS;
    int* part = lv;   // 2 * NT ints
    static_assert(NT != kSortThreadsSmall || (2 * NT <= TILE && BPT == 1), "the groups' sums fit in the tile's LDS");
    int x0 = 0, x1 = 0;
#pragma unroll 8
    for (int b = g; b < ntile; b += G) {
      const int x = offs[b * BINS + d];
      x0 += b < (int)blockIdx.x ? x : 0;
      x1 += x;
    }
    part[t] = x0;
    part[NT + t] = x1;
    __syncthreads();
    if (own)
#pragma unroll
      for (int q = 0; q < G; ++q) {
        first[0] += part[q * BINS + t];
        total[0] += part[NT + q * BINS + t];
      }
  } else if (own) {
#pragma unroll
    for (int j = 0; j < BPT; ++j) {
      first[j] = offs[(int64_t)(t * BPT + j) * ntile + blockIdx.x];
      total[j] = dtot[t * BPT + j];
    }
  }
  bins_excl_scan<NT, BPT>(total, [&](int j, int ex) {
    if (own) bo[t * BPT + j] = ex + first[j];
  });
  for (int q = t; q < NW * BINS / 2; q += NT) reinterpret_cast<uint32_t*>(&wc[0][0])[q] = 0;
  __syncthreads();
  Key kk[ITEMS];
#pragma unroll
  for (int r = 0; r < ITEMS; ++r) kk[r] = FIRST ? key_of<Key>((int64_t)in[r], lim) : (Key)in[r];
  int rk[ITEMS];
#pragma unroll
  for (int r = 0; r < ITEMS; ++r) {
    const bool valid = base + (int64_t)r * 64 + lane < n;
    const uint32_t d = digit_of<RB>(kk[r], shift);
    const uint64_t m = digit_peers(d, valid, RB);
    const int lr = __popcll(m & lanemask_lt());
    // every lane reads its digit's running count before the group's lowest lane adds the group's size: one wave's
    // LDS accesses take effect in program order
    const int before = valid ? (int)wc[w][d] : 0;
    rk[r] = valid ? before + lr : -1;
    if (valid && lr == 0) wc[w][d] = (uint16_t)(before + __popcll(m));
  }
  __syncthreads();
  {
    // per digit: exclusive scan over the waves, then the tile sorted by digit: digit d's items start at the exclusive
    // scan of the tile's digit counts
    int x[BPT];
#pragma unroll
    for (int j = 0; j < BPT; ++j) {
      x[j] = 0;
      if (own)
#pragma unroll
        for (int q = 0; q < NW; ++q) {
          const int c = wc[q][t * BPT + j];
          wc[q][t * BPT + j] = (uint16_t)x[j];
          x[j] += c;
        }
    }
    bins_excl_scan<NT, BPT>(x, [&](int j, int ex) {
      if (own) lbase[t * BPT + j] = ex;
    });
  }
  __syncthreads();
#pragma unroll
  for (int r = 0; r < ITEMS; ++r) {
    if (rk[r] >= 0) {
      const uint32_t d = digit_of<RB>(kk[r], shift);
      const int lp = lbase[d] + wc[w][d] + rk[r];
      lk[lp] = kk[r];
      lv[lp] = vv[r];
    }
  }
  __syncthreads();
  const int64_t rem = n - tile0;
  const int nvalid = rem < TILE ? (int)rem : TILE;
#pragma unroll
  for (int r = 0; r < ITEMS; ++r) {
    const int j = r * NT + t;
    if (j < nvalid) {
      const Key k = lk[j];
      const uint32_t d = digit_of<RB>(k, shift);
      const int64_t dst = (int64_t)bo[d] + (j - lbase[d]);
      if (dst >= 0 && dst < n) {
        dst_keys[dst] = k;
        dst_vals[dst] = lv[j];
      }
    }
  }
}

// Segment kernels take a tile of kSegBlock * ITEMS positions per block: wave w of the block the tile's w-th quarter,
// ITEMS rounds of 64 consecutive positions.  A position starts a segment (is a head) when its key differs from the one
// before it; a round's heads are one ballot, so positions are ranked with popcounts of the wave's ITEMS masks and the
// block synchronises once, not once per round.
constexpr int kSegWaves = kSegBlock / 64;

// x of lane l, and the block's wave index, as wave-uniform (scalar) values.
__device__ __forceinline__ int lane_value(int x, int l) { return __builtin_amdgcn_readlane(x, l); }
__device__ __forceinline__ int block_wave() { return __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6)); }

// What the sorted keys stand for: ids (PlainKeys), or one field's column after the other, each key an offset in its
// field's rows (FieldKeys, elr_dedup_plan_fields), where a column's first position is a head whatever its key.
struct PlainKeys {
  uint64_t lim;   // as in key_of; the key lim stands for ids that are no row: INT64_MAX, past every row
  template <typename Key>
  __device__ __forceinline__ int64_t id(Key k, int64_t) const {
    return lim && (uint64_t)k == lim ? INT64_MAX : (int64_t)k;
  }
  __device__ __forceinline__ bool starts(int64_t i) const { return i == 0; }
};
constexpr int kFieldMax = 128;   // fields per batch (the bounds travel as a kernel argument)
struct FieldBounds {
  int64_t lo[kFieldMax + 1];
};
struct FieldKeys {
  FieldBounds fb;
  uint32_t nrows;   // positions per column
  __device__ __forceinline__ int64_t id(uint32_t k, int64_t i) const {   // -1: an id outside its field's rows
    const uint32_t c = (uint32_t)i / nrows;
    const int64_t lo = fb.lo[c], R = fb.lo[c + 1] - lo;
    return (int64_t)k == R ? -1 : lo + (int64_t)k;
  }
  __device__ __forceinline__ bool starts(int64_t i) const { return (uint32_t)i % nrows == 0; }
};

// The wave's keys of sorted positions p0 + r * 64 + lane, and each round's head mask.
template <typename Key, int ITEMS, class Keys>
__device__ __forceinline__ void seg_heads(const Keys& keys, const Key* __restrict__ sk, int64_t p0, int64_t n,
                                          Key (&kk)[ITEMS], uint64_t (&hm)[ITEMS]) {
  const int lane = threadIdx.x & 63;
#pragma unroll
  for (int r = 0; r < ITEMS; ++r) {
    const int64_t i = p0 + r * 64 + lane;
    kk[r] = i < n ? sk[i] : (Key)0;
  }
  Key prev = p0 > 0 && p0 < n ? sk[p0 - 1] : (Key)0;   // the key before the round
#pragma unroll
  for (int r = 0; r < ITEMS; ++r) {
    const int64_t i = p0 + r * 64 + lane;
    Key left = __shfl_up(kk[r], 1, 64);
    if (lane == 0) left = prev;
    hm[r] = __builtin_amdgcn_ballot_w64(i < n && (keys.starts(i) || kk[r] != left));
    prev = __shfl(kk[r], 63, 64);
  }
}

// Segment heads: per-block head counts and first head position (n when the tile has none).  Also clears the counts
// that k_seg_apply's chunk plan adds to.
template <typename Key, int ITEMS, class Keys>
__global__ __launch_bounds__(kSegBlock) void k_seg_count(Keys keys, const Key* __restrict__ sk, int64_t n,
                                                         int64_t* __restrict__ bsum, int32_t* __restrict__ bfirst,
                                                         int64_t* __restrict__ d_E, int64_t* __restrict__ d_hot) {
  __shared__ int wcnt[kSegWaves];
  __shared__ int wfirst[kSegWaves];
  const int w = block_wave();
  const int64_t p0 = ((int64_t)blockIdx.x * kSegWaves + w) * (64 * ITEMS);
  Key kk[ITEMS];
  uint64_t hm[ITEMS];
  seg_heads<Key, ITEMS, Keys>(keys, sk, p0, n, kk, hm);
  int c = 0;
  int first = (int)n;
#pragma unroll
  for (int r = ITEMS - 1; r >= 0; --r) {
    c += __builtin_popcountll(hm[r]);
    if (hm[r]) first = (int)p0 + r * 64 + __builtin_ctzll(hm[r]);
  }
  if ((threadIdx.x & 63) == 0) {
    wcnt[w] = c;
    wfirst[w] = first;
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    int t = 0;
    int f = (int)n;
    for (int v = 0; v < kSegWaves; ++v) {
      t += wcnt[v];
      f = wfirst[v] < f ? wfirst[v] : f;
    }
    bsum[blockIdx.x] = t;
    bfirst[blockIdx.x] = f;
    if (blockIdx.x == 0) {
      *d_E = 0;
      *d_hot = 0;
    }
  }
}

// Grids of at most this many blocks take their block offsets by block_offset (a block reads at most 8 counts per
// thread); larger ones from a one-block scan launch (k_scan_blocks) between the count and apply launches (4.5 us; at
// config C3's 1,664 blocks the sums in the blocks save 3 us).
constexpr int64_t kFoldMaxBlocks = 2048;

// Sum of cnt[0 .. b) over the whole block, returned to every thread: the offset of block b from the per-block
// counts of the launch before, without a scan launch in between.
__device__ __forceinline__ int64_t block_offset(const int64_t* __restrict__ cnt, int64_t b) {
  __shared__ int64_t wpart[kSegBlock / 64];
  int64_t x = 0;
  for (int64_t i = threadIdx.x; i < b; i += kSegBlock) x += cnt[i];
#pragma unroll
  for (int d = 32; d >= 1; d >>= 1) x += __shfl_xor(x, d, 64);
  if ((threadIdx.x & 63) == 0) wpart[threadIdx.x >> 6] = x;
  __syncthreads();
  int64_t t = 0;
#pragma unroll
  for (int q = 0; q < kSegBlock / 64; ++q) t += wpart[q];
  return t;
}

// Sort path.  A segment of more than kHotLen occurrences is hot: the partial-chunk kernel sums all of its runs (its
// first chunk included) and one block of the final kernel folds the run sums, its four waves loading together.  Any
// other segment folds its first chunk in the final kernel's wave, and only its later chunks are partial chunks.
__device__ __forceinline__ int part_chunks(int64_t L) {
  return (int)(seg_hot(L) ? (L + kSegChunk - 1) / kSegChunk : (L - 1) / kSegChunk);
}

// Segment heads: unique ids, segment starts, each segment's first occurrence index and the inverse, and (hot_list not
// NULL) the segments of more than hot_len occurrences in hot_list[0 .. *d_hot) and, with chunk_off, the partial-chunk
// plan: chunk_off[u] = first work item of segment u's partial chunks, for the segments that have any, and
// chunk_seg[item] = u.  The block's first segment index
// is the sum of the earlier blocks' head counts (k_seg_count), or, with `scanned`, bcnt[block] after k_scan_blocks.
// The last block stores U to d_U (and n_unique) and seg_start[U] = n.
//
// A segment's length, which decides its chunks, is the distance to the next head: in its round's mask, in a later
// round's or wave's, or in a later tile (bfirst).  The work items of a block's chunks are reserved with one atomic
// add, so their order over the segments is not fixed; no sum depends on it (each group sum has its own parts row).
// One launch in place of three (heads with a block scan per round, chunk counts, chunk plan): 33 us against 20 + 8 +
// 24 and two scan launches of 4.6 at config C3's 3.4M positions, 11 against 16 + 7 + 23 at C5's 426k.
template <typename Key, int ITEMS, class Keys>
__global__ __launch_bounds__(kSegBlock) void k_seg_apply(Keys keys, const Key* __restrict__ sk,
                                                         const int32_t* __restrict__ sv, int64_t n, const int64_t* __restrict__ bcnt, int scanned,
                                                         const int32_t* __restrict__ bfirst,
                                                         int64_t* __restrict__ d_U, int64_t* __restrict__ n_unique,
                                                         int64_t* __restrict__ uniq, int64_t* __restrict__ seg_start,
                                                         int32_t* __restrict__ seg_occ0,
                                                         int64_t* __restrict__ inverse,
                                                         int32_t* __restrict__ chunk_off,
                                                         int32_t* __restrict__ chunk_seg,
                                                         int32_t* __restrict__ hot_list, int hot_len,
                                                         int64_t* __restrict__ d_hot, int64_t* __restrict__ d_E) {
  __shared__ int wcnt[kSegWaves], wext[kSegWaves], whot[kSegWaves];
  __shared__ int wfirst[kSegWaves];
  __shared__ int64_t res[2];
  const int lane = threadIdx.x & 63, w = block_wave();
  const int64_t nblk = gridDim.x, p0 = ((int64_t)blockIdx.x * kSegWaves + w) * (64 * ITEMS);
  Key kk[ITEMS];
  int32_t vv[ITEMS];
  uint64_t hm[ITEMS];
#pragma unroll
  for (int r = 0; r < ITEMS; ++r) {
    const int64_t i = p0 + r * 64 + lane;
    vv[r] = i < n ? sv[i] : -1;
  }
  seg_heads<Key, ITEMS, Keys>(keys, sk, p0, n, kk, hm);
  // the first head past this tile (n: none)
  int nxt = (int)n;
  for (int64_t b0 = (int64_t)blockIdx.x + 1; b0 < nblk; b0 += 64) {
    const int f = b0 + lane < nblk ? bfirst[b0 + lane] : (int)n;
    const uint64_t m = __builtin_amdgcn_ballot_w64(f < n);
    if (m) {
      nxt = lane_value(f, __builtin_ctzll(m));
      break;
    }
  }
  int c = 0;
  int first = (int)n;
#pragma unroll
  for (int r = ITEMS - 1; r >= 0; --r) {
    c += __builtin_popcountll(hm[r]);
    if (hm[r]) first = (int)p0 + r * 64 + __builtin_ctzll(hm[r]);
  }
  if (lane == 0) {
    wcnt[w] = c;
    wfirst[w] = first;
  }
  const int64_t before = scanned ? bcnt[blockIdx.x] : block_offset(bcnt, blockIdx.x);
  __syncthreads();
  int64_t run = before, tot = before;   // heads before this wave, and through this block
#pragma unroll
  for (int v = 0; v < kSegWaves; ++v) {
    run += v < w ? wcnt[v] : 0;
    tot += wcnt[v];
  }
#pragma unroll
  for (int v = kSegWaves - 1; v >= 0; --v)
    if (v > w && wfirst[v] < n) nxt = __builtin_amdgcn_readfirstlane(wfirst[v]);
  if (blockIdx.x == nblk - 1 && threadIdx.x == 0) {
    *d_U = tot;
    if (n_unique) *n_unique = tot;
    seg_start[tot] = n;
  }
  // the segments and the inverse; the lengths of this wave's segments, last round first
  int64_t end = run + c;      // segments through the round
  int ext = 0, hot = 0;       // this lane's partial chunks and hot segments
  uint32_t has = 0;           // rounds with a hot segment or one of more than one chunk (wave-uniform)
  int after[ITEMS];           // first head past each round
#pragma unroll
  for (int r = ITEMS - 1; r >= 0; --r) {
    const int64_t i = p0 + r * 64 + lane;
    const uint64_t m = hm[r];
    const bool head = (m >> lane) & 1;
    const int64_t u0 = end - __builtin_popcountll(m);   // segments before the round
    const int64_t u = u0 + __builtin_popcountll(m & lanemask_lt()) + (head ? 0 : -1);
    after[r] = nxt;
    if (head) {
      uniq[u] = keys.id(kk[r], i);
      seg_start[u] = i;
      seg_occ0[u] = vv[r];
    }
    if (inverse && vv[r] >= 0 && vv[r] < n) inverse[vv[r]] = u;
    if (hot_list) {
      const uint64_t up = lane == 63 ? 0ull : m >> (lane + 1);
      const int64_t L = head ? (up ? (int64_t)__builtin_ctzll(up) + 1 : (int64_t)nxt - i) : 1;
      const int e = chunk_off ? part_chunks(L) : 0;
      ext += e;
      hot += L > hot_len ? 1 : 0;
      has |= __builtin_amdgcn_ballot_w64(e > 0 || L > hot_len) ? 1u << r : 0u;
    }
    if (m) nxt = (int)p0 + r * 64 + __builtin_ctzll(m);
    end = u0;
  }
  if (!hot_list) return;
#pragma unroll
  for (int d = 32; d >= 1; d >>= 1) {
    ext += __shfl_xor(ext, d, 64);
    hot += __shfl_xor(hot, d, 64);
  }
  if (lane == 0) {
    wext[w] = ext;
    whot[w] = hot;
  }
  __syncthreads();
  if (threadIdx.x < 2) {
    int64_t x = 0;
    for (int v = 0; v < kSegWaves; ++v) x += threadIdx.x ? whot[v] : wext[v];
    res[threadIdx.x] = x ? (int64_t)atomicAdd(reinterpret_cast<unsigned long long*>(threadIdx.x ? d_hot : d_E),
                                              (unsigned long long)x)
                         : 0;
  }
  __syncthreads();
  if (!has) return;
  int64_t eat = res[0], hat = res[1];
  for (int v = 0; v < w; ++v) {
    eat += wext[v];
    hat += whot[v];
  }
  end = run + c;
#pragma unroll
  for (int r = ITEMS - 1; r >= 0; --r) {
    const uint64_t m = hm[r];
    const int64_t u0 = end - __builtin_popcountll(m);
    end = u0;
    if (!((has >> r) & 1u)) continue;
    const int64_t i = p0 + r * 64 + lane;
    const bool head = (m >> lane) & 1;
    const int32_t u = (int32_t)(u0 + __builtin_popcountll(m & lanemask_lt()));
    const uint64_t up = lane == 63 ? 0ull : m >> (lane + 1);
    const int64_t L = head ? (up ? (int64_t)__builtin_ctzll(up) + 1 : (int64_t)after[r] - i) : 1;
    const int e = chunk_off ? part_chunks(L) : 0, inc = wave_incl_scan<int>(e);
    if (e > 0) chunk_off[u] = (int32_t)(eat + inc - e);
    // the wave writes each segment's work items together (a hot segment has thousands)
    for (uint64_t q = __builtin_amdgcn_ballot_w64(e > 0); q; q &= q - 1) {
      const int l = __builtin_ctzll(q);
      const int qe = lane_value(e, l), qu = lane_value(u, l);
      const int64_t qo = eat + lane_value(inc - e, l);
      for (int k = lane; k < qe; k += 64) chunk_seg[qo + k] = qu;
    }
    eat += lane_value(inc, 63);
    const uint64_t hb = __builtin_amdgcn_ballot_w64(L > hot_len);
    if (L > hot_len) hot_list[hat + __builtin_popcountll(hb & lanemask_lt())] = u;
    hat += __builtin_popcountll(hb);
  }
}

// ---- dedup plan of a batch laid out by field -------------------------------------------------------------------
// A batch of nrows samples x nf fields in (sample, field) order, field c holding rows [lo[c], lo[c + 1]) of the
// table with the bounds ascending: every id of field c is below every id of field c + 1, so the stable sort of the
// whole batch is field 0's column sorted stably, then field 1's, and so on (within a column, sample order is
// occurrence order).  One block per field sorts its column of at most kFieldRows ids in LDS: LSD passes of at most
// kFieldDigit bits over the id's offset in its field, each key ranked as in k_radix_scatter (ballots, a running
// count per wave, a scan over the waves), the column re-read from LDS after each pass.  The segments and chunks then
// come from the general path's two launches (k_seg_count, k_seg_apply with FieldKeys), so the plan is the general
// path's, bit for bit, in four launches.  A thread holds as many keys as the column needs (1 to 16).  (The
// segments by one block per field, as the sort's, took 28 us of a 26-column batch of 426k; the two launches over
// the whole GPU 18, and the whole plan, beside a step's kernels, 104 -> 76.)  An id outside its field's rows takes
// the key R_c (the field's row count), sorts after the field's ids and comes out as -1 in uniq: a row out of range
// for the caller.
constexpr int kFieldThreads = 1024;
constexpr int kFieldItems = 16;
constexpr int64_t kFieldRows = (int64_t)kFieldThreads * kFieldItems;   // samples per batch: the row index is 16-bit
constexpr int kFieldDigit = 9;
constexpr int64_t kFieldSpanMax = (int64_t(1) << 31) - 2;   // rows per field: keys 0 .. R_c fit in 31 bits

// Passes and digit width for keys of `bits` bits, or in [0, span]: ceil(bits / kFieldDigit) passes of equal width.
__host__ __device__ __forceinline__ void digits_for(int bits, int& passes, int& rb) {
  passes = (bits + kFieldDigit - 1) / kFieldDigit;
  rb = (bits + passes - 1) / passes;
}
__device__ __forceinline__ void field_digits(int64_t span, int& passes, int& rb) {
  int bits = 1;
  while (bits < 31 && (int64_t(1) << bits) <= span) ++bits;
  digits_for(bits, passes, rb);
}

// A stable sort of at most kFieldThreads * ITEMS keys by one block in LDS: thread t of wave w holds items
// (w * ITEMS + r) * 64 + lane in kk[r] and ends with the sorted keys of those positions; the result is each sorted
// key's item index.  LSD passes of rb-bit digits, each key ranked as in k_radix_scatter (ballots, a running count per
// wave, a scan over the waves).  s.lk holds the sorted keys too.
template <typename Key, int ITEMS>
struct BlockSort {
  static constexpr int N = kFieldThreads * ITEMS, BINS = 1 << kFieldDigit, NW = kFieldThreads / 64;
  Key lk[N + 1];
  uint16_t lv[2][N];      // pass p writes lv[p & 1]
  uint16_t wc[NW][BINS];  // per wave: running count of digit d, then the count in earlier waves
  int lbase[BINS];
  int wtot[NW];
};

template <typename Key, int ITEMS>
__device__ __forceinline__ const uint16_t* block_sort(BlockSort<Key, ITEMS>& s, Key (&kk)[ITEMS], int n, int passes,
                                                      int rb) {
  constexpr int NW = kFieldThreads / 64, WSPAN = ITEMS * 64;
  static_assert(sizeof(BlockSort<Key, ITEMS>) + kLdsSlack <= kLdsBytes, "one block per CU");
  const int t = threadIdx.x, w = t >> 6, lane = t & 63;
  const int nbins = 1 << rb;
  const uint32_t mask = (uint32_t)nbins - 1u;
  for (int p = 0; p < passes; ++p) {
    const int shift = p * rb;
    const uint16_t* vsrc = s.lv[(p + 1) & 1];
    uint16_t* vdst = s.lv[p & 1];
    if (t < nbins)
#pragma unroll
      for (int q = 0; q < NW; ++q) s.wc[q][t] = 0;
    __syncthreads();
    int rk[ITEMS];
#pragma unroll
    for (int r = 0; r < ITEMS; ++r) {
      const bool valid = w * WSPAN + r * 64 + lane < n;
      const uint32_t d = (uint32_t)(kk[r] >> shift) & mask;
      uint64_t m = __ballot(valid);
      for (int b = 0; b < rb; ++b) {
        const bool bit = (d >> b) & 1u;
        const uint64_t bal = __ballot(bit);
        m &= bit ? bal : ~bal;
      }
      const int lr = __popcll(m & lanemask_lt());
      // one wave's LDS accesses take effect in program order: every lane reads the count before the lowest lane of
      // its digit group adds the group's size
      const int before = valid ? (int)s.wc[w][d] : 0;
      rk[r] = valid ? before + lr : -1;
      if (valid && lr == 0) s.wc[w][d] = (uint16_t)(before + __popcll(m));
    }
    __syncthreads();
    int run = 0;
    if (t < nbins)
#pragma unroll
      for (int q = 0; q < NW; ++q) {
        const int x = s.wc[q][t];
        s.wc[q][t] = (uint16_t)run;
        run += x;
      }
    {
      int v[1] = {run}, ex[1], tot[1];
      block_excl_scan<kFieldThreads, 1>(v, ex, tot);
      if (t < nbins) s.lbase[t] = ex[0];
    }
    __syncthreads();
#pragma unroll
    for (int r = 0; r < ITEMS; ++r)
      if (rk[r] >= 0) {
        const int j = w * WSPAN + r * 64 + lane;
        const uint32_t d = (uint32_t)(kk[r] >> shift) & mask;
        const int lp = s.lbase[d] + s.wc[w][d] + rk[r];
        s.lk[lp] = kk[r];
        vdst[lp] = p == 0 ? (uint16_t)j : vsrc[j];
      }
    __syncthreads();
    // (unconditional: items past n hold anything, and a load under a condition per item makes the compiler keep the
    // array as one 16-register value and spill it around every branch)
#pragma unroll
    for (int r = 0; r < ITEMS; ++r) kk[r] = s.lk[w * WSPAN + r * 64 + lane];
  }
  return s.lv[(passes - 1) & 1];
}

// Each field's ids as offsets in its field (the key R_c for an id outside it), field after field: keys[c * nrows + j].
// One block per field and kFieldKeyRows samples, so that the gather of a column (each wave's 64 loads touch 64
// different cache lines) is spread over the whole GPU instead of being done by the field's sorting block alone.
constexpr int kFieldKeyRows = 1024;
__global__ __launch_bounds__(256) void k_field_keys(const int64_t* __restrict__ ids, int64_t nrows, int nf,
                                                    FieldBounds fb, uint32_t* __restrict__ keys) {
  const int c = blockIdx.y;
  const int64_t lo = fb.lo[c], hi = fb.lo[c + 1];
  const int64_t j0 = (int64_t)blockIdx.x * kFieldKeyRows;
#pragma unroll
  for (int r = 0; r < kFieldKeyRows / 256; ++r) {
    const int64_t j = j0 + r * 256 + threadIdx.x;
    if (j < nrows) {
      const int64_t id = ids[j * nf + c];
      keys[(int64_t)c * nrows + j] = id >= lo && id < hi ? (uint32_t)(id - lo) : (uint32_t)(hi - lo);
    }
  }
}

// Each field's column sorted by one block (ITEMS keys per thread): skeys, and the occurrence index of each position.
template <int ITEMS>
__global__ __launch_bounds__(kFieldThreads) void k_field_sort(const uint32_t* __restrict__ keys, int64_t nrows,
                                                              int nf, FieldBounds fb, uint32_t* __restrict__ skeys,
                                                              int32_t* __restrict__ svals) {
  __shared__ BlockSort<uint32_t, ITEMS> s;
  const int c = blockIdx.x, w = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int n = (int)nrows;
  int passes, rb;
  field_digits(fb.lo[c + 1] - fb.lo[c], passes, rb);
  uint32_t kk[ITEMS];
#pragma unroll
  for (int r = 0; r < ITEMS; ++r) {
    const int j = (w * ITEMS + r) * 64 + lane;
    kk[r] = keys[(int64_t)c * nrows + (j < n ? j : 0)];
  }
  const uint16_t* vfin = block_sort<uint32_t, ITEMS>(s, kk, n, passes, rb);
  const int64_t out0 = (int64_t)c * nrows;
#pragma unroll
  for (int r = 0; r < ITEMS; ++r) {
    const int j = (w * ITEMS + r) * 64 + lane;
    if (j < n) {
      skeys[out0 + j] = kk[r];
      svals[out0 + j] = (int32_t)vfin[j] * nf + c;
    }
  }
}

// The whole dedup plan of at most kFieldThreads * ITEMS ids by one block: the sort in LDS, the segment heads from
// ballots, the inverse, the hot segments and the partial-chunk plan -- what the radix passes, k_seg_count and
// k_seg_apply leave, in one launch.  Against the general path's ten launches of 2 to 5 us each, every one waiting for
// the one before, one block's passes over LDS are the shorter chain: 12.8 us at 2,600 ids, and the whole update of a
// batch of 2,600 36.4 -> 18.0 us.  The line: whole updates of 7,800 ids 40.0 -> 35.1 and of 8,000 ids 58 -> 43 us by
// this kernel, its time growing with the ids while the general path's barely does.
constexpr int kSmallItems = 8;
constexpr int64_t kSmallPlan = kFieldThreads * kSmallItems;
template <typename Key, int ITEMS>
__global__ __launch_bounds__(kFieldThreads) void k_small_plan(const int64_t* __restrict__ ids, int n,
                                                              PlainKeys keys, int passes, int rb,
                                                              int32_t* __restrict__ svals, int64_t* __restrict__ d_tot,
                                                              int64_t* __restrict__ n_unique,
                                                              int64_t* __restrict__ uniq,
                                                              int64_t* __restrict__ seg_start,
                                                              int32_t* __restrict__ seg_occ0,
                                                              int64_t* __restrict__ inverse,
                                                              int32_t* __restrict__ chunk_off,
                                                              int32_t* __restrict__ chunk_seg,
                                                              int32_t* __restrict__ hot_list, int hot_len) {
  constexpr int NW = kFieldThreads / 64;
  __shared__ BlockSort<Key, ITEMS> s;
  __shared__ int wfirst[NW], ecnt, hcnt;
  const int t = threadIdx.x, w = block_wave(), lane = t & 63;
  Key kk[ITEMS];
#pragma unroll
  for (int r = 0; r < ITEMS; ++r) {
    const int j = (w * ITEMS + r) * 64 + lane;
    kk[r] = key_of<Key>(ids[j < n ? j : 0], keys.lim);
  }
  if (t == 0) ecnt = hcnt = 0;
  const uint16_t* vfin = block_sort<Key, ITEMS>(s, kk, n, passes, rb);
  uint64_t hm[ITEMS];
  int c = 0, first = n;
#pragma unroll
  for (int r = ITEMS - 1; r >= 0; --r) {
    const int j = (w * ITEMS + r) * 64 + lane;
    hm[r] = __builtin_amdgcn_ballot_w64(j < n && (j == 0 || s.lk[j > 0 ? j - 1 : 0] != kk[r]));
    c += __builtin_popcountll(hm[r]);
    if (hm[r]) first = (w * ITEMS + r) * 64 + __builtin_ctzll(hm[r]);
  }
  if (lane == 0) {
    s.wtot[w] = c;
    wfirst[w] = first;
  }
  __syncthreads();
  int run = 0, U = 0, nxt = n;
#pragma unroll
  for (int q = 0; q < NW; ++q) {
    run += q < w ? s.wtot[q] : 0;
    U += s.wtot[q];
  }
#pragma unroll
  for (int q = NW - 1; q >= 0; --q)
    if (q > w && wfirst[q] < n) nxt = wfirst[q];
  int end = run + c;
#pragma unroll
  for (int r = ITEMS - 1; r >= 0; --r) {
    const int j = (w * ITEMS + r) * 64 + lane;
    const uint64_t m = hm[r];
    const bool head = (m >> lane) & 1;
    const int u0 = end - __builtin_popcountll(m), u = u0 + __builtin_popcountll(m & lanemask_lt()) + (head ? 0 : -1);
    end = u0;
    if (j < n) {
      const int o = vfin[j];
      svals[j] = o;
      if (inverse) inverse[o] = u;
      if (head) {
        uniq[u] = keys.id(kk[r], j);
        seg_start[u] = j;
        seg_occ0[u] = o;
        if (hot_list) {
          const uint64_t up = lane == 63 ? 0ull : m >> (lane + 1);
          const int L = up ? (int)__builtin_ctzll(up) + 1 : nxt - j;
          const int e = chunk_off ? part_chunks(L) : 0;
          if (e > 0) {
            const int off = atomicAdd(&ecnt, e);
            chunk_off[u] = off;
            for (int k = 0; k < e; ++k) chunk_seg[off + k] = u;
          }
          if (L > hot_len) hot_list[atomicAdd(&hcnt, 1)] = u;
        }
      }
    }
    if (m) nxt = (w * ITEMS + r) * 64 + __builtin_ctzll(m);
  }
  __syncthreads();
  if (t == 0) {
    d_tot[0] = U;
    d_tot[1] = ecnt;
    d_tot[2] = hcnt;
    if (n_unique) *n_unique = U;
    seg_start[U] = n;
  }
}

// Does occurrence k of a segment (occurrence index o, previous one prev) start a new group?  Sort path
// (win_shift == 0): every kAtenGroup occurrences; windowed path: when its index window differs from the previous
// occurrence's.  Wave-uniform (all arguments are).
__device__ __forceinline__ bool group_head(int64_t k, int32_t o, int32_t prev, int win_shift) {
  return k == 0 || (win_shift ? (o >> win_shift) != (prev >> win_shift) : k % kAtenGroup == 0);
}

// Folds the gradients at sorted positions [p0, p1) (p1 - p0 <= 64), occurrences k0.. of their segment, into the
// open group acc and the segment total tot (this lane's NQ elements j = lane + 64 q < D).  Occurrence indices are
// loaded once per wave and broadcast with readlane; prev carries the previous occurrence index across calls.
template <int NQ>
__device__ __forceinline__ void fold_range(const float* __restrict__ grad, int64_t D, const int32_t* __restrict__ sv,
                                           int64_t p0, int64_t p1, int64_t k0, int win_shift, int32_t& prev,
                                           float (&acc)[NQ], float (&tot)[NQ]) {
  const int lane = threadIdx.x & 63;
  const int len = (int)(p1 - p0);
  const int32_t my = lane < len ? sv[p0 + lane] : 0;
  constexpr int UN = 8;
  for (int b0 = 0; b0 < len; b0 += UN) {
    float g[UN][NQ];
#pragma unroll
    for (int u = 0; u < UN; ++u) {
      if (b0 + u < len) {
        const int64_t o = (int64_t)__builtin_amdgcn_readlane(my, b0 + u);
        const float* row = grad + o * D;
#pragma unroll
        for (int q = 0; q < NQ; ++q) {
          const int64_t j = lane + 64 * q;
          g[u][q] = j < D ? __builtin_nontemporal_load(row + j) : 0.0f;
        }
      }
    }
#pragma unroll
    for (int u = 0; u < UN; ++u) {
      if (b0 + u < len) {
        const int32_t o = __builtin_amdgcn_readlane(my, b0 + u);
        const int64_t k = k0 + b0 + u;
        if (group_head(k, o, prev, win_shift)) {
#pragma unroll
          for (int q = 0; q < NQ; ++q) {
            if (k) tot[q] = tot[q] + acc[q];
            acc[q] = g[u][q];
          }
        } else {
#pragma unroll
          for (int q = 0; q < NQ; ++q) acc[q] = acc[q] + g[u][q];
        }
        prev = o;
      }
    }
  }
}

// The group sums of a segment's partial chunks are consecutive parts rows from chunk_off[u] * kGroupsPerChunk (every
// partial chunk but the last is full): ceil(L / kAtenGroup) of them for a hot segment, else
// ceil((L - kSegChunk) / kAtenGroup).  inline_len: the occurrences the segment's own wave folds.
__device__ __forceinline__ int64_t seg_parts(int64_t L, int win_shift) {
  if (win_shift) return 0;
  if (seg_hot(L)) return (L + kAtenGroup - 1) / kAtenGroup;
  return L <= kSegChunk ? 0 : (L - kSegChunk + kAtenGroup - 1) / kAtenGroup;
}
__device__ __forceinline__ int64_t inline_len(int64_t L, int win_shift) {
  if (win_shift) return L;
  return seg_hot(L) ? 0 : (L < kSegChunk ? L : kSegChunk);
}

// Final per-segment sum (the inline part -- the first chunk, or the whole segment on the windowed path -- then the
// extra chunks' group sums in order), then either written to out[uniq[u]] (MODE 0) or applied as an Adam step to
// state[uniq[u]] (MODE 1).  One wave per segment.
template <int NQ, int MODE>
__global__ __launch_bounds__(256) void k_seg_final(const float* __restrict__ grad, int64_t D,
                                                   const int32_t* __restrict__ sv,
                                                   const int64_t* __restrict__ seg_start,
                                                   const int64_t* __restrict__ uniq,
                                                   const int32_t* __restrict__ chunk_off,
                                                   const float* __restrict__ parts, const int64_t* __restrict__ d_U,
                                                   int win_shift, float* __restrict__ out, int64_t nrows,
                                                   AdamScalars s) {
  const int lane = threadIdx.x & 63;
  const int64_t U = *d_U;
  for (int64_t u = wave_id(); u < U; u += wave_count()) {
    const int64_t s0 = seg_start[u], s1 = seg_start[u + 1];
    const int64_t L = s1 - s0;
    const int64_t row = uniq ? uniq[u] : u;   // NULL: segment u goes to row u
    const int64_t inl = inline_len(L, win_shift);
    float acc[NQ], tot[NQ];
#pragma unroll
    for (int q = 0; q < NQ; ++q) acc[q] = tot[q] = 0.0f;
    int32_t prev = 0;
    for (int64_t b0 = 0; b0 < inl; b0 += 64)
      fold_range<NQ>(grad, D, sv, s0 + b0, s0 + (inl - b0 < 64 ? inl : b0 + 64), b0, win_shift, prev, acc, tot);
#pragma unroll
    for (int q = 0; q < NQ; ++q) tot[q] = tot[q] + acc[q];
    const int64_t np = seg_parts(L, win_shift);
    const float* pr = np ? parts + (int64_t)chunk_off[u] * kGroupsPerChunk * D : parts;
    constexpr int PB = 8;
    for (int64_t c0 = 0; c0 < np; c0 += PB) {
      float pc[PB][NQ];
#pragma unroll
      for (int e = 0; e < PB; ++e)
        if (c0 + e < np) {
#pragma unroll
          for (int q = 0; q < NQ; ++q) {
            const int64_t j = lane + 64 * q;
            pc[e][q] = j < D ? pr[(c0 + e) * D + j] : 0.0f;
          }
        }
#pragma unroll
      for (int e = 0; e < PB; ++e)
        if (c0 + e < np) {
#pragma unroll
          for (int q = 0; q < NQ; ++q) tot[q] = tot[q] + pc[e][q];
        }
    }
    if (row < 0 || row >= nrows) continue;
    if (MODE == 0) {
#pragma unroll
      for (int q = 0; q < NQ; ++q) {
        const int64_t j = lane + 64 * q;
        if (j < D) out[row * D + j] = tot[q];
      }
    } else {
      float* rec = out + row * 3 * D;
#pragma unroll
      for (int q = 0; q < NQ; ++q) {
        const int64_t j = lane + 64 * q;
        if (j < D) {
          float w = rec[j], m = rec[D + j], v = rec[2 * D + j];
          adam_elem(w, m, v, tot[q], s);
          rec[j] = w;
          rec[D + j] = m;
          rec[2 * D + j] = v;
        }
      }
    }
  }
}

// The final sums (and Adam, MODE 1) in the chunk layout (elr_rowio.h): LPR lanes per segment, 64 / LPR segments per
// wave, WIN: ATen's windowed order.  A one-occurrence segment, the common case, costs two dependent round trips (its
// metadata; its gradient row and state), and a longer one two more per kSubRows occurrences.  The first hot_blocks
// blocks take the segments of hot_list, one each at a time: the whole block loads the run sums (windowed: the
// gradients) into LDS, kSubStage floats of them, and one group adds them in order.  Against a wave per segment with
// 4 bytes a lane: 24 us against 37 at 107k occurrences, 40k segments of width 48 (most of it the dependent round trips of the
// 60-occurrence segments: 12 without them).
template <int NC>
constexpr int kSubRows = NC == 1 ? kAtenGroup : kAtenGroup / 2;
constexpr int kSubStage = 4096;   // floats: 16 KB, so that LDS leaves the wave count alone
template <int LPR, int NC, int MODE, bool WIN>
struct SegFinalSub {
  const float* grad;
  int64_t D;
  const int32_t* sv;
  const int64_t* seg_start;
  const int32_t* seg_occ0;
  const int64_t* uniq;
  const int32_t* chunk_off;
  const float* parts;
  const int64_t* d_U;
  int64_t u_base;
  const int32_t* hot_list;
  const int64_t* d_hot;
  int64_t hot_blocks;
  float* out;
  int64_t nrows;
  AdamScalars s;
  __device__ void operator()(int64_t block, int64_t nblocks) const;
  __device__ void hot(int64_t block) const;
  __device__ __forceinline__ void emit(int64_t row, int l, int nchunk, const RowFrag<4 * NC>& tot) const;
};

template <int LPR, int NC, int MODE, bool WIN>
__device__ __forceinline__ void SegFinalSub<LPR, NC, MODE, WIN>::emit(int64_t row, int l, int nchunk,
                                                                      const RowFrag<4 * NC>& tot) const {
  if (MODE == 0) {
    chunk_store<LPR, NC>(out + row * D, l, nchunk, tot);
  } else {
    float* rec = out + row * 3 * D;
    RowFrag<4 * NC> w = chunk_load<LPR, NC, false>(rec, l, nchunk),
                  m = chunk_load<LPR, NC, false>(rec + D, l, nchunk),
                  v = chunk_load<LPR, NC, false>(rec + 2 * D, l, nchunk);
    frag_adam<4 * NC>(w, m, v, tot, s);
    chunk_store<LPR, NC>(rec, l, nchunk, w);
    chunk_store<LPR, NC>(rec + D, l, nchunk, m);
    chunk_store<LPR, NC>(rec + 2 * D, l, nchunk, v);
  }
}

// A staging area's rows are loaded into registers while the one before is added, the row indices of the one after (WIN)
// with them, and the adding lanes read UN rows from LDS before the first addition: a row costs neither a round trip to
// memory nor one to LDS.  3,000 occurrences of one id in the windowed order, whole update: 413 -> 264 us at width 48,
// 489 -> 286 at 128, 1,262 -> 468 at 512 (each row read from LDS on its own, each staging area loaded between two
// barriers), against 344, 417 and 905 for one wave that loads 8 rows together.
template <int LPR, int NC, int MODE, bool WIN>
__device__ void SegFinalSub<LPR, NC, MODE, WIN>::hot(int64_t block) const {
  constexpr int NL = kSubStage / 4 / 256;   // chunks of a staging area per thread
  constexpr int UN = 8 / NC;
  __shared__ f32x4 stage[kSubStage / 4];
  __shared__ int32_t win[WIN ? kSubStage / 4 : 1];   // windowed: the staged rows' windows
  const int64_t nh = *d_hot;
  if (block >= nh) return;
  const int t = threadIdx.x, nchunk = (int)(D / 4), per = (kSubStage / 4) / nchunk;
  int rr[NL], cc[NL];   // this thread's chunks of a staging area: row and chunk (rr == per: none)
#pragma unroll
  for (int e = 0; e < NL; ++e) {
    const int q = t + e * 256;
    rr[e] = q / nchunk < per ? q / nchunk : per;
    cc[e] = q % nchunk;
  }
  for (int64_t h = block; h < nh; h += hot_blocks) {
    const int64_t u = hot_list[h], s0 = seg_start[u], L = seg_start[u + 1] - s0;
    const int64_t nr = WIN ? L : (L + kAtenGroup - 1) / kAtenGroup;   // rows to add: gradients, or run sums
    const f32x4* src = reinterpret_cast<const f32x4*>(
        WIN ? grad : parts + (int64_t)chunk_off[u] * kGroupsPerChunk * D);
    RowFrag<4 * NC> tot = frag_zero<4 * NC>(), acc = tot;
    int32_t prev = -1;
    int32_t ix[NL];    // rows of the staging area loaded next (rows past the last: the last)
    int32_t wn[NL];    // windows of the rows in x
    f32x4 x[NL];
    auto index = [&](int64_t r0) {
#pragma unroll
      for (int e = 0; e < NL; ++e) {
        const int64_t r = r0 + rr[e] < nr ? r0 + rr[e] : nr - 1;
        ix[e] = WIN ? sv[s0 + r] : (int32_t)r;
      }
    };
    auto load = [&] {
#pragma unroll
      for (int e = 0; e < NL; ++e) {
        x[e] = src[(int64_t)ix[e] * nchunk + cc[e]];
        wn[e] = ix[e] >> kAtenWinShift;
      }
    };
    index(0);
    load();
    index(per);
    for (int64_t r0 = 0; r0 < nr; r0 += per) {
      const int m = (int)(nr - r0 < per ? nr - r0 : per);
      __syncthreads();
#pragma unroll
      for (int e = 0; e < NL; ++e)
        if (rr[e] < m) {
          stage[rr[e] * nchunk + cc[e]] = x[e];
          if (WIN && cc[e] == 0) win[rr[e]] = wn[e];
        }
      __syncthreads();
      if (r0 + per < nr) {   // (block-uniform)
        load();
        index(r0 + 2 * per);
      }
      if (t < LPR) {
        for (int r = 0; r < m; r += UN) {
          RowFrag<4 * NC> y[UN];
          int32_t yw[UN];
#pragma unroll
          for (int i = 0; i < UN; ++i) {
            const int ri = r + i < m ? r + i : r;
            yw[i] = WIN ? __builtin_amdgcn_readfirstlane(win[ri]) : 0;
#pragma unroll
            for (int c = 0; c < NC; ++c) {
              const f32x4 g = stage[ri * nchunk + (t + c * LPR < nchunk ? t + c * LPR : 0)];
#pragma unroll
              for (int j = 0; j < 4; ++j) y[i].v[4 * c + j] = g[j];
            }
          }
#pragma unroll
          for (int i = 0; i < UN; ++i) {
            if (r + i >= m) continue;
            if (!WIN) {
              frag_add<4 * NC>(tot, y[i]);
            } else if (yw[i] != prev) {
              if (prev >= 0) frag_add<4 * NC>(tot, acc);
              acc = y[i];
              prev = yw[i];
            } else {
              frag_add<4 * NC>(acc, y[i]);
            }
          }
        }
      }
    }
    if (t < LPR) {
      if (WIN) frag_add<4 * NC>(tot, acc);
      const int64_t row = uniq ? uniq[u] : u;
      if (row >= 0 && row < nrows) emit(row, t, nchunk, tot);
    }
  }
}

template <int LPR, int NC, int MODE, bool WIN>
__device__ void SegFinalSub<LPR, NC, MODE, WIN>::operator()(int64_t block, int64_t) const {
  if (block < hot_blocks) {
    hot(block);
    return;
  }
  constexpr int GPW = 64 / LPR;
  const int lane = threadIdx.x & 63, l = lane & (LPR - 1);
  const int nchunk = (int)(D / 4);
  const int64_t u = u_base + ((block - hot_blocks) * 4 + (threadIdx.x >> 6)) * GPW + lane / LPR;
  if (u >= *d_U) return;
  const int64_t s0 = seg_start[u], L = seg_start[u + 1] - s0;
  const int64_t row = uniq ? uniq[u] : u;   // NULL: segment u goes to row u
  const int32_t o0 = seg_occ0[u];
  if (row < 0 || row >= nrows || (WIN ? L > kWinHot : seg_hot(L))) return;   // hot segments: a block's
  RowFrag<4 * NC> acc = chunk_load<LPR, NC, true>(grad + (int64_t)o0 * D, l, nchunk);
  float* rec = out + row * 3 * D;
  RowFrag<4 * NC> w, m, v;
  if (MODE == 1) {
    w = chunk_load<LPR, NC, false>(rec, l, nchunk);
    m = chunk_load<LPR, NC, false>(rec + D, l, nchunk);
    v = chunk_load<LPR, NC, false>(rec + 2 * D, l, nchunk);
  }
  const int inl = (int)(WIN ? L : (L < kSegChunk ? L : kSegChunk));
  RowFrag<4 * NC> tot = frag_zero<4 * NC>();
  int32_t prev = o0;
  int in_run = 1;   // occurrences of the open run (sort path)
  constexpr int R = kSubRows<NC>;
  int32_t o[R];
#pragma unroll
  for (int e = 0; e < R; ++e) o[e] = sv[s0 + (1 + e < inl ? 1 + e : 0)];
  for (int k0 = 1; k0 < inl; k0 += R) {
    // this batch's rows, then the next batch's indices, so that a batch costs one round trip
    RowFrag<4 * NC> g[R];
    int32_t on[R];
#pragma unroll
    for (int e = 0; e < R; ++e) g[e] = chunk_load<LPR, NC, true>(grad + (int64_t)o[e] * D, l, nchunk);
#pragma unroll
    for (int e = 0; e < R; ++e) on[e] = sv[s0 + (k0 + R + e < inl ? k0 + R + e : 0)];
#pragma unroll
    for (int e = 0; e < R; ++e) {
      if (k0 + e >= inl) continue;
      const bool head = WIN ? (o[e] >> kAtenWinShift) != (prev >> kAtenWinShift) : in_run == kAtenGroup;
      if (head) {
        frag_add<4 * NC>(tot, acc);
        acc = g[e];
        in_run = 1;
      } else {
        frag_add<4 * NC>(acc, g[e]);
        ++in_run;
      }
      prev = o[e];
    }
#pragma unroll
    for (int e = 0; e < R; ++e) o[e] = on[e];
  }
  frag_add<4 * NC>(tot, acc);
  if (!WIN && L > kSegChunk) {
    const int np = (int)((L - kSegChunk + kAtenGroup - 1) / kAtenGroup);
    const float* pr = parts + (int64_t)chunk_off[u] * kGroupsPerChunk * D;
    for (int c0 = 0; c0 < np; c0 += kSubRows<NC>) {
      RowFrag<4 * NC> pc[kSubRows<NC>];
#pragma unroll
      for (int e = 0; e < kSubRows<NC>; ++e)
        pc[e] = chunk_load<LPR, NC, false>(pr + (int64_t)(c0 + e < np ? c0 + e : c0) * D, l, nchunk);
#pragma unroll
      for (int e = 0; e < kSubRows<NC>; ++e)
        if (c0 + e < np) frag_add<4 * NC>(tot, pc[e]);
    }
  }
  if (MODE == 0) {
    chunk_store<LPR, NC>(out + row * D, l, nchunk, tot);
  } else {
    frag_adam<4 * NC>(w, m, v, tot, s);
    chunk_store<LPR, NC>(rec, l, nchunk, w);
    chunk_store<LPR, NC>(rec + D, l, nchunk, m);
    chunk_store<LPR, NC>(rec + 2 * D, l, nchunk, v);
  }
}

// Wave-per-row form of k_seg_final for D = 64*VPL (lane l holds floats [l*VPL, l*VPL + VPL)): no grid-stride
// loop, each wave owns kSegPerWave consecutive segments starting at u_base + wave * kSegPerWave; waves past U exit.
// All per-segment metadata (bounds, row id, first occurrence) are scalar loads issued together, then the first
// gradient row, the row's w, m, v (MODE 1) and the next 63 occurrence indices load in parallel: a one-occurrence
// segment -- the common case -- costs two dependent memory round trips.
constexpr int kSegPerWave = 2;

// The result of one segment: written to out[row] (MODE 0) or applied as an Adam step to state row `row` (MODE 1).
template <int VPL, int MODE>
__device__ __forceinline__ void seg_emit(float* __restrict__ out, int64_t row, const RowFrag<VPL>& sum,
                                         const AdamScalars& s) {
  constexpr int64_t D = 64 * VPL;
  const int lane = threadIdx.x & 63;
  if (MODE == 0) {
    frag_store<VPL>(out + row * D + lane * VPL, sum);
  } else {
    float* rec = out + row * 3 * D + lane * VPL;
    RowFrag<VPL> w = frag_load<VPL, false>(rec), m = frag_load<VPL, false>(rec + D),
                 v = frag_load<VPL, false>(rec + 2 * D);
    frag_adam<VPL>(w, m, v, sum, s);
    frag_store<VPL>(rec, w);
    frag_store<VPL>(rec + D, m);
    frag_store<VPL>(rec + 2 * D, v);
  }
}

// Hot segments, one block each (grid-stride over hot_list by hot_blocks blocks): the total is
// ((0 + G1) + G2) + ... over the segment's ceil(L / 10) run sums, consecutive parts rows.  The four waves load
// 4 * PB run sums together; then wave 0, 1, 2, 3 in turn adds its PB of them to the running total, which passes
// from wave to wave through LDS, so the additions keep their order.  Every loop bound is block-uniform.
template <int VPL, int MODE>
__device__ __forceinline__ void seg_hot_block(const int64_t* __restrict__ seg_start,
                                              const int64_t* __restrict__ uniq,
                                              const int32_t* __restrict__ chunk_off,
                                              const float* __restrict__ parts,
                                              const int32_t* __restrict__ hot_list, const int64_t* __restrict__ d_hot,
                                              int64_t hot_blocks, float* __restrict__ out, int64_t nrows,
                                              const AdamScalars& s, float* __restrict__ relay, int64_t block) {
  constexpr int64_t D = 64 * VPL;
  constexpr int PB = VPL <= 2 ? kSegParts : kSegParts / 2;
  constexpr int NWV = 4;
  const int lane = threadIdx.x & 63;
  const int wv = threadIdx.x >> 6;
  const int64_t nh = *d_hot;
  for (int64_t h = block; h < nh; h += hot_blocks) {
    const int64_t u = hot_list[h];
    const int64_t L = seg_start[u + 1] - seg_start[u];
    const int64_t nr = (L + kAtenGroup - 1) / kAtenGroup;
    const float* pr = parts + (int64_t)chunk_off[u] * kGroupsPerChunk * D + lane * VPL;
    for (int64_t i0 = 0; i0 < nr; i0 += NWV * PB) {
      const int64_t mine = i0 + wv * PB;
      RowFrag<VPL> pc[PB];
#pragma unroll
      for (int e = 0; e < PB; ++e)
        if (mine + e < nr) pc[e] = frag_load<VPL, false>(pr + (mine + e) * D);
      for (int w = 0; w < NWV; ++w) {
        if (wv == w && mine < nr) {
          RowFrag<VPL> tot;
          if (mine == 0) {
            tot = frag_zero<VPL>();
          } else {
#pragma unroll
            for (int j = 0; j < VPL; ++j) tot.v[j] = relay[lane * VPL + j];
          }
#pragma unroll
          for (int e = 0; e < PB; ++e)
            if (mine + e < nr) {
#pragma unroll
              for (int j = 0; j < VPL; ++j) tot.v[j] = tot.v[j] + pc[e].v[j];
            }
#pragma unroll
          for (int j = 0; j < VPL; ++j) relay[lane * VPL + j] = tot.v[j];
        }
        __syncthreads();
      }
    }
    if (wv == 0) {
      const int64_t row = uniq ? uniq[u] : u;
      if (row >= 0 && row < nrows) {
        RowFrag<VPL> tot;
#pragma unroll
        for (int j = 0; j < VPL; ++j) tot.v[j] = relay[lane * VPL + j];
        seg_emit<VPL, MODE>(out, row, tot, s);
      }
    }
    __syncthreads();   // the relay is reused by the block's next hot segment
  }
}

// The final kernel as a functor (elr_launch.h): block `block` of the launch, the first hot_blocks of them on the hot
// segments.  k_seg_final_wpr launches it on its own; the device-driven step also runs it beside the directory's
// first launch of the executor (k_run2).
template <int VPL, int MODE>
struct SegFinalWpr {
  const float* grad;
  const int32_t* sv;
  const int64_t* seg_start;
  const int32_t* seg_occ0;
  const int64_t* uniq;
  const int32_t* chunk_off;
  const float* parts;
  const int64_t* d_U;
  int64_t u_base;
  const int32_t* hot_list;
  const int64_t* d_hot;
  int64_t hot_blocks;
  float* out;
  int64_t nrows;
  AdamScalars s;
  __device__ void operator()(int64_t block, int64_t nblocks) const;
};

template <int VPL, int MODE>
__device__ void SegFinalWpr<VPL, MODE>::operator()(int64_t block, int64_t) const {
  constexpr int64_t D = 64 * VPL;
  constexpr int SW = kSegPerWave;
  __shared__ float relay[D];
  if (block < hot_blocks) {
    seg_hot_block<VPL, MODE>(seg_start, uniq, chunk_off, parts, hot_list, d_hot, hot_blocks, out, nrows, s, relay,
                             block);
    return;
  }
  const int lane = threadIdx.x & 63;
  const int64_t U = *d_U;
  const int64_t u0 = u_base + ((block - hot_blocks) * 4 + (threadIdx.x >> 6)) * SW;
  if (u0 >= U) return;
  int64_t s0[SW], len[SW], row[SW], o0[SW];
  bool ok[SW];
#pragma unroll
  for (int q = 0; q < SW; ++q) {
    const int64_t u = u0 + q;
    ok[q] = u < U;
    s0[q] = ok[q] ? seg_start[u] : 0;
    len[q] = ok[q] ? seg_start[u + 1] - s0[q] : 0;
    row[q] = ok[q] ? (uniq ? uniq[u] : u) : -1;   // NULL: segment u goes to row u
    o0[q] = ok[q] ? (int64_t)seg_occ0[u] : 0;
    ok[q] = ok[q] && row[q] >= 0 && row[q] < nrows && !seg_hot(len[q]);   // hot segments: a block's
  }
  RowFrag<VPL> w[SW], m[SW], v[SW], acc[SW];
  int32_t my[SW];
  // short: every segment of the wave fits one run of at most FB occurrences (wave-uniform: the lengths are scalar
  // loads).  Their remaining rows then load together, all segments' at once, before any addition.
  constexpr int FB = VPL <= 2 ? kAtenGroup : 4;
  bool short_segs = true;
#pragma unroll
  for (int q = 0; q < SW; ++q) {
    short_segs = short_segs && (!ok[q] || len[q] <= FB);
    if (!ok[q]) continue;
    acc[q] = frag_load<VPL, true>(grad + o0[q] * D + lane * VPL);
    if (MODE == 1) {
      const float* rec = out + row[q] * 3 * D + lane * VPL;
      w[q] = frag_load<VPL, false>(rec);
      m[q] = frag_load<VPL, false>(rec + D);
      v[q] = frag_load<VPL, false>(rec + 2 * D);
    }
    my[q] = (lane >= 1 && lane < len[q]) ? sv[s0[q] + lane] : 0;
  }
  if (short_segs) {
    // the same additions as the general loop below for one run: ((first + g1) + g2) + ..., then +0 + run
    RowFrag<VPL> g[SW][FB - 1];
#pragma unroll
    for (int q = 0; q < SW; ++q)
#pragma unroll
      for (int e = 1; e < FB; ++e)
        if (ok[q] && e < len[q]) {
          const int64_t o = (int64_t)__builtin_amdgcn_readlane(my[q], e);
          g[q][e - 1] = frag_load<VPL, true>(grad + o * D + lane * VPL);
        }
#pragma unroll
    for (int q = 0; q < SW; ++q) {
      if (!ok[q]) continue;
      RowFrag<VPL> run = acc[q];
#pragma unroll
      for (int e = 1; e < FB; ++e)
        if (e < len[q]) {
#pragma unroll
          for (int j = 0; j < VPL; ++j) run.v[j] = run.v[j] + g[q][e - 1].v[j];
        }
#pragma unroll
      for (int j = 0; j < VPL; ++j) acc[q].v[j] = 0.0f + run.v[j];
    }
  }
#pragma unroll
  for (int q = 0; q < SW; ++q) {
    if (!ok[q] || short_segs) continue;
    // the first chunk folds here, run by run (runs of kAtenGroup from the segment's first occurrence, which is
    // already in acc); then the later chunks' run sums, kSegParts at a time
    const int inl = (int)(len[q] < kSegChunk ? len[q] : kSegChunk);
    RowFrag<VPL> tot = frag_zero<VPL>();
    constexpr int RB = VPL <= 2 ? kAtenGroup : kAtenGroup / 2;   // rows of a run loaded together
    constexpr int PB = VPL <= 2 ? kSegParts : kSegParts / 2;     // run sums loaded together
    for (int r0 = 0; r0 < inl; r0 += kAtenGroup) {
      const int rl = inl - r0 < kAtenGroup ? inl - r0 : kAtenGroup;
      RowFrag<VPL> run = acc[q];
      for (int h = 0; h < rl; h += RB) {
        RowFrag<VPL> g[RB];
#pragma unroll
        for (int e = 0; e < RB; ++e)
          if (h + e < rl && r0 + h + e > 0) {
            const int64_t o = (int64_t)__builtin_amdgcn_readlane(my[q], r0 + h + e);
            g[e] = frag_load<VPL, true>(grad + o * D + lane * VPL);
          }
#pragma unroll
        for (int e = 0; e < RB; ++e) {
          if (h + e >= rl) continue;
          if (h + e == 0) {
            if (r0 > 0) run = g[e];   // run 0 starts from the preloaded first gradient
          } else {
#pragma unroll
            for (int j = 0; j < VPL; ++j) run.v[j] = run.v[j] + g[e].v[j];
          }
        }
      }
#pragma unroll
      for (int j = 0; j < VPL; ++j) tot.v[j] = tot.v[j] + run.v[j];
    }
    const int64_t np = seg_parts(len[q], 0);
    if (np) {
      const float* pr = parts + (int64_t)chunk_off[u0 + q] * kGroupsPerChunk * D + lane * VPL;
      for (int64_t c0 = 0; c0 < np; c0 += PB) {
        RowFrag<VPL> pc[PB];
#pragma unroll
        for (int e = 0; e < PB; ++e)
          if (c0 + e < np) pc[e] = frag_load<VPL, false>(pr + (c0 + e) * D);
#pragma unroll
        for (int e = 0; e < PB; ++e)
          if (c0 + e < np) {
#pragma unroll
            for (int j = 0; j < VPL; ++j) tot.v[j] = tot.v[j] + pc[e].v[j];
          }
      }
    }
    acc[q] = tot;
  }
#pragma unroll
  for (int q = 0; q < SW; ++q) {
    if (!ok[q]) continue;
    if (MODE == 0) {
      frag_store<VPL>(out + row[q] * D + lane * VPL, acc[q]);
    } else {
      frag_adam<VPL>(w[q], m[q], v[q], acc[q], s);
      float* rec = out + row[q] * 3 * D + lane * VPL;
      frag_store<VPL>(rec, w[q]);
      frag_store<VPL>(rec + D, m[q]);
      frag_store<VPL>(rec + 2 * D, v[q]);
    }
  }
}

template <int VPL, int MODE>
__global__ __launch_bounds__(256) void k_seg_final_wpr(SegFinalWpr<VPL, MODE> f) {
  f((int64_t)blockIdx.x, (int64_t)gridDim.x);
}

// ---- host side -------------------------------------------------------------------------------------------------
inline int64_t al256(int64_t b) { return (b + 255) & ~int64_t(255); }

// ATen's windowed order applies up to kAtenSmall indices: returns the window's shift there, 0 on the sort path.
inline int win_shift_for(int64_t n) { return n <= kAtenSmall ? kAtenWinShift : 0; }
// Bound of the hot segments of n occurrences (and the blocks that take them).
inline int64_t hot_max(int64_t n) { return n / (win_shift_for(n) ? kWinHot : kHotLen) + 1; }

// Scratch carve-up for n occurrences of width D.
struct DedupScratch {
  void* keys[2];
  int32_t* vals[2];
  int32_t* hist;      // [kRadixMaxBins * ntile] digit counts per sort tile (sort_tiles)
  int32_t* dtot;      // [kRadixMaxBins] digit totals
  int64_t* bsum;      // [n / (kSegBlock * seg_items_for(n)) + 1] heads per segment tile
  int32_t* bfirst;    // the same count: each tile's first head
  int64_t* d_tot;     // [3]: U, E (partial chunks), hot segments
  int64_t* uniq;      // [n]
  int64_t* seg_start; // [n + 1]
  int32_t* seg_occ0;  // [n] first occurrence index of each segment
  int32_t* chunk_off; // [n]
  int32_t* chunk_seg; // [nch]: n / kSegChunk + n / kHotLen + 2 bounds the partial chunks
  float* parts;       // [nch * kGroupsPerChunk * D] group sums of the partial chunks
  int32_t* hot_list;  // [hot_max(n)] hot segments
};

// (the segment tiles' counts, at most kSegPerSort tiles per sort tile, fit beside the digit counts)
constexpr int64_t kSegPerSort = kSortTile / (kSegBlock * kSegItemsSmall);
static_assert(kSegPerSort * 12 <= kRadixMaxBins * 4, "shared scratch");

inline int64_t dedup_scratch_bytes(int64_t n, int64_t D, DedupScratch* out, void* base) {
  const int64_t ntile = sort_tiles(n), nblk = cdiv(n, kSegBlock * seg_items_for(n));
  const int64_t nch = n / kSegChunk + n / kHotLen + 2;
  int64_t o = 0;
  char* b = (char*)base;
  auto take = [&](int64_t bytes) {
    void* p = b ? (void*)(b + o) : nullptr;
    o += al256(bytes);
    return p;
  };
  DedupScratch s;
  s.keys[0] = take(n * 8);
  s.keys[1] = take(n * 8);
  s.vals[0] = (int32_t*)take(n * 4);
  s.vals[1] = (int32_t*)take(n * 4);
  // the digit counts (the first half), then the segment tiles' counts; the digit totals (the first half).  The halves
  // that nothing reads, and the unused region, keep every n's scratch size, and with it the largest n that
  // elr_adam_dedup_noalloc takes, where it has been.
  s.hist = (int32_t*)take(kRadixMaxBins * ntile * 8);
  s.bsum = (int64_t*)(s.hist + kRadixMaxBins * ntile);
  s.bfirst = (int32_t*)(s.bsum + nblk);
  s.dtot = (int32_t*)take(kRadixMaxBins * 8);
  o += al256(ntile * 8);   // unused
  s.d_tot = (int64_t*)take(3 * 8);
  s.uniq = (int64_t*)take(n * 8);
  s.seg_start = (int64_t*)take((n + 1) * 8);
  s.seg_occ0 = (int32_t*)take(n * 4);
  s.chunk_off = (int32_t*)take(n * 4);
  s.chunk_seg = (int32_t*)take(nch * 4);
  s.parts = (float*)take(nch * kGroupsPerChunk * D * 4);
  s.hot_list = (int32_t*)take(hot_max(n) * 4);
  if (out) *out = s;
  return o;
}

// Widest digit of a sort with Key keys.  64-bit keys take 9 bits at most, the widest measured for them.  The scatter's LDS
// with 1,024 threads: 72 KiB at 10 bits of 32-bit keys, 68 at 9 of 64, so two blocks fit a CU (its static_assert).
template <typename Key>
constexpr int max_digit_bits() { return sizeof(Key) == 8 ? 9 : kRadixMaxBits; }

// Passes of a sort of key_bits-bit Key keys (sort_plan); the result sits in buffer (passes - 1) % 2.
template <typename Key>
inline int sort_passes(int key_bits) {
  int passes, rb;
  sort_plan(key_bits, max_digit_bits<Key>(), passes, rb);
  return passes;
}

// The low bits of a key that the radix passes of a key_bits-bit sort compare (at least key_bits).
inline int sort_cover(int key_bits) {
  int passes, rb;
  sort_plan(key_bits, key_bits <= 32 ? max_digit_bits<uint32_t>() : max_digit_bits<uint64_t>(), passes, rb);
  return passes * rb < 64 ? passes * rb : 64;
}

// Smallest b with bound < 2^b (at most 63): keys of b bits hold the ids in [0, bound) and at least one key more.  Only
// a bound that is a power of two takes a bit for it, and only 2^10, 2^20 and 2^30 a pass (100,000 ids of width 32: 83 us
// per update with 2^20 rows, 73 with 1,000,000).
inline int bits_over(int64_t bound) {
  int b = 1;
  while (b < 63 && (int64_t(1) << b) <= bound) ++b;
  return b;
}

// key_of's limit for ids of [0, bound) sorted with key_bits >= bits_over(bound): the highest key that the sort compares
// whole (at least bound).  Ids between bound and it keep their own keys.
inline uint64_t key_lim(int key_bits) {
  const int c = sort_cover(key_bits);
  return c < 64 ? (uint64_t(1) << c) - 1 : uint64_t(1) << 63;
}

// One pass over RB-bit digit p of the keys: histogram, scan (or none: fold), stable scatter from buffer cur (the
// caller's ids on the first pass) to buffer nxt.
template <typename Key, int RB, int NT>
static void radix_pass_nt(const int64_t* ids, int64_t n, uint64_t lim, int p, int cur, int nxt, DedupScratch& S, hipStream_t st) {
  const int64_t ntile = sort_tiles(n);
  const int shift = RB * p, fold = ntile <= kSortFoldTiles;
  const unsigned grid = (unsigned)ntile;
  constexpr int BINS = 1 << RB;
  constexpr unsigned kScanGrid = (unsigned)(BINS / (kHistScanThreads / 64));   // a wave per digit
  Key* kb[2] = {(Key*)S.keys[0], (Key*)S.keys[1]};
  if (p == 0) k_radix_hist<int64_t, Key, RB, NT><<<grid, NT, 0, st>>>(ids, n, lim, shift, S.hist, ntile, fold);
  else k_radix_hist<Key, Key, RB, NT><<<grid, NT, 0, st>>>(kb[cur], n, 0, shift, S.hist, ntile, fold);
  if (!fold) k_radix_hist_scan<<<kScanGrid, kHistScanThreads, 0, st>>>(S.hist, ntile, BINS, S.dtot);
  if (p == 0)
    k_radix_scatter<int64_t, Key, true, RB, NT><<<grid, NT, 0, st>>>(ids, nullptr, n, lim, shift, S.hist, S.dtot,
                                                                      (int)ntile, fold, kb[nxt], S.vals[nxt]);
  else
    k_radix_scatter<Key, Key, false, RB, NT><<<grid, NT, 0, st>>>(kb[cur], S.vals[cur], n, 0, shift, S.hist, S.dtot,
                                                                   (int)ntile, fold, kb[nxt], S.vals[nxt]);
}
template <typename Key, int RB>
static void radix_pass(const int64_t* ids, int64_t n, uint64_t lim, int p, int cur, int nxt, DedupScratch& S, hipStream_t st) {
  if (n >= kSortBig) radix_pass_nt<Key, RB, kSortThreadsBig>(ids, n, lim, p, cur, nxt, S, st);
  else radix_pass_nt<Key, RB, kSortThreadsSmall>(ids, n, lim, p, cur, nxt, S, st);
}

// Sort (ids, positions) by id; returns which buffer holds the result.
template <typename Key>
static int radix_sort(const int64_t* ids, int64_t n, uint64_t lim, int key_bits, DedupScratch& S, hipStream_t st) {
  int passes, rb;
  sort_plan(key_bits, max_digit_bits<Key>(), passes, rb);
  int cur = 0;
  for (int p = 0; p < passes; ++p) {
    const int nxt = p == 0 ? 0 : cur ^ 1;
    if constexpr (max_digit_bits<Key>() >= 10) {
      if (rb == 10) {
        radix_pass<Key, 10>(ids, n, lim, p, cur, nxt, S, st);
        cur = nxt;
        continue;
      }
    }
    if (rb == 9) radix_pass<Key, 9>(ids, n, lim, p, cur, nxt, S, st);
    else radix_pass<Key, 8>(ids, n, lim, p, cur, nxt, S, st);
    cur = nxt;
  }
  return cur;
}

// Segment heads (uniq / seg_start / inverse, U in d_tot[0]) of the sorted keys and, for segment sums (sums), the hot
// segments and the partial-chunk plan (E in d_tot[1]; the windowed path has no partial chunks).
template <typename Key, int ITEMS, class Keys>
static void seg_plan_items(const Keys& keys, const Key* sk, const int32_t* sv, int64_t n, DedupScratch& S, int64_t* uniq, int64_t* inverse,
                     int64_t* n_unique, bool sums, hipStream_t st) {
  const int64_t nblk = cdiv(n, kSegBlock * ITEMS);
  const int scanned = nblk > kFoldMaxBlocks;
  k_seg_count<Key, ITEMS, Keys><<<(unsigned)nblk, kSegBlock, 0, st>>>(keys, sk, n, S.bsum, S.bfirst, S.d_tot + 1, S.d_tot + 2);
  if (scanned) k_scan_blocks<<<1, kScanBlock, 0, st>>>(S.bsum, nblk);
  k_seg_apply<Key, ITEMS, Keys><<<(unsigned)nblk, kSegBlock, 0, st>>>(
      keys, sk, sv, n, S.bsum, scanned, S.bfirst, S.d_tot, n_unique, uniq, S.seg_start, S.seg_occ0, inverse,
      win_shift_for(n) ? nullptr : S.chunk_off, S.chunk_seg, sums ? S.hot_list : nullptr,
      (int)(win_shift_for(n) ? kWinHot : kHotLen), S.d_tot + 2, S.d_tot + 1);
}

template <typename Key, class Keys>
static void seg_plan(const Keys& keys, const Key* sk, const int32_t* sv, int64_t n, DedupScratch& S, int64_t* uniq,
                     int64_t* inverse, int64_t* n_unique, bool sums, hipStream_t st) {
  if (seg_items_for(n) == kSegItemsBig)
    seg_plan_items<Key, kSegItemsBig, Keys>(keys, sk, sv, n, S, uniq, inverse, n_unique, sums, st);
  else
    seg_plan_items<Key, kSegItemsSmall, Keys>(keys, sk, sv, n, S, uniq, inverse, n_unique, sums, st);
}

// Sort, segment heads and partial-chunk plan; returns which buffer holds the sorted positions.  The one-launch plan
// compares at least the bits that the radix passes do, so both paths keep the same ids together.
template <typename Key>
static int dedup_core_t(const int64_t* ids, int64_t n, int key_bits, uint64_t lim, DedupScratch& S, int64_t* uniq,
                        int64_t* inverse, int64_t* n_unique, bool sums, hipStream_t st) {
  const PlainKeys keys{lim};
  if (n <= kSmallPlan) {
    int passes, rb;
    digits_for(sort_cover(key_bits), passes, rb);
    const int cur = (sort_passes<Key>(key_bits) - 1) % 2;   // where the radix passes would leave the positions
    auto go = [&](auto kern) {
      kern<<<1, kFieldThreads, 0, st>>>(ids, (int)n, keys, passes, rb, S.vals[cur], S.d_tot, n_unique, uniq, S.seg_start,
                                        S.seg_occ0, inverse, win_shift_for(n) ? nullptr : S.chunk_off, S.chunk_seg,
                                        sums ? S.hot_list : nullptr, (int)(win_shift_for(n) ? kWinHot : kHotLen));
    };
    if (n <= kFieldThreads) go(k_small_plan<Key, 1>);
    else if (n <= 2 * kFieldThreads) go(k_small_plan<Key, 2>);
    else if (n <= 4 * kFieldThreads) go(k_small_plan<Key, 4>);
    else go(k_small_plan<Key, kSmallItems>);
    return cur;
  }
  const int cur = radix_sort<Key>(ids, n, lim, key_bits, S, st);
  const Key* sk = (const Key*)S.keys[cur];
  seg_plan<Key>(keys, sk, S.vals[cur], n, S, uniq, inverse, n_unique, sums, st);
  return cur;
}

static int dedup_core(const int64_t* ids, int64_t n, int key_bits, uint64_t lim, DedupScratch& S, int64_t* uniq_out,
                      int64_t* inverse, int64_t* n_unique, bool sums, hipStream_t st) {
  int64_t* uniq = uniq_out ? uniq_out : S.uniq;
  return key_bits <= 32 ? dedup_core_t<uint32_t>(ids, n, key_bits, lim, S, uniq, inverse, n_unique, sums, st)
                        : dedup_core_t<uint64_t>(ids, n, key_bits, lim, S, uniq, inverse, n_unique, sums, st);
}

template <int NQ>
inline SegPartials<NQ> seg_partials_of(const float* grad, int64_t D, const int32_t* sv, const DedupScratch& S) {
  return SegPartials<NQ>{grad, D, sv, S.seg_start, S.chunk_off, S.chunk_seg, S.d_tot + 1, S.parts};
}

template <int NQ, int MODE>
static void seg_reduce(const float* grad, int64_t D, const int32_t* sv, DedupScratch& S, const int64_t* uniq,
                       int64_t n, float* out, int64_t nrows, const AdamScalars& s, hipStream_t st, bool partials) {
  const int ws = win_shift_for(n);
  if (!ws && partials) launch1(seg_partials_of<NQ>(grad, D, sv, S), seg_partials_blocks(n), st);
  k_seg_final<NQ, MODE><<<wave_grid(n), 256, 0, st>>>(grad, D, sv, S.seg_start, uniq, S.chunk_off, S.parts, S.d_tot,
                                                       ws, out, nrows, s);
}

// The chunk-layout form: partial chunks (sort path), then the final kernel in launches of at most 2^22 blocks (U <= n;
// blocks past U exit at once), the first with a block per possible hot segment.
template <int MODE>
static void seg_reduce_sub(int lpr, const float* grad, int64_t D, const int32_t* sv, DedupScratch& S,
                           const int64_t* uniq, int64_t n, float* out, int64_t nrows, const AdamScalars& s,
                           hipStream_t st, bool partials) {
  const bool win = win_shift_for(n) != 0;
  if (!win && partials) {
    const SegPartialsLaunch L{seg_partials_of<1>(grad, D, sv, S), seg_partials_blocks(n)};
    seg_partials_visit(L, [&](const auto& f, int64_t nb) { launch1(f, nb, st); });
  }
  chunk_visit(lpr, D, [&](auto L_, auto N_) {
    constexpr int LPR = L_.value, NC = N_.value, SPB = 4 * (64 / LPR);   // segments per block
    const int64_t per = kOneShotBlocks * SPB;
    for (int64_t a = 0; a < n; a += per) {
      const int64_t m = n - a < per ? n - a : per, hb = a == 0 ? hot_max(n) : 0;
      auto go = [&](const auto& f) { launch1(f, hb + cdiv(m, SPB), st); };
      if (win)
        go(SegFinalSub<LPR, NC, MODE, true>{grad, D, sv, S.seg_start, S.seg_occ0, uniq, S.chunk_off, S.parts, S.d_tot, a,
                                            S.hot_list, S.d_tot + 2, hb, out, nrows, s});
      else
        go(SegFinalSub<LPR, NC, MODE, false>{grad, D, sv, S.seg_start, S.seg_occ0, uniq, S.chunk_off, S.parts, S.d_tot,
                                             a, S.hot_list, S.d_tot + 2, hb, out, nrows, s});
    }
  });
}

template <int VPL, int MODE>
static void seg_reduce_wpr(const float* grad, const int32_t* sv, DedupScratch& S, const int64_t* uniq, int64_t n,
                           float* out, int64_t nrows, const AdamScalars& s, hipStream_t st, bool partials) {
  constexpr int64_t D = 64 * VPL;   // sort path only (n > kAtenSmall)
  if (partials) launch1(seg_partials_of<VPL>(grad, D, sv, S), seg_partials_blocks(n), st);
  // one launch per range of at most 2^22 blocks (4 waves of kSegPerWave segments each); U <= n.  The first launch
  // starts with one block per possible hot segment (fewer than n / kHotLen; blocks beyond the count exit at once).
  const int64_t per = kOneShotBlocks * 4 * kSegPerWave;
  for (int64_t a = 0; a < n; a += per) {
    const int64_t m = n - a < per ? n - a : per;
    const int64_t hb = a == 0 ? hot_max(n) : 0;
    const SegFinalWpr<VPL, MODE> f{grad, sv, S.seg_start, S.seg_occ0, uniq, S.chunk_off, S.parts, S.d_tot, a,
                                   S.hot_list, S.d_tot + 2, hb, out, nrows, s};
    k_seg_final_wpr<VPL, MODE><<<(unsigned)(hb + cdiv(m, 4 * kSegPerWave)), 256, 0, st>>>(f);
  }
}

template <int MODE>
static int seg_reduce_d(const float* grad, int64_t D, const int32_t* sv, DedupScratch& S, const int64_t* uniq,
                        int64_t n, float* out, int64_t nrows, const AdamScalars& s, hipStream_t st,
                        bool partials = true) {
  // a wave per row for D = 64, 128, 256 and 512 on the sort path, else rows in chunks of 16 bytes (the windowed order
  // too), else (D % 4 != 0, unaligned arrays) a float per lane
  if (aligned16(grad) && aligned16(out) && !win_shift_for(n)) {
    switch (D) {
      case 64: seg_reduce_wpr<1, MODE>(grad, sv, S, uniq, n, out, nrows, s, st, partials); return ELR_OK;
      case 128: seg_reduce_wpr<2, MODE>(grad, sv, S, uniq, n, out, nrows, s, st, partials); return ELR_OK;
      case 256: seg_reduce_wpr<4, MODE>(grad, sv, S, uniq, n, out, nrows, s, st, partials); return ELR_OK;
      case 512: seg_reduce_wpr<8, MODE>(grad, sv, S, uniq, n, out, nrows, s, st, partials); return ELR_OK;
      default: break;
    }
  }
  if (const int lpr = chunk_lanes(D, grad, out)) {
    seg_reduce_sub<MODE>(lpr, grad, D, sv, S, uniq, n, out, nrows, s, st, partials);
    return ELR_OK;
  }
  const int64_t nq = cdiv(D, 64);
  switch (nq) {
    case 1: seg_reduce<1, MODE>(grad, D, sv, S, uniq, n, out, nrows, s, st, partials); break;
    case 2: seg_reduce<2, MODE>(grad, D, sv, S, uniq, n, out, nrows, s, st, partials); break;
    case 3:
    case 4: seg_reduce<4, MODE>(grad, D, sv, S, uniq, n, out, nrows, s, st, partials); break;
    case 5: case 6: case 7:
    case 8: seg_reduce<8, MODE>(grad, D, sv, S, uniq, n, out, nrows, s, st, partials); break;
    default: return ELR_EUNSUPPORTED;
  }
  return ELR_OK;
}

inline bool dedup_sizes_ok(int64_t n) { return n >= 0 && n < (int64_t(1) << 31); }

}  // namespace elr

extern "C" int64_t elr_dedup_scratch_bytes(int64_t n, int64_t D) {
  if (!elr::dedup_sizes_ok(n) || D < 0) return ELR_EINVAL;
  return elr::dedup_scratch_bytes(n, D < 1 ? 1 : D, nullptr, nullptr);
}

extern "C" int elr_unique(const int64_t* ids, int64_t n, int key_bits, int64_t* uniq, int64_t* inverse,
                          int64_t* n_unique, void* scratch, int64_t scratch_bytes, void* stream) {
  using namespace elr;
  if (!dedup_sizes_ok(n) || key_bits < 1 || key_bits > 64) return ELR_EINVAL;
  if (n == 0) return ELR_OK;
  if (!ids || !uniq || !n_unique || !scratch) return ELR_EINVAL;
  DedupScratch S;
  if (scratch_bytes < dedup_scratch_bytes(n, 1, &S, scratch)) return ELR_ECAPACITY;
  hipStream_t st = (hipStream_t)stream;
  dedup_core(ids, n, key_bits, 0, S, uniq, inverse, n_unique, false, st);
  return launch_status();
}

extern "C" int elr_segment_sum(const float* grad, const int64_t* idx, int64_t n, int64_t D, int64_t num_rows,
                               float* out, void* scratch, int64_t scratch_bytes, void* stream) {
  using namespace elr;
  if (!dedup_sizes_ok(n) || D < 1 || num_rows < 0) return ELR_EINVAL;
  if (n == 0) return ELR_OK;
  if (!grad || !idx || !out || !scratch) return ELR_EINVAL;
  if (D > 512) return ELR_EUNSUPPORTED;
  DedupScratch S;
  if (scratch_bytes < dedup_scratch_bytes(n, D, &S, scratch)) return ELR_ECAPACITY;
  hipStream_t st = (hipStream_t)stream;
  const int kb = bits_over(num_rows);
  const int cur = dedup_core(idx, n, kb, key_lim(kb), S, nullptr, nullptr, nullptr, true, st);
  const AdamScalars none{};
  const int rc = seg_reduce_d<0>(grad, D, S.vals[cur], S, S.uniq, n, out, num_rows, none, st);
  return rc != ELR_OK ? rc : launch_status();
}

extern "C" int elr_adam_dedup(float* state, int64_t C, const int64_t* ids, const float* grad, int64_t n, int64_t D,
                              const float sc[8], void* scratch, int64_t scratch_bytes, void* stream) {
  using namespace elr;
  if (!dedup_sizes_ok(n) || D < 1 || C < 0 || !sc) return ELR_EINVAL;
  if (n == 0) return ELR_OK;
  if (!state || !ids || !grad || !scratch) return ELR_EINVAL;
  if (D > 512) return ELR_EUNSUPPORTED;
  DedupScratch S;
  if (scratch_bytes < dedup_scratch_bytes(n, D, &S, scratch)) return ELR_ECAPACITY;
  hipStream_t st = (hipStream_t)stream;
  const AdamScalars s = make_scalars(sc);
  const int kb = bits_over(C);
  const int cur = dedup_core(ids, n, kb, key_lim(kb), S, nullptr, nullptr, nullptr, true, st);
  const int rc = seg_reduce_d<1>(grad, D, S.vals[cur], S, S.uniq, n, state, C, s, st);
  return rc != ELR_OK ? rc : launch_status();
}

// ---- dedup plan: one sort per batch, reused by the segment sum -------------------------------------------------
// elr_dedup_plan sorts the batch and finds its segments exactly as elr_unique does, and also lays out the extra
// chunks; the scratch then holds the plan (sorted positions, segment starts, first occurrences, chunk plan, U).
// elr_segment_sum_plan sums a gradient batch over that plan without sorting again.  The sorted result lives in the
// scratch buffer that the last radix pass wrote: with p passes, buffer (p - 1) % 2.
static int plan_result_buffer(int key_bits) {
  return ((key_bits <= 32 ? elr::sort_passes<uint32_t>(key_bits) : elr::sort_passes<uint64_t>(key_bits)) - 1) % 2;
}

extern "C" int64_t elr_dedup_plan_bytes(int64_t n, int64_t D) {
  using namespace elr;
  if (!dedup_sizes_ok(n) || D < 1) return ELR_EINVAL;
  return dedup_scratch_bytes(n, D, nullptr, nullptr);
}

static int dedup_plan(const int64_t* ids, int64_t n, int key_bits, uint64_t lim, int64_t* uniq, int64_t* inverse,
                      int64_t* n_unique, void* plan, int64_t plan_bytes, int64_t D, void* stream) {
  using namespace elr;
  if (!dedup_sizes_ok(n) || key_bits < 1 || key_bits > 64 || D < 1) return ELR_EINVAL;
  if (n == 0) return ELR_OK;
  if (!ids || !uniq || !n_unique || !plan) return ELR_EINVAL;
  DedupScratch S;
  if (plan_bytes < dedup_scratch_bytes(n, D, &S, plan)) return ELR_ECAPACITY;
  hipStream_t st = (hipStream_t)stream;
  const int cur = dedup_core(ids, n, key_bits, lim, S, uniq, inverse, n_unique, true, st);
  if (cur != plan_result_buffer(key_bits)) return ELR_EINVAL;
  return launch_status();
}

extern "C" int elr_dedup_plan(const int64_t* ids, int64_t n, int key_bits, int64_t* uniq, int64_t* inverse,
                              int64_t* n_unique, void* plan, int64_t plan_bytes, int64_t D, void* stream) {
  return dedup_plan(ids, n, key_bits, 0, uniq, inverse, n_unique, plan, plan_bytes, D, stream);
}

extern "C" int elr_dedup_plan_bounded(const int64_t* ids, int64_t n, int64_t bound, int64_t* uniq, int64_t* inverse,
                                      int64_t* n_unique, void* plan, int64_t plan_bytes, int64_t D, void* stream) {
  if (bound < 0) return ELR_EINVAL;
  const int kb = elr::bits_over(bound);
  return dedup_plan(ids, n, kb, elr::key_lim(kb), uniq, inverse, n_unique, plan, plan_bytes, D, stream);
}

extern "C" int elr_dedup_plan_fields(const int64_t* ids, int64_t nrows, int64_t nfields, const int64_t* field_lo,
                                     int key_bits, int64_t* uniq, int64_t* inverse, int64_t* n_unique, void* plan,
                                     int64_t plan_bytes, int64_t D, void* stream) {
  using namespace elr;
  if (nrows < 0 || nfields < 1 || !field_lo || key_bits < 1 || key_bits > 64 || D < 1) return ELR_EINVAL;
  if (nrows > 0 && nfields > ((int64_t(1) << 31) - 1) / nrows) return ELR_EINVAL;
  const int64_t n = nrows * nfields;
  if (n == 0) return ELR_OK;
  if (field_lo[0] < 0) return ELR_EINVAL;
  for (int64_t c = 0; c < nfields; ++c)
    if (field_lo[c + 1] < field_lo[c]) return ELR_EINVAL;
  bool general = nrows > kFieldRows || nfields > kFieldMax || n <= kAtenSmall;
  for (int64_t c = 0; c < nfields; ++c) general = general || field_lo[c + 1] - field_lo[c] > kFieldSpanMax;
  if (general)   // (key_bits that leave no key for an id past the last field: the ids as they are)
    return dedup_plan(ids, n, key_bits, key_bits >= bits_over(field_lo[nfields]) ? key_lim(key_bits) : 0, uniq, inverse,
                      n_unique, plan, plan_bytes, D, stream);
  if (!ids || !uniq || !n_unique || !plan) return ELR_EINVAL;
  DedupScratch S;
  if (plan_bytes < dedup_scratch_bytes(n, D, &S, plan)) return ELR_ECAPACITY;
  FieldBounds fb;
  for (int64_t c = 0; c <= nfields; ++c) fb.lo[c] = field_lo[c];
  hipStream_t st = (hipStream_t)stream;
  int32_t* sv = S.vals[plan_result_buffer(key_bits)];
  k_field_keys<<<dim3((unsigned)cdiv(nrows, kFieldKeyRows), (unsigned)nfields), 256, 0, st>>>(
      ids, nrows, (int)nfields, fb, (uint32_t*)S.keys[1]);
  auto sort = [&](auto kern) {
    kern<<<(unsigned)nfields, kFieldThreads, 0, st>>>((const uint32_t*)S.keys[1], nrows, (int)nfields, fb,
                                                      (uint32_t*)S.keys[0], sv);
  };
  const int64_t per = cdiv(nrows, kFieldThreads);
  if (per <= 1) sort(k_field_sort<1>);
  else if (per <= 2) sort(k_field_sort<2>);
  else if (per <= 4) sort(k_field_sort<4>);
  else if (per <= 8) sort(k_field_sort<8>);
  else sort(k_field_sort<kFieldItems>);
  seg_plan<uint32_t>(FieldKeys{fb, (uint32_t)nrows}, (const uint32_t*)S.keys[0], sv, n, S, uniq, inverse, n_unique, true,
                     st);
  return launch_status();
}

namespace elr {

int seg_partials_prep(const float* grad, int64_t n, int64_t D, int key_bits, const void* plan, int64_t plan_bytes,
                      SegPartialsLaunch& out) {
  out.blocks = 0;
  if (!dedup_sizes_ok(n) || D < 1 || key_bits < 1 || key_bits > 64) return ELR_EINVAL;
  if (n == 0) return ELR_OK;
  if (!grad || !plan) return ELR_EINVAL;
  if (D > 512) return ELR_EUNSUPPORTED;
  DedupScratch S;
  if (plan_bytes < dedup_scratch_bytes(n, D, &S, const_cast<void*>(plan))) return ELR_ECAPACITY;
  if (win_shift_for(n)) return ELR_OK;
  out.a = seg_partials_of<1>(grad, D, S.vals[plan_result_buffer(key_bits)], S);
  out.blocks = seg_partials_blocks(n);
  return ELR_OK;
}

// elr_segment_sum_plan, with or without the partial chunks (computed earlier by elr_plan_classify_seg).
static int segment_sum_plan(const float* grad, int64_t n, int64_t D, int key_bits, const void* plan,
                            int64_t plan_bytes, const int64_t* perm, float* out, int64_t out_rows, void* stream,
                            bool partials) {
  if (!dedup_sizes_ok(n) || D < 1 || key_bits < 1 || key_bits > 64 || out_rows < 0) return ELR_EINVAL;
  if (n == 0) return ELR_OK;
  if (!grad || !plan || !out) return ELR_EINVAL;
  if (D > 512) return ELR_EUNSUPPORTED;
  DedupScratch S;
  if (plan_bytes < dedup_scratch_bytes(n, D, &S, const_cast<void*>(plan))) return ELR_ECAPACITY;
  hipStream_t st = (hipStream_t)stream;
  const AdamScalars none{};
  const int rc = seg_reduce_d<0>(grad, D, S.vals[plan_result_buffer(key_bits)], S, perm, n, out, out_rows, none, st,
                                 partials);
  return rc != ELR_OK ? rc : launch_status();
}

template <int VPL>
static void seg_final_with(const float* grad, const int32_t* sv, DedupScratch& S, const int64_t* perm, int64_t n,
                           float* out, int64_t nrows, const DirLstepsHits& first, int64_t nb1, hipStream_t st) {
  const int64_t hb = hot_max(n);
  const SegFinalWpr<VPL, 0> f{grad, sv, S.seg_start, S.seg_occ0, perm, S.chunk_off, S.parts, S.d_tot, 0,
                              S.hot_list, S.d_tot + 2, hb, out, nrows, AdamScalars{}};
  launch2(first, nb1, f, hb + cdiv(n, 4 * kSegPerWave), st);
}

int segment_sum_plan_final_with(const float* grad, int64_t n, int64_t D, int key_bits, const void* plan,
                                int64_t plan_bytes, const int64_t* perm, float* out, int64_t out_rows,
                                const DirLstepsHits& first, int64_t nb1, void* stream) {
  if (!dedup_sizes_ok(n) || D < 1 || key_bits < 1 || key_bits > 64 || out_rows < 0 || nb1 < 0) return ELR_EINVAL;
  if (n == 0 || !grad || !plan || !out) return ELR_EUNSUPPORTED;
  // the wave-per-row final kernel in one launch: aligned rows of 64, 128, 256 or 512, the sort path, at most one
  // launch's worth of segments (seg_reduce_wpr)
  if (!aligned16(grad) || !aligned16(out) || win_shift_for(n) || n > kOneShotBlocks * 4 * kSegPerWave)
    return ELR_EUNSUPPORTED;
  DedupScratch S;
  if (plan_bytes < dedup_scratch_bytes(n, D, &S, const_cast<void*>(plan))) return ELR_ECAPACITY;
  const int32_t* sv = S.vals[plan_result_buffer(key_bits)];
  hipStream_t st = (hipStream_t)stream;
  switch (D) {
    case 64: seg_final_with<1>(grad, sv, S, perm, n, out, out_rows, first, nb1, st); break;
    case 128: seg_final_with<2>(grad, sv, S, perm, n, out, out_rows, first, nb1, st); break;
    case 256: seg_final_with<4>(grad, sv, S, perm, n, out, out_rows, first, nb1, st); break;
    case 512: seg_final_with<8>(grad, sv, S, perm, n, out, out_rows, first, nb1, st); break;
    default: return ELR_EUNSUPPORTED;
  }
  return launch_status();
}

}  // namespace elr

extern "C" int elr_segment_sum_plan(const float* grad, int64_t n, int64_t D, int key_bits, const void* plan,
                                    int64_t plan_bytes, const int64_t* perm, float* out, int64_t out_rows,
                                    void* stream) {
  return elr::segment_sum_plan(grad, n, D, key_bits, plan, plan_bytes, perm, out, out_rows, stream, true);
}

extern "C" int elr_segment_sum_plan_final(const float* grad, int64_t n, int64_t D, int key_bits, const void* plan,
                                          int64_t plan_bytes, const int64_t* perm, float* out, int64_t out_rows,
                                          void* stream) {
  return elr::segment_sum_plan(grad, n, D, key_bits, plan, plan_bytes, perm, out, out_rows, stream, false);
}

extern "C" int elr_adam_dedup_plan(float* state, int64_t C, const int64_t* uniq, const float* grad, int64_t n,
                                   int64_t D, int key_bits, const void* plan, int64_t plan_bytes, const float sc[8],
                                   void* stream) {
  using namespace elr;
  if (!dedup_sizes_ok(n) || D < 1 || C < 0 || key_bits < 1 || key_bits > 64 || !sc) return ELR_EINVAL;
  if (n == 0) return ELR_OK;
  if (!state || !uniq || !grad || !plan) return ELR_EINVAL;
  if (D > 512) return ELR_EUNSUPPORTED;
  DedupScratch S;
  if (plan_bytes < dedup_scratch_bytes(n, D, &S, const_cast<void*>(plan))) return ELR_ECAPACITY;
  hipStream_t st = (hipStream_t)stream;
  const int rc = seg_reduce_d<1>(grad, D, S.vals[plan_result_buffer(key_bits)], S, uniq, n, state, C,
                                 make_scalars(sc), st);
  return rc != ELR_OK ? rc : launch_status();
}

// ---- duplicate-id Adam that allocates nothing ------------------------------------------------------------------
// elr_adam_dedup with its scratch in a file-scope device array instead of a caller buffer, for callers that cannot
// allocate device memory (code under graph capture, tight serving loops).  The array (ELR_NOALLOC_SCRATCH_BYTES)
// exists once per GPU the library runs on, for the life of the process.  In host code `scratch` names only a
// host-side stand-in; the device address is obtained once per device with hipGetSymbolAddress, with that device
// current, and only that address is handed to kernels.  Every kernel writes the parts of the scratch it later
// reads (the hot-segment counter is zeroed by the segment kernel itself), so nothing needs clearing between calls.
// All calls on one GPU share its array: calls that overlap in time on one GPU (two streams, two host threads) race.
#include <atomic>
#include <mutex>

namespace elr {
constexpr int kNoAllocMaxDevices = 64;
std::atomic<void*> g_noalloc_ptr[kNoAllocMaxDevices];
std::mutex g_noalloc_mu;
}  // namespace elr

static __device__ __align__(256) unsigned char scratch[ELR_NOALLOC_SCRATCH_BYTES];

// Device address of `scratch` on the current device (resolved on the first call per device).  A stream of another
// device is refused (ELR_EINVAL): its kernels would be handed this device's address.
static int noalloc_scratch(void** out, hipStream_t stream) {
  using namespace elr;
  int dev = -1;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess) return (int)e;
  if (dev < 0 || dev >= kNoAllocMaxDevices) return ELR_EUNSUPPORTED;
  if (stream) {
    hipDevice_t sdev = -1;
    e = hipStreamGetDevice(stream, &sdev);
    if (e != hipSuccess) return (int)e;
    if ((int)sdev != dev) return ELR_EINVAL;
  }
  void* p = g_noalloc_ptr[dev].load(std::memory_order_acquire);
  if (!p) {
    std::lock_guard<std::mutex> g(g_noalloc_mu);
    p = g_noalloc_ptr[dev].load(std::memory_order_relaxed);
    if (!p) {
      e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
      if (e != hipSuccess) return (int)e;
      if (!p) return ELR_EINVAL;
      g_noalloc_ptr[dev].store(p, std::memory_order_release);
    }
  }
  *out = p;
  return ELR_OK;
}

extern "C" int elr_adam_dedup_noalloc(float* state, int64_t C, const int64_t* ids, const float* grad, int64_t n,
                                      int64_t D, const float sc[8], void* stream) {
  using namespace elr;
  if (!dedup_sizes_ok(n) || D < 1 || C < 0 || !sc) return ELR_EINVAL;
  if (n == 0) return ELR_OK;
  if (!state || !ids || !grad) return ELR_EINVAL;
  if (D > 512) return ELR_EUNSUPPORTED;
  if (dedup_scratch_bytes(n, D, nullptr, nullptr) > (int64_t)ELR_NOALLOC_SCRATCH_BYTES) return ELR_ECAPACITY;
  void* base = nullptr;
  const int rc = noalloc_scratch(&base, static_cast<hipStream_t>(stream));
  if (rc != ELR_OK) return rc;
  return elr_adam_dedup(state, C, ids, grad, n, D, sc, base, (int64_t)ELR_NOALLOC_SCRATCH_BYTES, stream);
}
