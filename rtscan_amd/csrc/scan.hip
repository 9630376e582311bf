// scan.hip -- kernel (a) direct streaming range scan, kernel (c) fused conjunction /
// AND+popcount, and the bitmap operations of the cuda_and.cu surface.
//
// Layout: a wave64 reads 256 consecutive rows per load instruction as one uint4 (4 rows)
// per lane, so lane l holds rows 4l..4l+3 of the 256.  Output word g (rows 32g..32g+31)
// is spread over the 8 lanes 8g..8g+7, 4 rows each: each lane places its 4 match bits at
// bit 31-4*(l%8)-j, an OR over the 8 lanes (DPP, no LDS) assembles the MSB-first word,
// and one lane per group stores it.
#include <string.h>

#include <algorithm>
#include <type_traits>

#include "common.h"
#include "transpose.h"

namespace rts {

template <int C>
struct ColPreds {
  const uint32_t *col[C];
  uint32_t lo[C];
  uint32_t span[C];  // hi - lo
};

// One row per lane for rows [r0, r0 + 64): 2 MSB-first words (ballot + bit reverse),
// stored by lanes 0 and 1; rows >= n contribute 0 bits.  Returns the popcount the lane
// stored (0 on other lanes).
template <int C, int MODE>
__device__ __forceinline__ uint32_t scan_chunk64(const ColPreds<C> &p, uint64_t r0, uint64_t n,
                                                 BITS *out, int lane) {
  const uint64_t r = r0 + lane;
  bool m = r < n;
  if (m) {
#pragma unroll
    for (int c = 0; c < C; c++) m = m && (p.col[c][r] - p.lo[c]) <= p.span[c];
  }
  const uint64_t b = __ballot(m);
  uint32_t pc = 0;
  if (lane < 2) {
    const uint64_t w = r0 / 32 + lane;
    if (w * 32 < n) {
      const uint32_t v = __brev(lane == 0 ? (uint32_t)b : (uint32_t)(b >> 32));
      pc = __popc(store_word<MODE>(out, w, v));
    }
  }
  return pc;
}

// Whole tiles of 256*U rows with 128-bit loads (all columns 16-byte aligned); the rows
// past the last whole tile (fewer than 256*U) are done by the grid's last block one row
// per lane.  One launch per scan, count included.
template <int C, int U, int MODE, bool COUNT>
__global__ __launch_bounds__(kBlock) void k_scan_tiles(ColPreds<C> p, uint64_t n, BITS *out,
                                                       CountSink sink) {
  const int lane = threadIdx.x & (kWave - 1);
  const uint64_t wave = (uint64_t)blockIdx.x * (kBlock / kWave) + threadIdx.x / kWave;
  const uint64_t nwaves = (uint64_t)gridDim.x * (kBlock / kWave);
  const uint64_t ntiles = n / (uint64_t)(256 * U);
  const uint32_t shift = 28 - 4 * (lane & 7);
  const bool writer = (lane & 7) == 0;
  uint32_t pc = 0;
  for (uint64_t t = wave; t < ntiles; t += nwaves) {
    const uint64_t row0 = t * (uint64_t)(256 * U);
    uint32_t nib[U];
#pragma unroll
    for (int u = 0; u < U; u++) nib[u] = 0xF;
#pragma unroll
    for (int c = 0; c < C; c++) {
      const uint4 *src = reinterpret_cast<const uint4 *>(p.col[c] + row0) + lane;
      uint4 v[U];
#pragma unroll
      for (int u = 0; u < U; u++) v[u] = load_stream(src + 64 * u);
#pragma unroll
      for (int u = 0; u < U; u++) nib[u] &= nibble4(v[u], p.lo[c], p.span[c]);
    }
#pragma unroll
    for (int u = 0; u < U; u++) {
      const uint32_t w = or_lanes8(nib[u] << shift);
      if (writer) {
        const uint32_t stored = store_word<MODE>(out, row0 / 32 + 8 * u + lane / 8, w);
        if (COUNT) pc += __popc(stored);
      }
    }
  }
  if (blockIdx.x == gridDim.x - 1) {
    const uint64_t begin = ntiles * (uint64_t)(256 * U);
    for (uint64_t r0 = begin + 64 * (threadIdx.x / kWave); r0 < n; r0 += kBlock)
      pc += scan_chunk64<C, MODE>(p, r0, n, out, lane);
  }
  if (COUNT) count_block_partial(pc, sink);
}

// Any alignment: one row per lane over all n rows.
template <int C, int MODE, bool COUNT>
__global__ __launch_bounds__(kBlock) void k_scan_rows(ColPreds<C> p, uint64_t n, BITS *out,
                                                      CountSink sink) {
  const int lane = threadIdx.x & (kWave - 1);
  const uint64_t wave = (uint64_t)blockIdx.x * (kBlock / kWave) + threadIdx.x / kWave;
  const uint64_t nwaves = (uint64_t)gridDim.x * (kBlock / kWave);
  const uint64_t nchunks = (n + 63) / 64;
  uint32_t pc = 0;
  for (uint64_t ch = wave; ch < nchunks; ch += nwaves)
    pc += scan_chunk64<C, MODE>(p, ch * 64, n, out, lane);
  if (COUNT) count_block_partial(pc, sink);
}

__global__ void k_zero_u64(unsigned long long *p) { *p = 0ull; }

// ------------------------------------------------------------------ bitmap operations

enum BitOp : int { kCopy = 0, kNot = 1, kAndNot = 2, kAnd = 3, kOr = 4, kFill = 5, kXorWith = 6 };

template <int OP>
__device__ __forceinline__ uint32_t bitop(uint32_t d, uint32_t a, uint32_t b, uint32_t v) {
  if (OP == kCopy) return a;
  if (OP == kNot) return ~a;
  if (OP == kAndNot) return b & ~a;
  if (OP == kAnd) return d & a;
  if (OP == kOr) return d | a;
  if (OP == kFill) return v;
  return d ^ a;
}

template <int OP>
__device__ __forceinline__ uint4 bitop4(uint4 d, uint4 a, uint4 b, uint32_t v) {
  return make_uint4(bitop<OP>(d.x, a.x, b.x, v), bitop<OP>(d.y, a.y, b.y, v),
                    bitop<OP>(d.z, a.z, b.z, v), bitop<OP>(d.w, a.w, b.w, v));
}

constexpr bool reads_dst(int op) { return op == kAnd || op == kOr || op == kXorWith; }
constexpr bool reads_a(int op) { return op != kFill; }
constexpr bool reads_b(int op) { return op == kAndNot; }

// dst[i] = OP(dst[i], a[i], b[i]) over `words` words; VEC: all pointers 16-byte aligned.
template <int OP, bool VEC>
__global__ __launch_bounds__(kBlock) void k_bitop(BITS *dst, const BITS *a, const BITS *b,
                                                  uint64_t words, uint32_t value) {
  const uint64_t tid = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  const uint64_t nth = (uint64_t)gridDim.x * blockDim.x;
  uint64_t done = 0;
  if (VEC) {
    const uint64_t n4 = words / 4;
    uint4 *d4 = reinterpret_cast<uint4 *>(dst);
    const uint4 *a4 = reinterpret_cast<const uint4 *>(a);
    const uint4 *b4 = reinterpret_cast<const uint4 *>(b);
    for (uint64_t i = tid; i < n4; i += nth) {
      uint4 dv = reads_dst(OP) ? d4[i] : make_uint4(0, 0, 0, 0);
      uint4 av = reads_a(OP) ? a4[i] : make_uint4(0, 0, 0, 0);
      uint4 bv = reads_b(OP) ? b4[i] : make_uint4(0, 0, 0, 0);
      d4[i] = bitop4<OP>(dv, av, bv, value);
    }
    done = n4 * 4;
  }
  for (uint64_t i = done + tid; i < words; i += nth) {
    uint32_t dv = reads_dst(OP) ? dst[i] : 0u;
    uint32_t av = reads_a(OP) ? a[i] : 0u;
    uint32_t bv = reads_b(OP) ? b[i] : 0u;
    dst[i] = bitop<OP>(dv, av, bv, value);
  }
}

// Toggle rows [0, rows) of a bitmap (refineWithCuda's intent, cuda_and.cu:3-10): whole
// words are negated, the partial last word only in its first rows % 32 bits.
__global__ __launch_bounds__(kBlock) void k_flip_rows(BITS *bm, uint64_t rows) {
  const uint64_t tid = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  const uint64_t nth = (uint64_t)gridDim.x * blockDim.x;
  const uint64_t full = rows / 32;
  for (uint64_t i = tid; i < full; i += nth) bm[i] = ~bm[i];
  if (tid == 0 && (rows & 31)) bm[full] ^= ~(0xFFFFFFFFu >> (rows & 31));
}

// ---------------------------------------------------------------- AND + popcount

constexpr int kMaxAnd = 8;
struct BitmapSet {
  const BITS *bm[kMaxAnd];
};

// out = AND of nb bitmaps over `words` words; the last word is masked by `last_mask`.
// out == nullptr: count only.
template <bool VEC, bool COUNT>
__global__ __launch_bounds__(kBlock) void k_and_popcount(BitmapSet s, int nb, uint64_t words,
                                                         uint32_t last_mask, BITS *out,
                                                         CountSink sink) {
  const uint64_t tid = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  const uint64_t nth = (uint64_t)gridDim.x * blockDim.x;
  uint32_t pc = 0;
  uint64_t done = 0;
  if (VEC) {
    const uint64_t n4 = words / 4;
    for (uint64_t i = tid; i < n4; i += nth) {
      uint4 acc = reinterpret_cast<const uint4 *>(s.bm[0])[i];
      for (int k = 1; k < nb; k++) {
        uint4 v = reinterpret_cast<const uint4 *>(s.bm[k])[i];
        acc.x &= v.x;
        acc.y &= v.y;
        acc.z &= v.z;
        acc.w &= v.w;
      }
      if (4 * i + 3 == words - 1) acc.w &= last_mask;
      if (out) reinterpret_cast<uint4 *>(out)[i] = acc;
      if (COUNT) pc += __popc(acc.x) + __popc(acc.y) + __popc(acc.z) + __popc(acc.w);
    }
    done = n4 * 4;
  }
  for (uint64_t i = done + tid; i < words; i += nth) {
    uint32_t acc = s.bm[0][i];
    for (int k = 1; k < nb; k++) acc &= s.bm[k][i];
    if (i == words - 1) acc &= last_mask;
    if (out) out[i] = acc;
    if (COUNT) pc += __popc(acc);
  }
  if (COUNT) count_block_partial(pc, sink);
}

// ------------------------------------------------- many predicates over one column

constexpr int kMultiPreds = 64;  // predicates per pass
constexpr int kMultiLaneRows = 32;                      // rows per lane: one bitmap word
constexpr int kMultiTileRows = kWave * kMultiLaneRows;  // 2048 rows per wave tile
constexpr unsigned kMultiMaxGrid = 4096;

constexpr int kStagedBlock = 512;         // threads of a workgroup whose words pass through LDS
constexpr int kStaged = 8;                // predicates whose words do so at once
// Bitmaps that do not start on cache lines: bytes of them from which on that pays.  In less
// the parts of a line meet in the caches before they are written, and the barriers show (33
// bitmaps of 5e7 rows, 206 MB, counted: 93 us without, 98 with); more is bound by the rate at
// which partial lines are written: 64 bitmaps of 1e8 rows, 800 MB, 322 -> 268 us (250 when
// they start on lines), 32, 400 MB, 197 -> 166; 64 of 2e8 rows 607 -> 500.
constexpr uint64_t kStagedBytes = 320u << 20;
constexpr uint32_t kHistEntries = 1024;  // row counts of a workgroup: all copies
constexpr unsigned kScanXcds = 8;
constexpr int kRankEntries = 2 * kMultiPreds + 2;       // ranges between the bounds, and one for no row

struct MultiPreds {
  uint32_t lo[kMultiPreds];
  uint32_t span[kMultiPreds];  // hi - lo
  uint64_t empty;              // bit p: predicate p matches no row
};

// Rows of the predicates of a launch.  A workgroup adds (1 << 44) | its rows to the predicate's
// accumulator of its group (blockIdx.x % kMultiGroups); the one whose ticket completes the
// group adds the group's rows to the predicate's last accumulator in the same way, and the
// one that completes that writes the count; all accumulators are left at zero.  A second
// kernel that summed the workgroups' rows took longer for every size: 64 predicates over 1e5
// rows 10.6 -> 9.2 us, 2^20 11.1 -> 9.6, 8e6 25.7 -> 23.2, 1e8 292 -> 287.  One accumulator a
// predicate (one group) is slower from 2^20 rows on (11.4, 8e6: 34.8), 4 to 32 groups are alike.
constexpr int kMultiGroups = 16;
constexpr size_t kMultiAccBytes = (size_t)(kMultiGroups + 1) * kMultiPreds * sizeof(unsigned long long);
struct MultiSink {
  unsigned long long *acc;  // per group, and once more, of each predicate
  unsigned long long *counts;
};
__device__ __forceinline__ void multi_count(const MultiSink &sink, int p, uint32_t rows) {
  constexpr unsigned long long kOne = 1ull << kCountTicketShift;
  const unsigned g = blockIdx.x % kMultiGroups;
  unsigned long long *acc = sink.acc + g * kMultiPreds + p;
  unsigned long long old = atomicAdd(acc, kOne | rows);
  if ((old >> kCountTicketShift) != (gridDim.x - g - 1) / kMultiGroups) return;
  atomicExch(acc, 0ull);
  const unsigned long long sum = (old & (kOne - 1)) + rows;
  acc = sink.acc + kMultiGroups * kMultiPreds + p;
  old = atomicAdd(acc, kOne | sum);
  if ((old >> kCountTicketShift) + 1 != min(gridDim.x, (unsigned)kMultiGroups)) return;
  sink.counts[p] = (old & (kOne - 1)) + sum;
  atomicExch(acc, 0ull);
}

__global__ __launch_bounds__(kBlock) void k_zero_multi(unsigned long long *acc) {
  for (size_t i = threadIdx.x; i < kMultiAccBytes / sizeof(*acc); i += kBlock) acc[i] = 0;
}

// Up to kMultiPreds closed ranges over one column in one pass.  A wave takes a tile of
// 2048 rows, lane l the 32 rows of bitmap word l (eight 16-byte loads of its own 128 bytes;
// the wave's loads cover the tile's 8 KB once), kept in registers; for every predicate p
// the lane shifts its rows' match bits into one MSB-first word (subtract, compare, add
// with carry per row: no cross-lane assembly) and the wave stores its 64 consecutive
// words of bitmap p (out + p * stride) with one instruction.  Rows past the whole tiles
// (or every row, for a column that is not 16-byte aligned) go one row per lane, 64 rows per
// wave step.  The predicates are split over gridDim.y groups of `pper` (workgroup y takes
// [y * pper, y * pper + pper)), so that a short column still fills the device; the groups
// read the same tiles, the later ones from L2.  COUNT: per-workgroup totals per predicate
// (DPP wave totals added in LDS) into the sink.
template <bool COUNT>
__global__ __launch_bounds__(kBlock) void k_scan_multi(const uint32_t *col, uint64_t n, uint64_t ntiles,
                                                       MultiPreds mp, int np, int pper, BITS *out,
                                                       uint64_t stride, MultiSink sink) {
  __shared__ uint32_t cnt[kMultiPreds];
  const int lane = threadIdx.x & (kWave - 1);
  const int pbeg = blockIdx.y * pper, pend = min(np, pbeg + pper);
  if (COUNT) {
    if (threadIdx.x < kMultiPreds) cnt[threadIdx.x] = 0;
    __syncthreads();
  }
  const uint64_t wave = (uint64_t)blockIdx.x * (kBlock / kWave) + threadIdx.x / kWave;
  const uint64_t nwaves = (uint64_t)gridDim.x * (kBlock / kWave);
  for (uint64_t t = wave; t < ntiles; t += nwaves) {
    const uint64_t row0 = t * (uint64_t)kMultiTileRows;
    const uint4 *src = reinterpret_cast<const uint4 *>(col + row0 + (uint64_t)kMultiLaneRows * lane);
    uint32_t x[kMultiLaneRows];
#pragma unroll
    for (int k = 0; k < kMultiLaneRows / 4; k++) {
      const uint4 v = src[k];
      x[4 * k] = v.x;
      x[4 * k + 1] = v.y;
      x[4 * k + 2] = v.z;
      x[4 * k + 3] = v.w;
    }
    BITS *o = out + row0 / 32 + lane;
    for (int p = pbeg; p < pend; p++) {
      uint32_t w = 0;
      if (!((mp.empty >> p) & 1)) {
        const uint32_t lo = mp.lo[p], span = mp.span[p];
#pragma unroll
        for (int r = 0; r < kMultiLaneRows; r++) w = w + w + (uint32_t)(x[r] - lo <= span);
      }
      o[p * stride] = w;
      if (COUNT) {
        const uint32_t c = wave_total(__popc(w));
        if (lane == 0 && c) atomicAdd(&cnt[p], c);
      }
    }
  }
  // rows past the whole tiles: one row per lane, 64 rows per wave step
  const uint64_t begin = ntiles * (uint64_t)kMultiTileRows;
  const uint64_t nchunks = (n - begin + 63) / 64;
  for (uint64_t c = wave; c < nchunks; c += nwaves) {
    const uint64_t r0 = begin + c * 64, r = r0 + lane;
    const uint32_t x = r < n ? col[r] : 0u;
    const uint64_t wd = r0 / 32 + (lane & 1);
    for (int p = pbeg; p < pend; p++) {
      const bool m = r < n && !((mp.empty >> p) & 1) && (x - mp.lo[p]) <= mp.span[p];
      const uint64_t b = __ballot(m);
      const uint32_t word = __brev((lane & 1) ? (uint32_t)(b >> 32) : (uint32_t)b);
      if (lane < 2 && wd * 32 < n) {
        out[p * stride + wd] = word;
        if (COUNT && word) atomicAdd(&cnt[p], (uint32_t)__popc(word));
      }
    }
  }
  if (COUNT) {
    __syncthreads();
    if ((int)threadIdx.x >= pbeg && (int)threadIdx.x < pend)
      multi_count(sink, threadIdx.x, cnt[threadIdx.x]);
  }
}

// The same pass for many predicates (direct_preds).  The predicates' 2 * np bounds cut
// the values into at most 2 * np + 1 ranges, and all rows of a range match the same
// predicates: a row's range is found by a binary search in LDS and the range's predicate mask
// (bit p: predicate p matches) read from a table, ~45 VALU instructions a row for 64
// predicates where testing each predicate takes three a row and predicate.  A wave takes
// 2048 rows.  Search: the wave's coalesced loads (16 bytes a lane) give lane l rows 4l..4l+3
// of each 256; the bounds lie in breadth-first order, so that one level's nodes (at most 64)
// are in different LDS banks.  The ranges' numbers are a byte each and go through LDS to the
// lane that owns the row's bitmap word.  Words: lane l looks up the masks of the 32 rows of
// word l and transposes the 32 x 32 bits in registers (two byte permutes a word, then three
// shift-and-select steps), which leaves the word of every predicate of a half (32
// predicates) in a register; the wave stores 64 consecutive words of each bitmap.  COUNT:
// rows per range by LDS adds, which make each predicate's rows at the end (popcounts of the
// words cost 180 us more at 64 predicates).  1e8 rows, 64 predicates, counted: 732 us by
// testing each predicate, 268 this way, 176 of it when nothing is stored.
struct RankedPreds {
  uint32_t tree[128];             // [1, 2^levels): bounds but the smallest, breadth-first, padded with 2^32 - 1
  uint32_t mask[2][kRankEntries];  // predicates matching range r, 32 per half; the last entry is 0
  uint8_t r0[kMultiPreds], r1[kMultiPreds];  // predicate p matches the ranges [r0, r1)
  uint32_t first;                 // the smallest bound
  int levels;
  uint32_t last;    // the last range
  uint32_t copies;  // copies of the ranges' row counts (a power of two up to 64), stride entries apart
  uint32_t stride;
};

// The bitmap words of the wave's 64 word positions from w0 on: rank4 holds the lane's 32
// ranges, four a word.  FULL: np = 32 * HALVES and every position is inside the bitmap.
template <int HALVES, bool FULL>
__device__ __forceinline__ void store_ranked(uint32_t (&rank4)[8], const uint32_t (&mask)[HALVES][kRankEntries],
                                             int half0, int np, BITS *out, uint64_t stride, uint64_t w0, bool in,
                                             int lane) {
#pragma unroll 1
  for (int h = 0; h < HALVES; h++) {
    uint32_t a[32];
    // the halves look their masks up separately: without this the 32 addresses stay in registers
#pragma unroll
    for (int r = 0; r < 8; r++) asm volatile("" : "+v"(rank4[r]));
#pragma unroll
    for (int r = 0; r < 32; r++) a[r] = mask[h][(rank4[r / 4] >> (8 * (r & 3))) & 0xFF];
    transpose32(a);
    const int p0 = 32 * (half0 + h);
    BITS *o = out + (uint64_t)p0 * stride + w0;
    int left = np - p0;
#pragma unroll
    for (int p = 0; p < 32; p++) {
      if (FULL || (p < left && in)) o[lane] = a[31 - p];
      o += stride;
      // one running address and count, not 32 of each kept in scalar registers
      asm volatile("" : "+s"(o), "+s"(left));
    }
  }
}

// As store_ranked for a workgroup of whole tiles, in step: the waves' words pass through LDS,
// so that one wave stores the workgroup's 2 KB of a predicate at once, and fewer cache lines
// are filled by several stores (256 bytes a store: 2.7 TB/s where the bitmaps do not start on
// lines, 1 KB: 3.9, 4 KB: 4.7).  64 / 32 predicates, workgroups of 256 (1 KB) and of 512: 1e8 rows
// 280 / 173 and 268 / 166 us, 1e8 + 1 297 and 275, 2e8 511 and 500; 40 of 99,999,900 203 and 207.
// Bitmaps at 16-byte offsets take non-temporal 16-byte stores (64 / 32 of 1e8 rows, counted, 4-byte
// stores 273 / 172 us, these 267 / 167; of 2e8 523 / 338, 492 / 313); 4-byte ones are slower
// non-temporal (in workgroups of 256, 64 of 1e8 rows 322 -> 336).  w0: of wave 0.
template <int HALVES, bool FULL>
__device__ __forceinline__ void store_ranked_staged(uint32_t (&rank4)[8], const uint32_t (&mask)[HALVES][kRankEntries],
                                                    uint32_t (&words)[2][kStaged][kStagedBlock], int half0, int np, BITS *out,
                                                    uint64_t stride, uint64_t w0, int wv, int lane) {
#pragma unroll 1
  for (int h = 0; h < HALVES; h++) {
    uint32_t a[32];
#pragma unroll
    for (int r = 0; r < 8; r++) asm volatile("" : "+v"(rank4[r]));  // as in store_ranked
#pragma unroll
    for (int r = 0; r < 32; r++) a[r] = mask[h][(rank4[r / 4] >> (8 * (r & 3))) & 0xFF];
    transpose32(a);
    const int p0 = 32 * (half0 + h) + wv;
    BITS *o = out + (uint64_t)p0 * stride + w0;
    const bool vec = (((uint64_t)out | stride * sizeof(BITS)) & 15) == 0;
    int left = np - p0;
#pragma unroll
    for (int k = 0; k < 32; k += kStaged) {
      uint32_t(&buf)[kStaged][kStagedBlock] = words[k / kStaged % 2];
#pragma unroll
      for (int q = 0; q < kStaged; q++) buf[q][kWave * wv + lane] = a[31 - k - q];
      __syncthreads();
#pragma unroll
      for (int q = 0; q < kStaged; q += kStagedBlock / kWave) {
        if (FULL || left > 0) {
          if (vec) {
#pragma unroll
            for (int j = 0; j < kStagedBlock / kWave / 4; j++)
              __builtin_nontemporal_store(reinterpret_cast<const u32x4 *>(buf[q + wv])[kWave * j + lane],
                                          reinterpret_cast<u32x4 *>(o) + kWave * j + lane);
          } else {
#pragma unroll
            for (int j = 0; j < kStagedBlock / kWave; j++) o[kWave * j + lane] = buf[q + wv][kWave * j + lane];
          }
        }
        o += stride * (kStagedBlock / kWave);
        left -= kStagedBlock / kWave;
        asm volatile("" : "+s"(left));
      }
    }
  }
}

template <int HALVES, bool COUNT, bool FULL, bool STAGED>
__global__ __launch_bounds__(STAGED ? kStagedBlock : kBlock) void k_scan_ranked(const uint32_t *col, uint64_t n, uint64_t whole,
                                                        RankedPreds rp, int np, BITS *out, uint64_t stride,
                                                        uint32_t run, MultiSink sink) {
  constexpr int B = STAGED ? kStagedBlock : kBlock;
  __shared__ uint32_t tree[128];
  __shared__ uint32_t mask[HALVES][kRankEntries];
  __shared__ alignas(16) uint32_t xch[B / kWave][kMultiTileRows / 4];
  __shared__ alignas(16) uint32_t staged[2][kStaged][kStagedBlock];
  // rows per range (COUNT), in as many copies as fit (four for 64 predicates, one a lane for
  // four): a wave's rows of one range would otherwise add to one address one after another
  // (3 predicates over 2^25 rows, counted: 48 us with four copies)
  __shared__ uint32_t hist[COUNT ? kHistEntries : 1];
  __shared__ uint32_t below[COUNT ? kRankEntries : 1];
  const int lane = threadIdx.x & (kWave - 1);
  const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
  const int half0 = HALVES == 1 ? blockIdx.y : 0;  // one half a workgroup: which one
  if (threadIdx.x < 128) tree[threadIdx.x] = rp.tree[threadIdx.x];
  for (int i = threadIdx.x; i < HALVES * kRankEntries; i += B)
    mask[i / kRankEntries][i % kRankEntries] = rp.mask[half0 + i / kRankEntries][i % kRankEntries];
  if (COUNT)
    for (uint32_t i = threadIdx.x; i < kHistEntries; i += B) hist[i] = 0;
  __syncthreads();
  const uint64_t words = words_for_rows(n), ntiles = (n + kMultiTileRows - 1) / kMultiTileRows;
  const uint32_t first = rp.first, root = rp.tree[1];
  const int levels = rp.levels;
  const uint32_t leaf0 = 1u << levels;
  const uint32_t top = rp.last;
  uint32_t *const hw = hist + (COUNT ? (lane & (rp.copies - 1)) * rp.stride : 0);
  uint32_t *const xw = xch[wv];
  // the ranks of the wave's tile, written to xw in row order, back as lane l's 32 rows of word l
  auto exchange = [&](uint32_t(&rank4)[8]) {
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");  // the wave's own exchange: LDS keeps its order
    __builtin_amdgcn_wave_barrier();
    const uint4 ra = *reinterpret_cast<const uint4 *>(xw + 8 * lane), rb = *reinterpret_cast<const uint4 *>(xw + 8 * lane + 4);
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
    rank4[0] = ra.x, rank4[1] = ra.y, rank4[2] = ra.z, rank4[3] = ra.w;
    rank4[4] = rb.x, rank4[5] = rb.y, rank4[6] = rb.z, rank4[7] = rb.w;
  };
  // workgroup step i of XCD x -> tile of wave 0: runs of `run` steps to an XCD, so that lines
  // that neighbouring tiles share (bitmaps that do not start on a 128-byte line) mostly meet
  // in one L2
  const uint64_t xcd = blockIdx.x % kScanXcds, step0 = blockIdx.x / kScanXcds, steps = gridDim.x / kScanXcds;
  auto tile_of = [&](uint64_t i) {
    return (i / run * run * kScanXcds + xcd * run + i % run) * (B / kWave) + wv;
  };
  uint4 v[8];
  auto load = [&](uint64_t t) {
    const uint4 *src = reinterpret_cast<const uint4 *>(col + t * (uint64_t)kMultiTileRows) + lane;
#pragma unroll
    for (int k = 0; k < 8; k++) v[k] = load_stream(src + 64 * k);
  };
  uint64_t step = step0, t = tile_of(step0);
  // whole: every row of the tile exists, and the next tile's loads go out before this one's
  // stores
  auto tile = [&](auto whole_tile) __attribute__((always_inline)) {
    constexpr bool kWhole = decltype(whole_tile)::value;
    uint32_t i[32];
#pragma unroll
    for (int k = 0; k < 8; k++) {
      i[4 * k] = v[k].x >= root ? 3 : 2;
      i[4 * k + 1] = v[k].y >= root ? 3 : 2;
      i[4 * k + 2] = v[k].z >= root ? 3 : 2;
      i[4 * k + 3] = v[k].w >= root ? 3 : 2;
    }
    for (int l = 1; l < levels; l++) {
#pragma unroll
      for (int k = 0; k < 8; k++) {
        const uint32_t t0 = tree[i[4 * k]], t1 = tree[i[4 * k + 1]], t2 = tree[i[4 * k + 2]], t3 = tree[i[4 * k + 3]];
        i[4 * k] = 2 * i[4 * k] + (v[k].x >= t0);
        i[4 * k + 1] = 2 * i[4 * k + 1] + (v[k].y >= t1);
        i[4 * k + 2] = 2 * i[4 * k + 2] + (v[k].z >= t2);
        i[4 * k + 3] = 2 * i[4 * k + 3] + (v[k].w >= t3);
      }
    }
#pragma unroll
    for (int k = 0; k < 8; k++) {
      uint32_t r[4] = {i[4 * k] - leaf0 + (v[k].x >= first), i[4 * k + 1] - leaf0 + (v[k].y >= first),
                       i[4 * k + 2] - leaf0 + (v[k].z >= first), i[4 * k + 3] - leaf0 + (v[k].w >= first)};
#pragma unroll
      for (int j = 0; j < 4; j++) {
        const bool row = kWhole || t * (uint64_t)kMultiTileRows + 256 * k + 4 * lane + j < n;
        // 2^32 - 1 is not below the padding bounds: its range is the last
        if (COUNT && row) atomicAdd(&hw[min(r[j], top)], 1u);
        if (!row) r[j] = kRankEntries - 1;  // the range that no predicate matches
      }
      xw[64 * k + lane] = r[0] | r[1] << 8 | r[2] << 16 | r[3] << 24;
    }
    const uint64_t w0 = t * (kMultiTileRows / 32);
    // loads and stores complete in one order: issued before the stores, the next tile's
    // loads do not wait for them
    step += steps;
    t = tile_of(step);
    if (kWhole && t < whole) load(t);
    uint32_t rank4[8];
    exchange(rank4);
    if constexpr (kWhole && STAGED)
      store_ranked_staged<HALVES, FULL>(rank4, mask, staged, half0, np, out, stride, w0 - wv * (kMultiTileRows / 32), wv, lane);
    else
      store_ranked<HALVES, kWhole && FULL>(rank4, mask, half0, np, out, stride, w0, kWhole || w0 + lane < words, lane);
  };
  // the first tile apart, so that every tile of the loop finds its loads issued before the
  // stores of the one before
  if (t < whole) {
    load(t);
    tile(std::true_type{});
    while (t < whole) tile(std::true_type{});
  }
  // a column that is not 16-byte aligned, and the rows past the whole tiles: the same rows,
  // loaded one by one where they exist
  while (t < ntiles) {
    const uint64_t row = t * (uint64_t)kMultiTileRows + 4 * lane;
#pragma unroll
    for (int k = 0; k < 8; k++) {
      const uint64_t r = row + 256 * k;
      v[k] = make_uint4(r < n ? col[r] : 0, r + 1 < n ? col[r + 1] : 0, r + 2 < n ? col[r + 2] : 0, r + 3 < n ? col[r + 3] : 0);
    }
    tile(std::false_type{});
  }
  if (COUNT) {
    __syncthreads();
    // rows of each range over the copies, then rows below each range, then each predicate's
    for (uint32_t r = threadIdx.x; r < kRankEntries; r += B) {
      uint32_t a = 0;
      if (r <= top)
        for (uint32_t c = 0; c < rp.copies; c++) a += hist[c * rp.stride + r];
      below[r] = a;
    }
    __syncthreads();
    if (threadIdx.x < kWave) {
      const int r = 2 * lane;  // 2 * kWave + 2 entries: the last two follow the scan
      const uint32_t a = below[r], b = below[r + 1], last = below[2 * kWave];
      uint32_t sum = a + b;
#pragma unroll
      for (int o = 1; o < kWave; o <<= 1) {
        const uint32_t u = __shfl_up(sum, o, kWave);
        if (lane >= o) sum += u;
      }
      below[r] = sum - a - b;
      below[r + 1] = sum - b;
      if (lane == kWave - 1) {
        below[2 * kWave] = sum;
        below[2 * kWave + 1] = sum + last;
      }
    }
    __syncthreads();
    const int p = 32 * half0 + (int)threadIdx.x;
    if (threadIdx.x < 32 * HALVES && p < np)
      multi_count(sink, p, below[rp.r1[p]] - below[rp.r0[p]]);
  }
}

// ------------------------------------------------------------------ host launchers

static inline bool aligned16(const void *p) { return ((uintptr_t)p & 15) == 0; }

static unsigned grid_for(uint64_t work_items, unsigned per_block, unsigned cap) {
  uint64_t g = (work_items + per_block - 1) / per_block;
  if (g < 1) g = 1;
  if (g > cap) g = cap;
  return (unsigned)g;
}

static unsigned stream_grid_cap() { return (unsigned)std::max(1, device_cu_count()) * 8u; }

// The scan kernel runs one 1024-row tile per wave without a grid-stride loop up to this
// many workgroups (16 waves per CU of 256 CUs in flight with room to spare), which measured
// faster than a persistent grid of 8 workgroups per CU.
static unsigned scan_grid_cap() { return (unsigned)std::min<int>(kMaxCountBlocks, std::max(1, device_cu_count()) * 128); }

// A counted scan runs 32 workgroups per compute unit over the tiles instead: each workgroup
// then ends with one count reduction and one accumulator add for ~3 of the uncounted grid's
// workgroups.  On uniform columns scanned back to back: 1e8-row counted scan 68.9 -> 65.2
// us, 4-column conjunction 262 -> 254 us (8 per CU: 67.2 and 257); on the mixed-distribution
// 1e8 x 4 table, queries interleaved with other paths, the conjunctions were unchanged.
static unsigned counted_scan_grid_cap() { return (unsigned)std::min<int>(kMaxCountBlocks, std::max(1, device_cu_count()) * 32); }

template <int OP>
static hipError_t launch_bitop(BITS *dst, const BITS *a, const BITS *b, uint64_t words,
                               uint32_t value, hipStream_t s) {
  if (words == 0) return hipSuccess;
  const bool vec = aligned16(dst) && (!reads_a(OP) || aligned16(a)) && (!reads_b(OP) || aligned16(b));
  const unsigned grid = grid_for(vec ? (words + 3) / 4 : words, kBlock, stream_grid_cap());
  if (vec)
    hipLaunchKernelGGL((k_bitop<OP, true>), dim3(grid), dim3(kBlock), 0, s, dst, a, b, words, value);
  else
    hipLaunchKernelGGL((k_bitop<OP, false>), dim3(grid), dim3(kBlock), 0, s, dst, a, b, words, value);
  return hipGetLastError();
}

constexpr int kTileU = 4;  // uint4 loads per lane per column per tile: 1024 rows per wave tile

template <int C, int MODE, bool COUNT>
static hipError_t launch_scan_c(const ColPreds<C> &p, uint64_t n, BITS *out, CountSink sink,
                                hipStream_t s) {
  bool vec = true;
  for (int c = 0; c < C; c++) vec = vec && aligned16(p.col[c]);
  unsigned grid;
  if (vec) {
    const uint64_t ntiles = n / (256ull * kTileU);
    grid = grid_for(std::max<uint64_t>(ntiles, 1), kBlock / kWave, sink.out ? counted_scan_grid_cap() : scan_grid_cap());
    hipLaunchKernelGGL((k_scan_tiles<C, kTileU, MODE, COUNT>), dim3(grid), dim3(kBlock), 0, s, p,
                       n, out, sink);
  } else {
    grid = grid_for((n + 63) / 64, kBlock / kWave, stream_grid_cap());
    hipLaunchKernelGGL((k_scan_rows<C, MODE, COUNT>), dim3(grid), dim3(kBlock), 0, s, p, n, out,
                       sink);
  }
  hipError_t e = hipGetLastError();
  if (e != hipSuccess || !COUNT) return e;
  return launch_count_finalize(sink, grid, s);
}

template <int C, int MODE>
static hipError_t launch_scan(const ColPreds<C> &p, uint64_t n, BITS *out,
                              unsigned long long *count, hipStream_t s, uint32_t *partials) {
  if (count) {
    const CountSink sink = partials ? CountSink{count, partials, nullptr} : stream_count_sink(count, s);
    if (!sink.partials && !sink.acc) return hipErrorOutOfMemory;
    return launch_scan_c<C, MODE, true>(p, n, out, sink, s);
  }
  return launch_scan_c<C, MODE, false>(p, n, out, CountSink{nullptr, nullptr, nullptr}, s);
}

// Empty predicate: all-zero bitmap (set/and modes), zero count.
static hipError_t launch_empty(uint64_t n, BITS *out, unsigned long long *count, int mode,
                               hipStream_t s) {
  if (count) {
    hipLaunchKernelGGL(k_zero_u64, dim3(1), dim3(1), 0, s, count);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
  }
  if (mode == kStoreXor) return hipSuccess;
  return launch_bitop<kFill>(out, nullptr, nullptr, words_for_rows(n), 0u, s);
}

template <int C>
static hipError_t scan_group(const CODE *const *cols, const CODE *lo, const CODE *hi, uint64_t n,
                             BITS *out, unsigned long long *count, int mode, hipStream_t s,
                             uint32_t *partials) {
  ColPreds<C> p;
  for (int c = 0; c < C; c++) {
    p.col[c] = cols[c];
    p.lo[c] = lo[c];
    p.span[c] = hi[c] - lo[c];
  }
  if (mode == kStoreSet) return launch_scan<C, kStoreSet>(p, n, out, count, s, partials);
  if (mode == kStoreXor) return launch_scan<C, kStoreXor>(p, n, out, count, s, partials);
  return launch_scan<C, kStoreAnd>(p, n, out, count, s, partials);
}

// Conjunction over any number of columns: groups of up to 4 columns per pass, the first
// pass in `mode`, later passes AND into the result; the popcount on the last pass, its
// per-workgroup partials in `partials` (kMaxCountBlocks slots) when given, else in the
// calling thread's scratch for the stream.
hipError_t scan_conjunction(const CODE *const *cols, const CODE *lo, const CODE *hi, int ncols,
                            uint64_t n, BITS *out, unsigned long long *count, int mode,
                            hipStream_t s, uint32_t *partials) {
  if (ncols < 1 || !cols || !lo || !hi) return hipErrorInvalidValue;
  if (mode == kStoreXor && ncols > 4) return hipErrorInvalidValue;
  if (n == 0) return count ? launch_empty(0, out, count, kStoreXor, s) : hipSuccess;
  if (!out) return hipErrorInvalidValue;
  for (int c = 0; c < ncols; c++) {
    if (!cols[c]) return hipErrorInvalidValue;
    if (lo[c] > hi[c]) return launch_empty(n, out, count, mode, s);
  }
  int done = 0;
  while (done < ncols) {
    const int g = std::min(4, ncols - done);
    const bool last = done + g == ncols;
    const int m = done == 0 ? mode : (int)kStoreAnd;
    unsigned long long *cnt = last ? count : nullptr;
    hipError_t e;
    switch (g) {
      case 1: e = scan_group<1>(cols + done, lo + done, hi + done, n, out, cnt, m, s, partials); break;
      case 2: e = scan_group<2>(cols + done, lo + done, hi + done, n, out, cnt, m, s, partials); break;
      case 3: e = scan_group<3>(cols + done, lo + done, hi + done, n, out, cnt, m, s, partials); break;
      default: e = scan_group<4>(cols + done, lo + done, hi + done, n, out, cnt, m, s, partials); break;
    }
    if (e != hipSuccess) return e;
    done += g;
  }
  return hipSuccess;
}

// Range table of up to kMultiPreds predicates: the distinct bounds lo and hi + 1 in order
// (range r = the values with r bounds at or below them), as k_scan_ranked searches them.
static RankedPreds rank_table(const CODE *lo, const CODE *hi, int np) {
  RankedPreds t;
  uint32_t b[2 * kMultiPreds];  // no host memory: a caller in C cannot take an exception
  size_t nb = 0;
  for (int p = 0; p < np; p++) {
    if (lo[p] > hi[p]) continue;
    b[nb++] = lo[p];
    if (hi[p] != 0xFFFFFFFFu) b[nb++] = hi[p] + 1;
  }
  std::sort(b, b + nb);
  nb = std::unique(b, b + nb) - b;
  memset(t.mask, 0, sizeof(t.mask));
  memset(t.r0, 0, sizeof(t.r0));
  memset(t.r1, 0, sizeof(t.r1));
  for (int p = 0; p < np; p++) {
    if (lo[p] > hi[p]) continue;
    const size_t r0 = std::lower_bound(b, b + nb, lo[p]) - b + 1;
    // a value of 2^32 - 1 also passes the padding bounds: the last range's mask fills up
    const size_t r1 = hi[p] == 0xFFFFFFFFu ? kRankEntries - 1 : std::lower_bound(b, b + nb, hi[p] + 1) - b + 1;
    t.r0[p] = (uint8_t)r0;
    t.r1[p] = (uint8_t)r1;
    for (size_t r = r0; r < r1; r++) t.mask[p / 32][r] |= 1u << (p % 32);
  }
  t.last = (uint32_t)nb;
  t.stride = (t.last + 1) | 1;  // odd: the copies start in different LDS banks
  t.copies = 64;
  while (t.copies * t.stride > kHistEntries) t.copies /= 2;
  t.first = nb == 0 ? 0xFFFFFFFFu : b[0];
  t.levels = 1;
  while ((1u << t.levels) < nb) t.levels++;  // 2^levels - 1 nodes for the bounds but the first
  for (uint32_t &v : t.tree) v = 0xFFFFFFFFu;
  for (int l = 0; l < t.levels; l++)  // node i of level l: the bound in the middle of its span
    for (uint32_t i = 0; i < 1u << l; i++) {
      const size_t at = ((2 * (size_t)i + 1) << (t.levels - 1 - l));  // 1 .. 2^levels - 1
      if (at < nb) t.tree[(1u << l) + i] = b[at];
    }
  return t;
}

template <int HALVES>
static void launch_ranked(const uint32_t *col, uint64_t n, const RankedPreds &t, int np, BITS *out, uint64_t stride,
                          uint32_t run, const MultiSink &sink, dim3 grid, hipStream_t s) {
  const bool full = np == 32 * HALVES * (int)grid.y;
  const bool staged = ((uintptr_t)out % 128 || stride * sizeof(BITS) % 128) &&
                      (uint64_t)np * words_for_rows(n) * sizeof(BITS) >= kStagedBytes;
  // staged, a workgroup's waves go in step: whole tiles for all of them
  const uint64_t tiles = aligned16(col) ? n / kMultiTileRows : 0, whole = staged ? tiles / (kStagedBlock / kWave) * (kStagedBlock / kWave) : tiles;
  if (staged) {
    grid.x = (grid.x * kBlock / kStagedBlock + kScanXcds - 1) / kScanXcds * kScanXcds;
    run = std::max<uint32_t>(1, run * kBlock / kStagedBlock);
  }
  auto go = [&](auto count, auto full, auto staged) {
    k_scan_ranked<HALVES, decltype(count)::value, decltype(full)::value, decltype(staged)::value>
        <<<grid, decltype(staged)::value ? kStagedBlock : kBlock, 0, s>>>(col, n, whole, t, np, out, stride, run, sink);
  };
  auto pick = [&](auto count) {
    constexpr std::true_type yes{};
    constexpr std::false_type no{};
    if (staged)
      full ? go(count, yes, yes) : go(count, no, yes);
    else
      full ? go(count, yes, no) : go(count, no, no);
  };
  sink.counts ? pick(std::true_type{}) : pick(std::false_type{});
}

// Predicates up to which a pass tests each one (k_scan_multi) instead of searching
// (k_scan_ranked).  The search costs a row the same for any number of predicates up to 32 and
// half as much again up to 64, a test three instructions a row and predicate; on a short
// column the search's chain of dependent steps (one tile a wave) is what shows.  Measured, tests
// against search, counted / not: 2^18 rows, 64 predicates 7.5 : 9.1 / 6.5 : 7.4; 2^19 rows, 36:
// 7.8 : 9.3 / 6.2 : 7.4, 48: 9.6 : 9.3 / 7.7 : 7.6; 2^20 rows, 20: 8.5 : 8.9 / 6.8 : 6.9, 24: 9.6 :
// 9.0 / 7.7 : 7.0, 64: 14.1 : 10.1 / 12.1 : 8.0; 1.5e6 rows, 16: 9.7 : 9.2 / 7.7 : 6.8; 4.2e6 rows, 8:
// 9.8 : 10.0 / 8.3 : 7.8, 10: 10.5 : 10.7 / 9.0 : 8.4, 12: 11.6 : 10.7 / 10.1 : 8.4; 6e6 rows, 8: 12.0 : 12.2 /
// 10.1 : 9.6, 10: 14.4 : 13.2 / 12.6 : 10.7; counted, 1e8 rows, 5: 95 : 99, 8: 110 : 100, 16: 194 : 117, 32:
// 374 : 166, 64: 730 : 268 (250 when every bitmap starts on a 128-byte line: what is left is the
// writes' rate).
static int direct_preds(uint64_t n) {
  return n < 3u << 17 ? kMultiPreds : n < 1u << 20 ? 40 : n < 5u << 18 ? 20 : n < 1u << 22 ? 16 : n < 5u << 20 ? 9 : 8;
}

hipError_t scan_ranges(const CODE *col, uint64_t n, const CODE *lo, const CODE *hi, int np, BITS *out,
                       uint64_t stride, unsigned long long *counts, hipStream_t s) {
  if (!col || !lo || !hi || np < 1 || (n && !out)) return hipErrorInvalidValue;
  const uint64_t words = words_for_rows(n);
  if (np > 1 && stride < words) return hipErrorInvalidValue;
  if (n == 0) {
    if (counts) return hipMemsetAsync(counts, 0, (size_t)np * sizeof(unsigned long long), s);
    return hipSuccess;
  }
  const unsigned cus = (unsigned)std::max(1, device_cu_count());
  MultiSink sink{};
  if (counts) {
    void *acc = nullptr;
    bool *fresh = nullptr;
    hipStreamCaptureStatus capture = hipStreamCaptureStatusNone;
    hipError_t e = thread_scratch(kScratchMulti, s, 2 * kMultiAccBytes, 0, &acc, nullptr, &fresh);
    if (e == hipSuccess && s) e = hipStreamIsCapturing(s, &capture);
    if (e != hipSuccess) return e;
    sink.acc = static_cast<unsigned long long *>(acc);
    const bool captured = capture != hipStreamCaptureStatusNone;
    if (captured) sink.acc += kMultiAccBytes / sizeof(*sink.acc);
    // The kernels leave the accumulators at zero; new ones start there too.  A captured launch may be
    // replayed on any stream, beside the ones that its own has queued by then: it has accumulators
    // apart from theirs, and clears them, which two replays at once may leave in any state.
    if (*fresh || captured) {
      hipLaunchKernelGGL(k_zero_multi, dim3(1), dim3(kBlock), 0, s, sink.acc);
      e = hipGetLastError();
      if (e != hipSuccess) return e;
      if (!captured) *fresh = false;
    }
  }
  for (int p0 = 0; p0 < np; p0 += kMultiPreds) {  // one pass over the column per 64 predicates
    const int k = std::min(kMultiPreds, np - p0);
    BITS *o = out + (uint64_t)p0 * stride;
    unsigned grid;
    if (counts) sink.counts = counts + p0;
    if (k > direct_preds(n)) {
      const RankedPreds t = rank_table(lo + p0, hi + p0, k);
      const uint64_t wgtiles = (n + kMultiTileRows * (kBlock / kWave) - 1) / (kMultiTileRows * (kBlock / kWave));
      // a tile a wave while the workgroups all fit at once (4 per compute unit); a long
      // column takes more, shorter workgroups, which even out (1e8 rows, 64 predicates: 338
      // us with 4 per compute unit, 322 with 16, stored from registers; 1e7 rows: 32 against 38), and gives an XCD
      // runs of 16 steps (337 against 366 us)
      const bool large = wgtiles >= cus * 16;
      grid = grid_for(wgtiles, 1, std::min<unsigned>(kMultiMaxGrid, cus * (large ? 16 : 4)));
      grid = (grid + kScanXcds - 1) / kScanXcds * kScanXcds;
      const uint32_t run = large ? 16 : 1;
      if (k <= 32)
        launch_ranked<1>(col, n, t, k, o, stride, run, sink, dim3(grid), s);
      else if (grid < cus * 2)  // the halves in workgroups of their own, so that a short column fills the device
        launch_ranked<1>(col, n, t, k, o, stride, run, sink, dim3(grid, 2), s);
      else
        launch_ranked<2>(col, n, t, k, o, stride, run, sink, dim3(grid), s);
    } else {
      const uint64_t ntiles = aligned16(col) ? n / kMultiTileRows : 0;
      const uint64_t waves = std::max<uint64_t>(ntiles, (n - ntiles * kMultiTileRows + 63) / 64);
      grid = grid_for(waves, kBlock / kWave, std::min<unsigned>(kMultiMaxGrid, stream_grid_cap() * 2));
      MultiPreds mp{};
      for (int p = 0; p < k; p++) {
        if (lo[p0 + p] > hi[p0 + p]) {
          mp.empty |= 1ull << p;
        } else {
          mp.lo[p] = lo[p0 + p];
          mp.span[p] = hi[p0 + p] - lo[p0 + p];
        }
      }
      // predicate groups: enough workgroups for 4 per compute unit, at least 8 predicates each
      const unsigned want = cus * 4;
      const int groups = (int)std::max<unsigned>(1, std::min<unsigned>((k + 7) / 8, (want + grid - 1) / grid));
      const int pper = (k + groups - 1) / groups;
      const dim3 g2(grid, (unsigned)((k + pper - 1) / pper));
      if (counts)
        hipLaunchKernelGGL(k_scan_multi<true>, g2, dim3(kBlock), 0, s, col, n, ntiles, mp, k, pper, o, stride,
                           sink);
      else
        hipLaunchKernelGGL(k_scan_multi<false>, g2, dim3(kBlock), 0, s, col, n, ntiles, mp, k, pper, o, stride,
                           sink);
    }
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
  }
  return hipSuccess;
}

hipError_t bitmap_and_popcount(const BITS *const *bms, int nb, uint64_t n, BITS *out,
                               unsigned long long *count, hipStream_t s) {
  if (nb < 1 || !bms || (!out && nb > kMaxAnd)) return hipErrorInvalidValue;
  const uint64_t words = words_for_rows(n);
  if (words == 0) {
    if (!count) return hipSuccess;
    hipLaunchKernelGGL(k_zero_u64, dim3(1), dim3(1), 0, s, count);
    return hipGetLastError();
  }
  const CountSink counted = count ? stream_count_sink(count, s) : CountSink{nullptr, nullptr, nullptr};
  if (count && !counted.acc) return hipErrorOutOfMemory;
  // Chains of more than kMaxAnd inputs: AND the first kMaxAnd into `out`, continue from it.
  int done = 0;
  while (true) {
    BitmapSet set;
    int k = 0;
    if (done > 0) set.bm[k++] = out;
    while (k < kMaxAnd && done < nb) {
      if (!bms[done]) return hipErrorInvalidValue;
      set.bm[k++] = bms[done++];
    }
    const bool last = done == nb;
    bool vec = !out || aligned16(out);
    for (int i = 0; i < k; i++) vec = vec && aligned16(set.bm[i]);
    const unsigned grid = grid_for(vec ? (words + 3) / 4 : words, kBlock, stream_grid_cap());
    const uint32_t lm = tail_mask(n);
    const CountSink sink = last ? counted : CountSink{nullptr, nullptr, nullptr};
#define RTS_LAUNCH_AND(V, C)                                                                    \
  hipLaunchKernelGGL((k_and_popcount<V, C>), dim3(grid), dim3(kBlock), 0, s, set, k, words, lm, \
                     out, sink)
    if (vec) {
      if (sink.out) RTS_LAUNCH_AND(true, true); else RTS_LAUNCH_AND(true, false);
    } else {
      if (sink.out) RTS_LAUNCH_AND(false, true); else RTS_LAUNCH_AND(false, false);
    }
#undef RTS_LAUNCH_AND
    hipError_t e = hipGetLastError();
    if (e == hipSuccess && sink.out) e = launch_count_finalize(sink, grid, s);
    if (e != hipSuccess || last) return e;
  }
}

hipError_t bitop(int op, BITS *dst, const BITS *a, const BITS *b, uint64_t words, uint32_t value,
                 hipStream_t s) {
  switch (op) {
    case kCopy: return launch_bitop<kCopy>(dst, a, b, words, value, s);
    case kNot: return launch_bitop<kNot>(dst, a, b, words, value, s);
    case kAndNot: return launch_bitop<kAndNot>(dst, a, b, words, value, s);
    case kAnd: return launch_bitop<kAnd>(dst, a, b, words, value, s);
    case kOr: return launch_bitop<kOr>(dst, a, b, words, value, s);
    case kFill: return launch_bitop<kFill>(dst, a, b, words, value, s);
    case kXorWith: return launch_bitop<kXorWith>(dst, a, b, words, value, s);
    default: return hipErrorInvalidValue;
  }
}

hipError_t flip_rows(BITS *bm, uint64_t rows, hipStream_t s) {
  if (rows == 0) return hipSuccess;
  const unsigned grid = grid_for(rows / 32 + 1, kBlock, stream_grid_cap());
  hipLaunchKernelGGL(k_flip_rows, dim3(grid), dim3(kBlock), 0, s, bm, rows);
  return hipGetLastError();
}

}  // namespace rts
