// sort_rows.hip -- stable radix sort of (value, row) by value, 8 bits a pass.
//
// A pass counts its digit per tile, turns the counts into each (digit, tile)'s first place
// (one scan over digits and tiles) and moves the tiles' rows there.  Moving is bound by
// memory, so the rows of a tile are laid out by digit in LDS first and each digit's go out
// as one run (32 rows, 128 bytes, of a tile of 8192 with all digits in use).  Values and rows
// go through the same LDS one after the other, half the LDS of laying out pairs.  The first
// pass reads no rows (a row's number is its place).  1e8 rows: 1.85 ms for uniform values,
// 1.58 for one value (the library sort that this replaced: 3.0 ms); a pass moves its 1.6 GB
// in 0.33 ms, at the rate of a copy, and counts in 0.11.  1e6 rows: 0.07 ms, by the launches.
#include <hip/hip_runtime.h>
#include <hipcub/hipcub.hpp>

#include <algorithm>

#include "common.h"
#include "sort_rows.h"

namespace rts {
namespace {

constexpr int kDigits = 256, kDigitBits = 8;
// Workgroups of k_sort_move, and their rows a thread.  Twice the waves at half the rows of
// 512 x 16, with as many rows in flight and shorter chains of ranking: 1e8 uniform rows 2.01 ->
// 1.85 ms, 2e7 0.41 -> 0.40 (1024 x 10, x 12 and x 16: 1.87, 1.79, 2.25 and 0.39, 0.42, 0.52).
constexpr int kThreads = 1024, kSteps = 8;
constexpr int kShortThreads = 512;
constexpr int kCountThreads = 256;
constexpr int kCopies = 4;  // one / eight copies: 2.57 / 1.60 ms for 1e8 equal values, 1.91 / 2.04 for uniform ones
constexpr unsigned kRun = 32, kShortRun = 1;

// Tile of a workgroup: workgroup b runs on XCD b % 8, and an XCD takes runs of kRun
// neighbouring tiles, whose counts share lines and whose digits' runs join, so that these
// lines are completed in one L2 (workgroups of 512, 1e8 uniform rows: 2.83 ms with neighbouring
// tiles on different XCDs; of 1024: 1.99 with runs of 8, 1.85 with 32, 1.77 with 64, which make
// 6e6 rows take 186 us against 166).
constexpr unsigned kSortXcds = 8;
__device__ __forceinline__ int64_t tile_of_block(unsigned run) {
  const unsigned j = blockIdx.x / kSortXcds;
  return (int64_t)(j / run) * (kSortXcds * run) + blockIdx.x % kSortXcds * run + j % run;
}

// counts[d * ntiles + t], SHORT: counts[t * kDigits + d], = rows of tile t with digit d.
// kCopies count arrays a wave, so that the lanes of a skewed column do not all add to one
// address.
template <int TILE, bool SHORT>
__global__ __launch_bounds__(kCountThreads) void k_sort_counts(const CODE *val, int64_t n, int shift, int64_t ntiles,
                                                               uint32_t *counts) {
  constexpr int kArrays = kCountThreads / kWave * kCopies, kPad = kDigits + 1;
  constexpr int kVec = TILE / 4 / kCountThreads;
  __shared__ uint32_t cnt[kArrays * kPad];
  const int64_t t = tile_of_block(SHORT ? kShortRun : kRun);
  if (t >= ntiles) return;
  for (int i = threadIdx.x; i < kArrays * kPad; i += kCountThreads) cnt[i] = 0;
  __syncthreads();
  uint32_t *mine = cnt + (threadIdx.x / kWave * kCopies + threadIdx.x % kCopies) * kPad;
  auto add = [&](CODE v) { atomicAdd(&mine[(v >> shift) & (kDigits - 1)], 1u); };
  const int64_t r0 = t * TILE;
  if (r0 + TILE <= n && ((uintptr_t)val & 15) == 0) {
    const uint4 *src = reinterpret_cast<const uint4 *>(val + r0) + threadIdx.x;
    uint4 v[kVec];
#pragma unroll
    for (int i = 0; i < kVec; i++) v[i] = src[i * kCountThreads];
#pragma unroll
    for (int i = 0; i < kVec; i++) add(v[i].x), add(v[i].y), add(v[i].z), add(v[i].w);
  } else {
    const int64_t r1 = min(n, r0 + TILE);
#pragma unroll 8
    for (int64_t r = r0 + threadIdx.x; r < r1; r += kCountThreads) add(val[r]);
  }
  __syncthreads();
  for (int d = threadIdx.x; d < kDigits; d += kCountThreads) {
    uint32_t c = 0;
#pragma unroll
    for (int a = 0; a < kArrays; a++) c += cnt[a * kPad + d];
    counts[SHORT ? t * kDigits + d : d * ntiles + t] = c;
  }
}

// LDS of the ranking of a tile's rows by digit.
template <int THREADS>
struct RankLds {
  alignas(16) uint32_t wcnt[THREADS / kWave][kDigits];
  uint32_t part[kDigits / kWave];
};

// place[i] = slot of the thread's row i (row w0 + i * kWave of the tile, below `left`) when
// the tile's rows are laid out by digit.  Returns, for threads d below kDigits, the digit's
// first slot.
template <int THREADS, int STEPS>
__device__ __forceinline__ uint32_t rank_tile(RankLds<THREADS> &l, CODE (&x)[STEPS], int shift, uint32_t w0, uint32_t left,
                                              uint32_t (&place)[STEPS]) {
  constexpr int kWaves = THREADS / kWave;
  const int lane = threadIdx.x & (kWave - 1), wv = threadIdx.x / kWave;
  const int d = threadIdx.x;  // the digit of threads below kDigits
  for (int i = threadIdx.x; i < kWaves * kDigits; i += THREADS) (&l.wcnt[0][0])[i] = 0;
  __syncthreads();
  // a row's place among its wave's rows of the digit: the count so far plus the lanes before
  // it with the digit (one ballot a bit)
  uint32_t *const mine = l.wcnt[wv];
#pragma unroll
  for (int i = 0; i < STEPS; i++) {
    const uint32_t digit = (x[i] >> shift) & (kDigits - 1);
    const bool row = w0 + i * kWave < left;
    const uint64_t rows = __ballot(row);
    uint32_t lo = (uint32_t)rows, hi = (uint32_t)(rows >> 32);
#pragma unroll
    for (int b = 0; b < kDigitBits; b++) {
      const uint32_t bit = (uint32_t)((int32_t)(digit << (31 - b)) >> 31);
      const uint64_t with = __ballot(bit != 0);
      lo &= ~((uint32_t)with ^ bit);
      hi &= ~((uint32_t)(with >> 32) ^ bit);
    }
    const uint32_t before = __builtin_amdgcn_mbcnt_hi(hi, __builtin_amdgcn_mbcnt_lo(lo, 0));
    place[i] = mine[digit] + before;
    // the wave's LDS accesses run in order: this step's reads, then the first lane's add
    if (before == 0 && row) atomicAdd(&mine[digit], (uint32_t)(__popc(lo) + __popc(hi)));
    asm volatile("" : "+v"(x[i]));  // the digits' LDS addresses are worked out again below, not kept
  }
  __syncthreads();
  // slots of the tile: digits in order, a digit's waves in order
  uint32_t total = 0;
  if (d < kDigits)
    for (int w = 0; w < kWaves; w++) total += l.wcnt[w][d];
  uint32_t upto = total;
#pragma unroll
  for (int o = 1; o < kWave; o <<= 1) {
    const uint32_t u = __shfl_up(upto, o, kWave);
    if (lane >= o) upto += u;
  }
  if (lane == kWave - 1 && d < kDigits) l.part[wv] = upto;
  __syncthreads();
  uint32_t first = 0;
  if (d < kDigits) {
    uint32_t slot = upto - total;
    for (int w = 0; w < wv; w++) slot += l.part[w];
    first = slot;
#pragma unroll
    for (int w = 0; w < kWaves; w++) {
      const uint32_t c = l.wcnt[w][d];
      l.wcnt[w][d] = slot;
      slot += c;
    }
  }
  __syncthreads();
#pragma unroll
  for (int i = 0; i < STEPS; i++) place[i] += mine[(x[i] >> shift) & (kDigits - 1)];
  return first;
}

// For threads d below kDigits, the first place of digit d of tile t from all tiles' counts
// (tile after tile): the rows of lower digits and, of the digit, of the tiles before.  A wave
// adds up every kWaves-th tile, four digits a lane, with kPlaceTiles tiles' loads in flight:
// their latency is what a pass over a short column waits for.
template <int THREADS>
__device__ __forceinline__ uint32_t first_places(uint32_t *lds, RankLds<THREADS> &l, const uint32_t *counts,
                                                 int64_t ntiles, int64_t t) {
  constexpr int kWaves = THREADS / kWave, kPlaceTiles = 16;
  static_assert(kDigits == 4 * kWave, "four digits a lane");
  const int d = threadIdx.x, lane = threadIdx.x & (kWave - 1), wv = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
  const int tiles = (int)ntiles, own = (int)t;
  uint4 before = make_uint4(0, 0, 0, 0), all = before;
  const uint4 *src = reinterpret_cast<const uint4 *>(counts) + lane;
  for (int u0 = wv; u0 < tiles; u0 += kWaves * kPlaceTiles) {
    uint4 c[kPlaceTiles];
#pragma unroll
    for (int k = 0; k < kPlaceTiles; k++) {
      const int u = u0 + k * kWaves;
      c[k] = u < tiles ? src[(int64_t)u * kWave] : make_uint4(0, 0, 0, 0);
    }
#pragma unroll
    for (int k = 0; k < kPlaceTiles; k++) {
      const uint32_t m = u0 + k * kWaves < own ? 0xFFFFFFFFu : 0;
      all.x += c[k].x, all.y += c[k].y, all.z += c[k].z, all.w += c[k].w;
      before.x += c[k].x & m, before.y += c[k].y & m, before.z += c[k].z & m, before.w += c[k].w & m;
    }
  }
  reinterpret_cast<uint4 *>(lds + wv * kDigits)[lane] = before;
  reinterpret_cast<uint4 *>(l.wcnt[wv])[lane] = all;
  __syncthreads();
  uint32_t first = 0, total = 0, upto = 0;
  if (d < kDigits) {
#pragma unroll
    for (int w = 0; w < kWaves; w++) first += lds[w * kDigits + d], total += l.wcnt[w][d];
    upto = total;
#pragma unroll
    for (int o = 1; o < kWave; o <<= 1) {
      const uint32_t u = __shfl_up(upto, o, kWave);
      if (lane >= o) upto += u;
    }
    if (lane == kWave - 1) l.part[d / kWave] = upto;
  }
  __syncthreads();
  if (d < kDigits)
    for (int w = 0; w < d / kWave; w++) first += l.part[w];
  return first + upto - total;
}

// The rows of a tile to their places of this pass; places: the scanned counts, the first place
// of each (digit, tile), or, SHORT, the counts, from which the workgroup makes its own tile's.
template <int THREADS, int STEPS, bool SHORT, bool FIRST>
__global__ __launch_bounds__(THREADS) __attribute__((amdgpu_waves_per_eu(5))) void k_sort_move(
    const CODE *val, const uint32_t *pos, int64_t n, int shift, int64_t ntiles, const uint32_t *places, CODE *out_val,
    uint32_t *out_pos) {
  constexpr int kWaves = THREADS / kWave, kTile = THREADS * STEPS;
  static_assert(!SHORT || kTile >= kWaves * kDigits, "first_places");
  alignas(16) __shared__ uint32_t stage[kTile];
  __shared__ RankLds<THREADS> rank;
  __shared__ uint32_t delta[kDigits];  // place - slot in the tile
  const int lane = threadIdx.x & (kWave - 1), wv = threadIdx.x / kWave;
  const int d = threadIdx.x;  // the digit of threads below kDigits
  const int64_t t = tile_of_block(SHORT ? kShortRun : kRun);
  if (t >= ntiles) return;
  const int64_t c0 = t * kTile;
  const uint32_t left = (uint32_t)min((int64_t)kTile, n - c0);
  const uint32_t w0 = wv * (kTile / kWaves) + lane;
  CODE x[STEPS];
  uint32_t p[STEPS], place[STEPS];
#pragma unroll
  for (int i = 0; i < STEPS; i++) x[i] = w0 + i * kWave < left ? val[c0 + w0 + i * kWave] : 0;
  const uint32_t first = SHORT ? first_places(stage, rank, places, ntiles, t) : d < kDigits ? places[d * ntiles + t] : 0;
  const uint32_t slot = rank_tile(rank, x, shift, w0, left, place);
  if (d < kDigits) delta[d] = first - slot;
#pragma unroll
  for (int i = 0; i < STEPS; i++)
    if (w0 + i * kWave < left) stage[place[i]] = x[i];
  if (!FIRST) {
#pragma unroll
    for (int i = 0; i < STEPS; i++) p[i] = w0 + i * kWave < left ? pos[c0 + w0 + i * kWave] : 0;
  }
  __syncthreads();
  uint32_t dest[STEPS];
#pragma unroll
  for (int i = 0; i < STEPS; i++) {
    const uint32_t e = threadIdx.x + i * THREADS;
    if (e < left) {
      const CODE v = stage[e];
      dest[i] = delta[(v >> shift) & (kDigits - 1)] + e;
      out_val[dest[i]] = v;
    }
  }
  __syncthreads();
#pragma unroll
  for (int i = 0; i < STEPS; i++)
    if (w0 + i * kWave < left) stage[place[i]] = FIRST ? (uint32_t)c0 + w0 + i * kWave : p[i];
  __syncthreads();
#pragma unroll
  for (int i = 0; i < STEPS; i++) {
    const uint32_t e = threadIdx.x + i * THREADS;
    if (e < left) out_pos[dest[i]] = stage[e];
  }
}

// Shorter columns are sorted by the library, which takes fewer launches for them (3e4 rows 39 us
// against 44, 65536 41 against 37).
constexpr int64_t kLibraryRows = (int64_t)1 << 16;
// Up to this many rows a pass does without a scan, every workgroup adds up the counts of all
// tiles instead, and the fewer the rows, the smaller are the tiles, so that they fill the
// device.  Sorts of 200, 300, 500 thousand, 1, 1.4, 2, 3 and 4 million rows, us: tiles of 2048
// rows 47, 50, 58, 95, 142, 211, 385, 619; of 4096 58, 52, 57, 69, 96, 107, 168, 238; of 8192
// 71, 78, 69, 81, 101, 90, 119, 135; with a scan 93, 102, 96, 106, 122, 108, 128, 129.
constexpr int64_t kShortRows = (int64_t)7 << 19;
int short_steps(int64_t n) { return n <= 3 << 17 ? 4 : n <= 3 << 19 ? 8 : 16; }

__global__ void k_iota(uint32_t *p, uint32_t n) {
  const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) p[i] = i;
}

int64_t tiles_of(int64_t n) {
  const int64_t rows = n <= kShortRows ? kShortThreads * short_steps(n) : kThreads * kSteps;
  return (n + rows - 1) / rows;
}

// One pass without a scan.
template <int STEPS>
hipError_t short_pass(const CODE *v, const uint32_t *p, int64_t n, int shift, int64_t tiles, uint32_t *counts, CODE *ov,
                      uint32_t *op, dim3 grid, hipStream_t s) {
  hipLaunchKernelGGL((k_sort_counts<kShortThreads * STEPS, true>), grid, dim3(kCountThreads), 0, s, v, n, shift, tiles, counts);
  const hipError_t e = hipGetLastError();
  if (e != hipSuccess) return e;
  if (p)
    hipLaunchKernelGGL((k_sort_move<kShortThreads, STEPS, true, false>), grid, dim3(kShortThreads), 0, s, v, p, n,
                       shift, tiles, counts, ov, op);
  else
    hipLaunchKernelGGL((k_sort_move<kShortThreads, STEPS, true, true>), grid, dim3(kShortThreads), 0, s, v, p, n,
                       shift, tiles, counts, ov, op);
  return hipGetLastError();
}

size_t up16(size_t b) { return (b + 15) & ~(size_t)15; }

size_t scan_bytes(int64_t tiles) {
  size_t need = 0;
  (void)hipcub::DeviceScan::ExclusiveSum(nullptr, need, (uint32_t *)nullptr, (uint32_t *)nullptr, tiles * kDigits,
                                         (hipStream_t) nullptr);
  return need;
}

}  // namespace

size_t sort_rows_workspace(int64_t n) {
  if (n < kLibraryRows) {
    size_t need = 0;
    (void)hipcub::DeviceRadixSort::SortPairs(nullptr, need, (const CODE *)nullptr, (CODE *)nullptr,
                                             (const uint32_t *)nullptr, (uint32_t *)nullptr, (int)n, 0, 32,
                                             (hipStream_t) nullptr);
    return up16(n * sizeof(uint32_t)) + up16(need);
  }
  const int64_t tiles = tiles_of(n);
  return 2 * up16(n * sizeof(uint32_t)) + 2 * up16(tiles * kDigits * sizeof(uint32_t)) + up16(scan_bytes(tiles));
}

hipError_t sort_rows(const CODE *col, int64_t n, CODE *val, uint32_t *pos, void *work, hipStream_t s) {
  const int64_t tiles = tiles_of(n);
  if (n < kLibraryRows) {
    uint32_t *const iota = static_cast<uint32_t *>(work);
    size_t need = sort_rows_workspace(n) - up16(n * sizeof(uint32_t));
    hipLaunchKernelGGL(k_iota, dim3((unsigned)((n + kBlock - 1) / kBlock)), dim3(kBlock), 0, s, iota, (uint32_t)n);
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    return hipcub::DeviceRadixSort::SortPairs(static_cast<char *>(work) + up16(n * sizeof(uint32_t)), need, col, val,
                                              iota, pos, (int)n, 0, 32, s);
  }
  const unsigned round = kSortXcds * (n <= kShortRows ? kShortRun : kRun);
  const dim3 grid((unsigned)((tiles + round - 1) / round * round));
  char *w = static_cast<char *>(work);
  auto take = [&w](size_t bytes) {
    char *p = w;
    w += up16(bytes);
    return p;
  };
  CODE *const wval = reinterpret_cast<CODE *>(take(n * sizeof(CODE)));
  uint32_t *const wpos = reinterpret_cast<uint32_t *>(take(n * sizeof(uint32_t)));
  uint32_t *const counts = reinterpret_cast<uint32_t *>(take(tiles * kDigits * sizeof(uint32_t)));
  uint32_t *const places = reinterpret_cast<uint32_t *>(take(tiles * kDigits * sizeof(uint32_t)));
  const size_t scan = scan_bytes(tiles);
  const CODE *v = col;
  const uint32_t *p = nullptr;
  for (int pass = 0; pass < 32 / kDigitBits; pass++) {  // an even number: the last pass writes val and pos
    const int shift = pass * kDigitBits;
    CODE *const ov = pass & 1 ? val : wval;
    uint32_t *const op = pass & 1 ? pos : wpos;
    hipError_t e;
    if (n <= kShortRows) {
      const int steps = short_steps(n);
      e = steps == 4   ? short_pass<4>(v, p, n, shift, tiles, counts, ov, op, grid, s)
          : steps == 8 ? short_pass<8>(v, p, n, shift, tiles, counts, ov, op, grid, s)
                       : short_pass<16>(v, p, n, shift, tiles, counts, ov, op, grid, s);
    } else {
      hipLaunchKernelGGL((k_sort_counts<kThreads * kSteps, false>), grid, dim3(kCountThreads), 0, s, v, n, shift, tiles,
                         counts);
      e = hipGetLastError();
      size_t need = scan;
      if (e == hipSuccess) e = hipcub::DeviceScan::ExclusiveSum(w, need, counts, places, tiles * kDigits, s);
      if (e != hipSuccess) return e;
      if (p)
        hipLaunchKernelGGL((k_sort_move<kThreads, kSteps, false, false>), grid, dim3(kThreads), 0, s, v, p, n, shift,
                           tiles, places, ov, op);
      else
        hipLaunchKernelGGL((k_sort_move<kThreads, kSteps, false, true>), grid, dim3(kThreads), 0, s, v, p, n, shift,
                           tiles, places, ov, op);
      e = hipGetLastError();
    }
    if (e != hipSuccess) return e;
    v = ov;
    p = op;
  }
  return hipSuccess;
}

}  // namespace rts
