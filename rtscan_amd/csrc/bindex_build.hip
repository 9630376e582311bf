// bindex_build.hip -- GPU build of the device-resident BinDex (init_bindex,
// bindex.cpp:599-671, and its GPU-driver twin init_bindex_in_GPU, bindex_cuda.cpp:164-282).
//
// The reference sorts on the host with an unstable parallel sort, builds the 127 filter
// vectors with 127 host passes, then issues one cudaMalloc + cudaMemcpy per 3276-row block
// (~30k per column at 1e8 rows).  Here everything stays on the device: one stable radix
// sort of (value, row), one kernel for the area starts, the bin starts (each area cut into
// `sub` equal-count bins) and their ranks, one pass over the column for all bins-1
// filter vectors and the bin keys, and one stable partition of the rows by bin key for the
// row-ordered B lists and their tile directory.
#include <hipcub/hipcub.hpp>

#include <stdio.h>
#include <string.h>

#include <algorithm>
#include <mutex>

#include "bindex_dev.h"
#include "sort_rows.h"

namespace rts {

// What the build finds out on the device, for the host in one copy and for the kernels after.
struct BuildHead {
  int64_t idx[kAreas];       // first sorted slot of each area
  int64_t rk[2 * kMaxBins];  // as start_ranks
  CODE starts[kAreas], estarts[kMaxBins];
  uint32_t boff[kMaxBins + 1];
  CODE data_max;
  uint8_t light[kMaxBins];  // a bin start of at most kLightStartRows rows goes into its bin's list
};

// Area starts (bindex.cpp:613-631): start[i] = sorted[i * avg]; if it equals the previous
// start the area begins mid-run at i * avg, otherwise at the first occurrence of the value.
// Bin starts: area a (sorted slots [idx[a], idx[a + 1])) cut into `sub` equal-count bins;
// bin a * sub + j starts at the value in slot idx[a] + j * len / sub, so bin a * sub is
// the area's own start.  Ranks of the bin starts: searched between the neighbouring bins'
// slots, unless a run reaches over one.  Bound by latency, chains of a dozen or two loads in
// one workgroup (15 us at 1e6 rows, 26 at 1e8).  Three kernels with the host between them, and the
// blocks' slots from the host, in its place: a build of 1e6 rows and 256 bins 423 us against 308
// (1e5: 353, 245); with what has changed elsewhere since, 240.
constexpr int kStartThreads = 1024;
__global__ __launch_bounds__(kStartThreads) void k_build_starts(const CODE *sorted, int64_t n, int sub, BuildHead *head) {
  __shared__ int64_t idx[kAreas + 1];
  const int i = threadIdx.x;
  if (i < kAreas) {
    const int64_t avg = n / kAreas;
    const CODE v = sorted[i * avg];
    int64_t hi = i * avg;
    if (i > 0 && v != sorted[(i - 1) * avg]) {  // first slot in (lo, hi] holding v
      int64_t lo = (i - 1) * avg;
      while (lo + 1 < hi) {
        const int64_t mid = lo + (hi - lo) / 2;
        if (sorted[mid] < v)
          lo = mid;
        else
          hi = mid;
      }
    }
    idx[i] = hi;
    head->idx[i] = hi;
    head->starts[i] = v;
  }
  if (i == 0) {
    idx[kAreas] = n;
    head->data_max = sorted[n - 1];
  }
  __syncthreads();
  const int bins = kAreas * sub;
  auto slot = [&](int b) {
    const int64_t s0 = idx[b / sub];
    return s0 + b % sub * (idx[b / sub + 1] - s0) / sub;
  };
  for (int r = i; r < 2 * bins; r += kStartThreads) {
    const int b = r / 2;
    const bool above = r & 1;  // first slot with a value > v, else with one >= v
    const int64_t at = slot(b);
    const CODE v = sorted[at];
    int64_t lo, hi;
    if (above) {
      const int64_t next = b + 1 < bins ? slot(b + 1) : n;
      const bool ends = next == n || sorted[next] > v;
      lo = ends ? at + 1 : next + 1;
      hi = ends ? next : n;
    } else {
      const int64_t prev = b > 0 ? slot(b - 1) : 0;
      const bool begins = sorted[prev] < v;
      lo = begins ? prev + 1 : 0;
      hi = begins ? at : prev;
    }
    while (lo < hi) {
      const int64_t mid = lo + (hi - lo) / 2;
      const CODE x = sorted[mid];
      if (above ? x > v : x >= v)
        hi = mid;
      else
        lo = mid + 1;
    }
    head->rk[r] = lo;
    const int64_t other = __shfl_xor((long long)lo, 1, kWave);
    if (above) {
      head->estarts[b] = v;
      head->light[b] = lo - other <= kLightStartRows;
    }
  }
}

// out[i] = sorted[i * kRankSample] for i < m.
__global__ void k_rank_samples(const CODE *sorted, int64_t m, CODE *out) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < m) out[i] = sorted[i * kRankSample];
}

// 2 i + (v >= t), in two instructions.
static __device__ __forceinline__ uint32_t descend_from(uint32_t i, uint32_t v, uint32_t t) {
  asm("v_cmp_ge_u32 vcc, %1, %2\n\tv_addc_co_u32 %0, vcc, %0, %0, vcc" : "+v"(i) : "v"(v), "v"(t) : "vcc");
  return i;
}

// Eight bytes, x = rows 0 to 3 and y = 4 to 7 from the top byte down, as an 8 x 8 bit matrix
// transposed: then byte 3 - k of x (k < 4) and byte 7 - k of y hold bit 7 - k of the rows,
// row 0 topmost.
__device__ __forceinline__ void transpose8(uint32_t &x, uint32_t &y) {
  uint32_t t = (x ^ x >> 7) & 0x00AA00AAu;
  x ^= t ^ t << 7;
  t = (y ^ y >> 7) & 0x00AA00AAu;
  y ^= t ^ t << 7;
  t = (x ^ x >> 14) & 0x0000CCCCu;
  x ^= t ^ t << 14;
  t = (y ^ y >> 14) & 0x0000CCCCu;
  y ^= t ^ t << 14;
  t = (x & 0xF0F0F0F0u) | (y >> 4 & 0x0F0F0F0Fu);
  y = (x << 4 & 0xF0F0F0F0u) | (y & 0x0F0F0F0Fu);
  x = t;
}

// One pass over the column: all bins-1 filter vectors (fv[k] bit i = x_i < estart[k+1],
// set_fv_val_less, bindex.cpp:553-560) and each row's list key (its bin if estart[bin] <
// x, or x = estart[bin] with light[bin] set, else `bins` = in no list).  A wave takes 2048
// consecutive rows, 64 words of every filter vector.  Each lane finds the bins t of 32 rows
// (a search of M levels in LDS, the rows' chains side by side; rows 256 j + 4 lane + i, so
// that loads and the keys' stores are consecutive over the lanes), which go through LDS to
// the lane that makes their word, and are transposed there into M bit slices, MSB-first like
// the bitmaps.  With t = 16 h + l, fv[16 h + l] = (rows below h) | (rows of h) & (rows of at
// most l): one instruction a word once the 16 words of l and those of h are made.  A row past
// n is in no filter vector; the words past the last (up to the 64-word padded stride) are
// written as zeros.
//
// Bound by the writes (1e8 rows, 128 bins: 1.6 GB of filter vectors, 0.2 of keys, 438 us).  Taking
// each fv[k] from all M slices, a search loop a row and the slices a bit at a time cost 170
// instructions a row, and 620 us; now 50.  1e6 rows, 256 bins: 44 -> 14 us.
constexpr int kFvTileRows = 2048;
template <int M>
__global__ __launch_bounds__(kBlock) void k_build_fvs(const CODE *col, int64_t n, const CODE *starts,
                                                      const uint8_t *light, BITS *fvs, int64_t fv_stride,
                                                      uint16_t *keys) {
  constexpr int kBins = 1 << M;
  __shared__ uint32_t tree[kBins];   // [1, kBins): starts but the first, breadth-first
  __shared__ CODE unlisted[kBins];   // the value of the bin that is in no list, or one that isn't in the bin
  __shared__ alignas(16) uint16_t xch[kBlock / kWave][kFvTileRows];
  for (int i = threadIdx.x; i < kBins; i += kBlock) {
    // a light start's bin holds no value below it, nor (a start of 0) 2^32 - 1, the last bin's
    unlisted[i] = light[i] ? starts[i] - 1 : starts[i];
    if (i) {
      const int level = 31 - __clz(i);
      tree[i] = starts[(2 * (i - (1 << level)) + 1) << (M - 1 - level)];
    }
  }
  __syncthreads();
  const int lane = threadIdx.x & (kWave - 1), wv = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
  uint16_t *const xw = xch[wv];
  const int64_t wave = (int64_t)blockIdx.x * (kBlock / kWave) + wv, nwaves = (int64_t)gridDim.x * (kBlock / kWave);
  const int64_t ntiles = (n + kFvTileRows - 1) / kFvTileRows;
  const uint32_t root = tree[1], node2 = tree[2], node3 = tree[3];
  for (int64_t tile = wave; tile < ntiles; tile += nwaves) {
    const int64_t row0 = tile * kFvTileRows;
    const bool whole = row0 + kFvTileRows <= n;
    CODE x[32];
    if (whole && ((uintptr_t)col & 15) == 0) {
      const uint4 *src = reinterpret_cast<const uint4 *>(col + row0) + lane;
#pragma unroll
      for (int j = 0; j < 8; j++) {
        const uint4 v = load_stream(src + 64 * j);
        x[4 * j] = v.x, x[4 * j + 1] = v.y, x[4 * j + 2] = v.z, x[4 * j + 3] = v.w;
      }
    } else {
#pragma unroll
      for (int j = 0; j < 32; j++) x[j] = col[min(row0 + 256 * (j / 4) + 4 * lane + j % 4, n - 1)];
    }
    uint32_t t[32];
#pragma unroll
    for (int j = 0; j < 32; j++) {
      const bool up = x[j] >= root;
      t[j] = descend_from(up ? 3 : 2, x[j], up ? node3 : node2);
    }
    for (int l = 2; l < M; l++) {
#pragma unroll
      for (int j = 0; j < 32; j++) t[j] = descend_from(t[j], x[j], tree[t[j]]);
    }
#pragma unroll
    for (int j = 0; j < 32; j += 4) {
      uint32_t key[4];
#pragma unroll
      for (int i = 0; i < 4; i++) {
        t[j + i] -= kBins;
        key[i] = x[j + i] != unlisted[t[j + i]] ? t[j + i] : (uint32_t)kBins;
      }
      const int at = 64 * j + 4 * lane;
      const uint2 k4 = make_uint2(key[0] | key[1] << 16, key[2] | key[3] << 16);
      if (whole) {
        *reinterpret_cast<uint2 *>(keys + row0 + at) = k4;
      } else {
#pragma unroll
        for (int i = 0; i < 4; i++)
          if (row0 + at + i < n) keys[row0 + at + i] = (uint16_t)key[i];
      }
      *reinterpret_cast<uint2 *>(xw + at) = make_uint2(t[j] | t[j + 1] << 16, t[j + 2] | t[j + 3] << 16);
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");  // the wave's own exchange: LDS keeps its order
    __builtin_amdgcn_wave_barrier();
    // slices of the lane's 32 rows, in groups of eight
    uint32_t part[4][2], slice[M], high[2] = {0, 0};
#pragma unroll
    for (int g = 0; g < 4; g++) {
      const uint4 v = reinterpret_cast<const uint4 *>(xw + 32 * lane)[g];  // rows 8 g + 1, 8 g, ...
      part[g][0] = __builtin_amdgcn_perm(v.x, v.y, 0x04060002);
      part[g][1] = __builtin_amdgcn_perm(v.z, v.w, 0x04060002);
      transpose8(part[g][0], part[g][1]);
      if (M > 8) {
#pragma unroll
        for (int b = 8; b < M; b++)
          for (const uint32_t w : {v.x, v.y, v.z, v.w})
            high[b - 8] = high[b - 8] << 2 | (w >> b & 1) << 1 | (w >> (16 + b) & 1);
      }
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
#pragma unroll
    for (int b = 0; b < M; b++) {
      if (b < 8) {  // byte b % 4 of part[g][0] for the upper, [1] for the lower four bits; group 0 topmost
        constexpr uint32_t kPair = 0x04000C0C;
        const int h = b < 4;
        const uint32_t sel = kPair + 0x01010000u * (b % 4);
        slice[b] = __builtin_amdgcn_perm(part[0][h], part[1][h], sel) |
                   __builtin_amdgcn_perm(part[2][h], part[3][h], 0x0C0C0400u + 0x0101u * (b % 4));
      } else {
        slice[b] = high[b - 8];
      }
    }
    const int64_t left = n - row0 - 32 * lane;  // rows of the lane's word
    const uint32_t valid = left >= 32 ? ~0u : left <= 0 ? 0u : ~0u << (32 - left);
    uint32_t upto[16];  // rows with t % 16 <= l
#pragma unroll
    for (int l = 0; l < 16; l++) {
      uint32_t eq = ~0u;
#pragma unroll
      for (int b = 0; b < 4; b++) eq &= l >> b & 1 ? slice[b] : ~slice[b];
      upto[l] = l ? upto[l - 1] | eq : eq;
    }
    BITS *dst = fvs + tile * (kFvTileRows / 32);
    uint32_t below = 0;  // rows with t / 16 < h
#pragma unroll 1
    for (int h = 0; h < kBins / 16; h++) {
      uint32_t eq = valid;
#pragma unroll
      for (int b = 4; b < M; b++) eq &= slice[b] ^ (h >> (b - 4) & 1 ? 0u : ~0u);
#pragma unroll
      for (int l = 0; l < 16; l++) {
        if (l < 15 || h < kBins / 16 - 1) dst[lane] = below | (eq & upto[l]);
        dst += fv_stride;
        asm volatile("" : "+s"(dst));  // one running address, not 16
      }
      below |= eq;
    }
  }
}

// B lists by one stable partition of the rows by list key, with no sort and no gather: rows
// per (bin, directory tile) -> one exclusive scan over bins and tiles, which is the tile
// directory -> every tile's entries written where the directory says.  (Sorting 16-bit keys
// with their rows and gathering the values afterwards, a random 4-byte read a row, took 2.7
// ms at 1e8 rows and 128 bins; this takes 0.5.)

// counts[k * (ntiles + 1) + t] = rows of tile t of tile_rows rows with key k (k < bins), and 0
// for t = ntiles.  One workgroup per tile, and one for the zeros; LDS adds, a count copy per
// wave.
__global__ __launch_bounds__(kBlock) void k_list_counts(const uint16_t *keys, int64_t n, int bins, int64_t ntiles,
                                                        int tile_rows, uint32_t *counts) {
  extern __shared__ uint32_t cnt[];  // kBlock / kWave copies of bins + 1
  const int64_t t = blockIdx.x;
  const int copies = kBlock / kWave, per = bins + 1;
  for (int i = threadIdx.x; i < copies * per; i += kBlock) cnt[i] = 0;
  __syncthreads();
  uint32_t *mine = cnt + threadIdx.x / kWave * per;
  const int64_t r0 = t * tile_rows, r1 = std::min<int64_t>(n, r0 + tile_rows);
  if (r0 + tile_rows <= n) {
    const uint4 *src = reinterpret_cast<const uint4 *>(keys + r0);  // 8 keys each
#pragma unroll 4
    for (int i = threadIdx.x; i < tile_rows / 8; i += kBlock) {
      const uint4 v = src[i];
      for (const uint32_t w : {v.x, v.y, v.z, v.w}) {
        if ((int)(w & 0xFFFF) < bins) atomicAdd(&mine[w & 0xFFFF], 1u);
        if ((int)(w >> 16) < bins) atomicAdd(&mine[w >> 16], 1u);
      }
    }
  } else {
    for (int64_t r = r0 + threadIdx.x; r < r1; r += kBlock)
      if (keys[r] < bins) atomicAdd(&mine[keys[r]], 1u);
  }
  __syncthreads();
  for (int k = threadIdx.x; k < bins; k += kBlock) {
    uint32_t c = 0;
    for (int w = 0; w < copies; w++) c += cnt[w * per + k];
    counts[k * (ntiles + 1) + t] = c;
  }
}

// The entries (row, value) of tiles of tile_rows rows with the directory `dir`, a workgroup a
// tile, in chunks of kPartRows rows.  In a chunk each wave takes kPartRows / waves rows, 64
// a step: a row's place among its wave's rows of the same key is the count so far (LDS, one
// counter per key and wave) plus the lanes before it with the same key (NB ballots, one per
// key bit).  The chunk is then laid out by key in LDS and written out in that order, so that
// a bin's entries go to memory as one run (kPartRows / bins entries of 8 bytes) and in row
// order.
constexpr int kPartRows = 4096;
constexpr int kPartRowBits = 12;
template <int NB>
__global__ __launch_bounds__(kBlock) void k_list_entries(const CODE *col, const uint16_t *keys, int64_t n, int bins,
                                                         int64_t ntiles, int tile_rows, const uint32_t *dir, uint2 *bent) {
  constexpr int kWaves = kBlock / kWave, kSteps = kPartRows / kBlock, kPer = (1 << (NB - 1)) / kBlock + 1;
  extern __shared__ uint2 part_lds[];
  uint2 *const stage = part_lds;                                           // kPartRows entries
  uint32_t *const wcnt = reinterpret_cast<uint32_t *>(stage + kPartRows);  // per wave: bins + 1
  uint32_t *const next = wcnt + kWaves * (bins + 1);                       // bins: the bin's next entry
  uint32_t *const delta = next + bins;                                     // bins: entry - slot of the chunk
  __shared__ uint32_t wsum[kWaves];
  const int lane = threadIdx.x & (kWave - 1), wv = threadIdx.x / kWave;
  const int64_t t = blockIdx.x;
  for (int k = threadIdx.x; k < bins; k += kBlock) next[k] = dir[k * (ntiles + 1) + t];
  const int64_t p0 = t * tile_rows, p1 = std::min<int64_t>(n, p0 + tile_rows);
  for (int64_t c0 = p0; c0 < p1; c0 += kPartRows) {
    uint32_t key[kSteps], place[kSteps];
    CODE x[kSteps];
    const uint32_t left = (uint32_t)std::min<int64_t>(kPartRows, p1 - c0);
    const uint32_t w0 = wv * (kPartRows / kWaves) + lane;
#pragma unroll
    for (int i = 0; i < kSteps; i++) {
      const uint32_t r = w0 + i * kWave;
      key[i] = r < left ? keys[c0 + r] : (uint32_t)bins;
      x[i] = r < left ? col[c0 + r] : 0;
    }
    for (int i = threadIdx.x; i < kWaves * (bins + 1); i += kBlock) wcnt[i] = 0;
    __syncthreads();  // also: the chunk before has been written out
    uint32_t *const mine = wcnt + wv * (bins + 1);
#pragma unroll
    for (int i = 0; i < kSteps; i++) {
      uint64_t same = ~0ull;
#pragma unroll
      for (int b = 0; b < NB; b++) {
        const bool bit = (key[i] >> b) & 1;
        const uint64_t with = __ballot(bit);
        same &= bit ? with : ~with;
      }
      const uint32_t before = __builtin_amdgcn_mbcnt_hi((uint32_t)(same >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)same, 0));
      place[i] = mine[key[i]] + before;
      // the wave's LDS accesses run in order: this step's reads, then the first lane's add
      if (before == 0) atomicAdd(&mine[key[i]], (uint32_t)__popcll(same));
    }
    __syncthreads();
    // slots of the chunk: bins in order, a bin's waves in order (kPer bins a thread)
    uint32_t total[kPer], sum = 0;
    const int k0 = threadIdx.x * kPer;
#pragma unroll
    for (int q = 0; q < kPer; q++) {
      total[q] = 0;
      if (k0 + q < bins)
        for (int w = 0; w < kWaves; w++) total[q] += wcnt[w * (bins + 1) + k0 + q];
      sum += total[q];
    }
    uint32_t upto = sum;
#pragma unroll
    for (int o = 1; o < kWave; o <<= 1) {
      const uint32_t u = __shfl_up(upto, o, kWave);
      if (lane >= o) upto += u;
    }
    if (lane == kWave - 1) wsum[wv] = upto;
    __syncthreads();
    uint32_t slot = upto - sum, entries = 0;
    for (int w = 0; w < kWaves; w++) {
      if (w < wv) slot += wsum[w];
      entries += wsum[w];
    }
#pragma unroll
    for (int q = 0; q < kPer; q++) {
      if (k0 + q < bins) {
        delta[k0 + q] = next[k0 + q] - slot;
        next[k0 + q] += total[q];
        for (int w = 0; w < kWaves; w++) {
          const uint32_t c = wcnt[w * (bins + 1) + k0 + q];
          wcnt[w * (bins + 1) + k0 + q] = slot;
          slot += c;
        }
      }
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < kSteps; i++)
      if ((int)key[i] < bins) stage[mine[key[i]] + place[i]] = make_uint2(key[i] << kPartRowBits | (w0 + i * kWave), x[i]);
    __syncthreads();
    for (uint32_t e = threadIdx.x; e < entries; e += kBlock) {
      const uint2 v = stage[e];
      bent[delta[v.x >> kPartRowBits] + e] = make_uint2((uint32_t)c0 + (v.x & (kPartRows - 1)), v.y);
    }
  }
}

// bdir[k * (ntiles + 1) + t] = the same of a directory of `parts` times the tiles.
__global__ void k_thin_directory(const uint32_t *fine, int bins, int64_t ntiles, int parts, uint32_t *bdir) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= bins * (ntiles + 1)) return;
  const int64_t k = i / (ntiles + 1), t = i % (ntiles + 1);
  bdir[i] = fine[k * (ntiles * parts + 1) + t * parts];
}

// boff[k] = boff2[k] = the directory's first entry of bin k, for k in [0, bins] (its rows end at the next bin's).
__global__ void k_bin_offsets(const uint32_t *bdir, int64_t ntiles, int bins, uint32_t *boff, uint32_t *boff2) {
  const int k = blockIdx.x * blockDim.x + threadIdx.x;
  if (k <= bins) boff[k] = boff2[k] = k < bins ? bdir[k * (ntiles + 1)] : bdir[bins * (ntiles + 1) - 1];
}

// bdir[k * (ntiles + 1) + t] = first entry of bin k with row >= t * tile_rows
__global__ void k_tile_directory(const uint2 *bent, const uint32_t *boff, int bins, int64_t ntiles,
                                 int64_t tile_rows, uint32_t *bdir) {
  const int64_t id = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  const int64_t per = ntiles + 1;
  if (id >= per * bins) return;
  const int k = (int)(id / per);
  const uint64_t row = (uint64_t)(id % per) * (uint64_t)tile_rows;
  uint32_t lo = boff[k], hi = boff[k + 1];
  while (lo < hi) {
    const uint32_t mid = lo + (hi - lo) / 2;
    if (bent[mid].x < row)
      lo = mid + 1;
    else
      hi = mid;
  }
  bdir[id] = lo;
}

hipError_t launch_tile_directory(const rts_bindex_dev *d, int64_t ntiles, int64_t tile_rows, uint32_t *bdir,
                                 hipStream_t s) {
  const int64_t items = (int64_t)d->bins * (ntiles + 1);
  hipLaunchKernelGGL(k_tile_directory, dim3((unsigned)((items + kBlock - 1) / kBlock)), dim3(kBlock), 0, s,
                     d->bent, d->boff, d->bins, ntiles, tile_rows, bdir);
  return hipGetLastError();
}

// Blocks of an area of `len` rows (init_area, bindex.cpp:410-427).
__host__ __device__ __forceinline__ int64_t area_blocks(int64_t len) {
  return (len + RTS_BLOCK_INIT_SIZE - 1) / RTS_BLOCK_INIT_SIZE;
}

// First and last value of every 3276-row block of every area, in order, for the host-side
// in_which_block.  A workgroup an area.
__global__ __launch_bounds__(kAreas) void k_block_bounds(const CODE *sorted, int64_t n, const int64_t *idx, CODE *first,
                                                         CODE *last) {
  __shared__ unsigned long long before;
  const int a = blockIdx.x, t = threadIdx.x;
  auto len = [&](int k) { return (k + 1 < kAreas ? idx[k + 1] : n) - idx[k]; };
  if (t == 0) before = 0;
  __syncthreads();
  if (t < a) atomicAdd(&before, (unsigned long long)area_blocks(len(t)));
  __syncthreads();
  const int64_t s0 = idx[a], rows = len(a), blocks = area_blocks(rows);
  for (int64_t b = t; b < blocks; b += kAreas) {
    const int64_t r = b * RTS_BLOCK_INIT_SIZE;
    first[before + b] = sorted[s0 + r];
    last[before + b] = sorted[s0 + min(r + RTS_BLOCK_INIT_SIZE, rows) - 1];
  }
}

static unsigned blocks_for(int64_t items, int per = kBlock) {
  int64_t g = (items + per - 1) / per;
  const int64_t cap = (int64_t)device_cu_count() * 16;
  return (unsigned)std::max<int64_t>(1, std::min(g, cap));
}

#define RTS_TRY(x)                      \
  do {                                  \
    hipError_t _e = (x);                \
    if (_e != hipSuccess) {             \
      err = _e;                         \
      goto fail;                        \
    }                                   \
  } while (0)

// rk[2k] = first sorted slot with value >= estarts[k], rk[2k + 1] = first with value >
// estarts[k] (binary searches over the sorted column, one thread per bin start).
__global__ void k_start_ranks(const CODE *sorted, int64_t n, const CODE *estarts, int bins, int64_t *rk) {
  const int k = blockIdx.x * blockDim.x + threadIdx.x;
  if (k >= bins) return;
  const CODE v = estarts[k];
  int64_t lo = 0, hi = n;  // first slot with sorted >= v
  while (lo < hi) {
    const int64_t mid = (lo + hi) >> 1;
    if (sorted[mid] < v)
      lo = mid + 1;
    else
      hi = mid;
  }
  rk[2 * k] = lo;
  hi = n;  // first slot with sorted > v
  while (lo < hi) {
    const int64_t mid = (lo + hi) >> 1;
    if (sorted[mid] <= v)
      lo = mid + 1;
    else
      hi = mid;
  }
  rk[2 * k + 1] = lo;
}

hipError_t start_ranks(const rts_bindex_dev *d, std::vector<int64_t> &rk, hipStream_t s) {
  const int bins = d->bins;
  CODE *est = nullptr;
  int64_t *rk_d = nullptr;
  rk.assign(2 * (size_t)bins, 0);
  hipError_t e = pool_alloc(&est, bins * sizeof(CODE));
  if (e == hipSuccess) e = pool_alloc(&rk_d, 2 * (size_t)bins * sizeof(int64_t));
  if (e == hipSuccess) e = hipMemcpyAsync(est, d->estarts.data(), bins * sizeof(CODE), hipMemcpyHostToDevice, s);
  if (e == hipSuccess) {
    hipLaunchKernelGGL(k_start_ranks, dim3((bins + kBlock - 1) / kBlock), dim3(kBlock), 0, s, d->sorted_val, d->n,
                       est, bins, rk_d);
    e = hipGetLastError();
  }
  if (e == hipSuccess) e = hipMemcpyAsync(rk.data(), rk_d, 2 * (size_t)bins * sizeof(int64_t), hipMemcpyDeviceToHost, s);
  if (e == hipSuccess) e = hipStreamSynchronize(s);
  pool_free(est, e == hipSuccess);
  pool_free(rk_d, e == hipSuccess);
  return e;
}

void mark_complete_bins(rts_bindex_dev *d, const std::vector<int64_t> &rk) {
  d->complete.assign(d->bins, 0);
  for (int k = 0; k < d->bins; k++) {
    const int64_t rows = (k + 1 < d->bins ? rk[2 * (k + 1)] : d->n) - rk[2 * k];
    d->complete[k] = (int64_t)(d->boff_host[k + 1] - d->boff_host[k]) == rows;
  }
}

hipError_t rank_samples(rts_bindex_dev *d, hipStream_t s) {
  const int64_t m = (d->n + kRankSample - 1) / kRankSample;
  CODE *smp = nullptr;
  d->rank_samples.assign(m, 0);
  hipError_t e = pool_alloc(&smp, m * sizeof(CODE));
  if (e == hipSuccess) {
    hipLaunchKernelGGL(k_rank_samples, dim3((unsigned)((m + kBlock - 1) / kBlock)), dim3(kBlock), 0, s,
                       d->sorted_val, m, smp);
    e = hipGetLastError();
  }
  if (e == hipSuccess) e = hipMemcpyAsync(d->rank_samples.data(), smp, m * sizeof(CODE), hipMemcpyDeviceToHost, s);
  if (e == hipSuccess) e = hipStreamSynchronize(s);
  pool_free(smp, e == hipSuccess);
  return e;
}

static void free_dev(rts_bindex_dev *d) {
  if (!d) return;
  // queries of any stream may still read the arrays: wait for them, as hipFree does
  int dev = 0;
  const bool here = hipGetDevice(&dev) == hipSuccess;
  const bool away = here && d->device != dev && hipSetDevice(d->device) == hipSuccess;
  const bool idle = here && (away || d->device == dev) && device_wait();
  for (void *p : {(void *)d->sorted_val, (void *)d->sorted_pos, (void *)d->fvs, (void *)d->bent, (void *)d->boff,
                  (void *)d->bdir})
    pool_free(p, idle);
  if (away) (void)hipSetDevice(dev);
  (void)hipFree(d->owned_column);
  delete d;
}

// pos_block views of every block over the sorted arrays `val` / `pos` (device or host):
// block b of area k covers slots [start_k + b * 3276, ...) (init_pos_block,
// bindex.cpp:300-309).
static void make_block_views(const rts_bindex_dev *d, CODE *val, int32_t *pos, std::vector<pos_block> &blk,
                             std::vector<pos_block *> &ptrs) {
  blk.clear();
  for (int k = 0; k < kAreas; k++) {
    const int64_t len = d->area_len[k];
    const int nb = (int)(len <= RTS_BLOCK_INIT_SIZE ? 1 : (len + RTS_BLOCK_INIT_SIZE - 1) / RTS_BLOCK_INIT_SIZE);
    for (int b = 0; b < nb; b++) {
      const int64_t s0 = d->area_start[k] + (int64_t)b * RTS_BLOCK_INIT_SIZE;
      const int64_t s1 = std::min<int64_t>(s0 + RTS_BLOCK_INIT_SIZE, d->area_start[k] + len);
      blk.push_back(pos_block{(POSTYPE *)(pos + s0), val + s0, (int)(s1 - s0)});
    }
  }
  ptrs.resize(blk.size());
  for (size_t i = 0; i < blk.size(); i++) ptrs[i] = &blk[i];
}

// The reference-shaped descriptor (bindex.h:126-138) over a complete device index: areas
// and their blocks (bindex.cpp:633-652), start values, counts, filter-vector pointers.
void describe(BinDex *bx, rts_bindex_dev *d, const CODE *col) {
  d->area_store.resize(kAreas);
  d->area_gpu_store.resize(kAreas);
  make_block_views(d, d->sorted_val, d->sorted_pos, d->blk_dev, d->blkp_dev);
  int64_t b0 = 0;
  for (int k = 0; k < kAreas; k++) {
    Area &a = d->area_store[k];
    const int64_t len = d->area_len[k];
    a.blockNum = (int)(len <= RTS_BLOCK_INIT_SIZE ? 1 : (len + RTS_BLOCK_INIT_SIZE - 1) / RTS_BLOCK_INIT_SIZE);
    a.length = (int)len;
    a.start = (POSTYPE)d->area_start[k];
    a.blockFirst = d->block_first.data() + b0;
    a.blockLast = d->block_last.data() + b0;
    a.blocks = d->blkp_host.empty() ? nullptr : d->blkp_host.data() + b0;
    Area &g = d->area_gpu_store[k];
    g = a;
    g.blocks = d->blkp_dev.data() + b0;
    b0 += a.blockNum;
  }
  bx->length = (POSTYPE)d->n;
  bx->data_min = d->starts[0];
  for (int k = 0; k < kAreas; k++) {
    bx->areas[k] = &d->area_store[k];
    bx->areaStartValues[k] = d->starts[k];
    bx->area_counts[k] = (POSTYPE)(d->area_start[k] + d->area_len[k]);
    bx->areasInGPU[k] = &d->area_gpu_store[k];
  }
  for (int k = 0; k < kAreas - 1; k++) {
    bx->filterVectors[k] = nullptr;
    bx->filterVectorsInGPU[k] = d->fvs + (size_t)((k + 1) * d->sub - 1) * d->fv_stride;
  }
  bx->rawDataInGPU = const_cast<CODE *>(col);
  bx->dev = d;
}

// Host copies of the sorted arrays and the host pos_block views over them.
hipError_t bindex_host_blocks(BinDex *bx) {
  if (!bx || !bx->dev) return hipErrorInvalidValue;
  rts_bindex_dev *d = bx->dev;
  if (!d->blkp_host.empty()) return hipSuccess;
  d->host_val.resize(d->n);
  d->host_pos.resize(d->n);
  hipError_t e = hipMemcpy(d->host_val.data(), d->sorted_val, d->n * sizeof(CODE), hipMemcpyDeviceToHost);
  if (e == hipSuccess)
    e = hipMemcpy(d->host_pos.data(), d->sorted_pos, d->n * sizeof(int32_t), hipMemcpyDeviceToHost);
  if (e != hipSuccess) {
    std::vector<CODE>().swap(d->host_val);
    std::vector<int32_t>().swap(d->host_pos);
    return e;
  }
  make_block_views(d, d->host_val.data(), d->host_pos.data(), d->blk_host, d->blkp_host);
  int64_t b0 = 0;
  for (int k = 0; k < kAreas; k++) {
    d->area_store[k].blocks = d->blkp_host.data() + b0;
    b0 += d->area_store[k].blockNum;
  }
  return hipSuccess;
}

// Values of the sorted column that are copied to the host with the starts, at most (64 KB).
constexpr int64_t kStagedTail = 1 << 14;

hipError_t bindex_build(BinDex *bx, const CODE *col, int64_t n, CODE *owned, int sub, hipStream_t s) {
  hipError_t err = hipSuccess;
  rts_bindex_dev *d = nullptr;
  uint32_t *counts = nullptr;
  uint16_t *keys = nullptr;
  void *sort_tmp = nullptr, *tmp = nullptr;
  size_t need = 0;
  BuildHead *head_d = nullptr;
  std::vector<BuildHead> head(1);
  CODE *tail_d = nullptr;  // rank samples, then the blocks' first and last values
  const int64_t samples = (n + kRankSample - 1) / kRankSample, max_blocks = n / RTS_BLOCK_INIT_SIZE + kAreas;
  std::vector<CODE> tail;
  // few: copied with the head and moved on the host
  const bool tail_host = samples + 2 * max_blocks <= kStagedTail;
  int64_t nblocks = 0;
  uint32_t nb = 0, *fine = nullptr;
  int bins = 0, parts = 1;
  std::vector<int64_t> rk;

  if (!bx || !col || n < kAreas || n > 0x7FFFFFFFll || (sub != 1 && sub != 2 && sub != 4 && sub != 8))
    return hipErrorInvalidValue;
  memset(bx, 0, sizeof(*bx));
  d = new rts_bindex_dev();
  RTS_TRY(hipGetDevice(&d->device));
  d->n = n;
  d->words = (n + 31) / 32;
  d->fv_stride = (d->words + kFvStrideAlign - 1) / kFvStrideAlign * kFvStrideAlign;
  d->ntiles = (n + kTileRows - 1) / kTileRows;
  d->owned_column = owned;
  d->sub = sub;
  d->bins = bins = kAreas * sub;

  // 1. stable sort of (value, row)
  RTS_TRY(pool_alloc(&d->sorted_val, n * sizeof(CODE)));
  RTS_TRY(pool_alloc(&d->sorted_pos, n * sizeof(int32_t)));
  RTS_TRY(pool_alloc(&sort_tmp, sort_rows_workspace(n)));
  RTS_TRY(sort_rows(col, n, d->sorted_val, (uint32_t *)d->sorted_pos, sort_tmp, s));

  // 2. area and bin starts; the values the host keeps of the sorted column
  RTS_TRY(pool_alloc(&head_d, sizeof(BuildHead)));
  hipLaunchKernelGGL(k_build_starts, dim3(1), dim3(kStartThreads), 0, s, d->sorted_val, n, sub, head_d);
  RTS_TRY(hipGetLastError());
  RTS_TRY(pool_alloc(&tail_d, (samples + 2 * max_blocks) * sizeof(CODE)));
  hipLaunchKernelGGL(k_rank_samples, dim3((unsigned)((samples + kBlock - 1) / kBlock)), dim3(kBlock), 0, s,
                     d->sorted_val, samples, tail_d);
  RTS_TRY(hipGetLastError());
  hipLaunchKernelGGL(k_block_bounds, dim3(kAreas), dim3(kAreas), 0, s, d->sorted_val, n, head_d->idx, tail_d + samples,
                     tail_d + samples + max_blocks);
  RTS_TRY(hipGetLastError());

  // 3. filter vectors + list keys
  RTS_TRY(pool_alloc(&d->fvs, (size_t)(bins - 1) * d->fv_stride * sizeof(BITS)));
  RTS_TRY(pool_alloc(&keys, n * sizeof(uint16_t)));
  {
    const dim3 grid(blocks_for((n + kFvTileRows - 1) / kFvTileRows, kBlock / kWave));
#define RTS_BUILD_FVS(M)                                                                                        \
  hipLaunchKernelGGL(k_build_fvs<M>, grid, dim3(kBlock), 0, s, col, n, head_d->estarts, head_d->light, d->fvs, \
                     d->fv_stride, keys)
    if (bins == 128) RTS_BUILD_FVS(7);
    else if (bins == 256) RTS_BUILD_FVS(8);
    else if (bins == 512) RTS_BUILD_FVS(9);
    else RTS_BUILD_FVS(10);
#undef RTS_BUILD_FVS
  }
  RTS_TRY(hipGetLastError());

  // 4. tile directory and B lists.  A short column's tiles are cut into up to 8 parts, to fill the
  //    device, with a directory of their own (1e6 rows, 256 bins: counts 19 -> 4 us, entries
  //    40 -> 10, where the parts counted the rows of their tile before them themselves)
  while (parts < kTileRows / kPartRows && n > (int64_t)kPartRows * parts && d->ntiles * parts < 4 * (int64_t)device_cu_count())
    parts *= 2;
  {
    const int64_t tiles = d->ntiles * parts, items = (int64_t)bins * (tiles + 1);
    RTS_TRY(pool_alloc(&d->bdir, (int64_t)bins * (d->ntiles + 1) * sizeof(uint32_t)));
    if (parts > 1) RTS_TRY(pool_alloc(&fine, items * sizeof(uint32_t)));
    uint32_t *const dir = parts > 1 ? fine : d->bdir;
    RTS_TRY(pool_alloc(&counts, items * sizeof(uint32_t)));
    RTS_TRY(hipcub::DeviceScan::ExclusiveSum(nullptr, need, counts, dir, items, s));
    RTS_TRY(pool_alloc(&tmp, need));
    hipLaunchKernelGGL(k_list_counts, dim3((unsigned)(tiles + 1)), dim3(kBlock),
                       kBlock / kWave * (bins + 1) * sizeof(uint32_t), s, keys, n, bins, tiles, kTileRows / parts, counts);
    RTS_TRY(hipGetLastError());
    RTS_TRY(hipcub::DeviceScan::ExclusiveSum(tmp, need, counts, dir, items, s));
    if (parts > 1) {
      hipLaunchKernelGGL(k_thin_directory, dim3((unsigned)((bins * (d->ntiles + 1) + kBlock - 1) / kBlock)), dim3(kBlock),
                         0, s, fine, bins, d->ntiles, parts, d->bdir);
      RTS_TRY(hipGetLastError());
    }
    RTS_TRY(pool_alloc(&d->boff, (bins + 1) * sizeof(uint32_t)));
    hipLaunchKernelGGL(k_bin_offsets, dim3((bins + 1 + kBlock - 1) / kBlock), dim3(kBlock), 0, s, d->bdir, d->ntiles,
                       bins, d->boff, head_d->boff);
    RTS_TRY(hipGetLastError());
  }
  RTS_TRY(hipMemcpyAsync(head.data(), head_d, sizeof(BuildHead), hipMemcpyDeviceToHost, s));
  if (tail_host) {
    tail.resize(samples + 2 * max_blocks);
    RTS_TRY(hipMemcpyAsync(tail.data(), tail_d, tail.size() * sizeof(CODE), hipMemcpyDeviceToHost, s));
  }
  RTS_TRY(hipStreamSynchronize(s));
  memcpy(d->starts, head[0].starts, sizeof(d->starts));
  d->estarts.assign(head[0].estarts, head[0].estarts + bins);
  d->boff_host.assign(head[0].boff, head[0].boff + bins + 1);
  bx->data_max = head[0].data_max;
  nb = d->boff_host[bins];
  d->nb = nb;
  rk.assign(head[0].rk, head[0].rk + 2 * bins);
  mark_complete_bins(d, rk);
  RTS_TRY(pool_alloc(&d->bent, std::max<uint32_t>(nb, 1) * sizeof(uint2)));
  if (nb) {
    const int64_t tiles = d->ntiles * parts;
    const dim3 grid((unsigned)tiles);
    const size_t lds = kPartRows * sizeof(uint2) + (kBlock / kWave * (bins + 1) + 2 * bins) * sizeof(uint32_t);
#define RTS_LIST_ENTRIES(NB)                                                                             \
  hipLaunchKernelGGL(k_list_entries<NB>, grid, dim3(kBlock), lds, s, col, keys, n, bins, tiles, kTileRows / parts, \
                     parts > 1 ? fine : d->bdir, d->bent)
    if (bins <= 128) RTS_LIST_ENTRIES(8);
    else if (bins <= 256) RTS_LIST_ENTRIES(9);
    else if (bins <= 512) RTS_LIST_ENTRIES(10);
    else RTS_LIST_ENTRIES(11);
#undef RTS_LIST_ENTRIES
    RTS_TRY(hipGetLastError());
  }

  // 5. host descriptor: areas (bindex.cpp:633-652) and their blocks
  for (int k = 0; k < kAreas; k++) {
    d->area_start[k] = head[0].idx[k];
    d->area_len[k] = (k < kAreas - 1 ? head[0].idx[k + 1] : n) - head[0].idx[k];
    nblocks += area_blocks(d->area_len[k]);
  }
  if (tail_host) {
    const CODE *t = tail.data();
    d->rank_samples.assign(t, t + samples);
    d->block_first.assign(t + samples, t + samples + nblocks);
    d->block_last.assign(t + samples + max_blocks, t + samples + max_blocks + nblocks);
  } else {
    d->rank_samples.resize(samples);
    d->block_first.resize(nblocks);
    d->block_last.resize(nblocks);
    RTS_TRY(hipMemcpyAsync(d->rank_samples.data(), tail_d, samples * sizeof(CODE), hipMemcpyDeviceToHost, s));
    RTS_TRY(hipMemcpyAsync(d->block_first.data(), tail_d + samples, nblocks * sizeof(CODE), hipMemcpyDeviceToHost, s));
    RTS_TRY(hipMemcpyAsync(d->block_last.data(), tail_d + samples + max_blocks, nblocks * sizeof(CODE),
                           hipMemcpyDeviceToHost, s));
  }
  RTS_TRY(hipStreamSynchronize(s));

  describe(bx, d, col);
  d = nullptr;

fail:
  {
    const bool idle = hipStreamSynchronize(s) == hipSuccess;  // before other calls get the workspaces
    for (void *p : {sort_tmp, (void *)counts, (void *)keys, tmp, (void *)fine, (void *)head_d, (void *)tail_d})
      pool_free(p, idle);
  }
  if (d) {
    d->owned_column = nullptr;  // the caller frees what it passed in on failure
    free_dev(d);
  }
  return err;
}

void bindex_free(BinDex *bx) {
  if (!bx) return;
  free_dev(bx->dev);
  memset(bx, 0, sizeof(*bx));
}

}  // namespace rts

// ----------------------------------------------------------------- snapshot (persistence)
//
// File layout (host byte order, little-endian on MI355X hosts):
//   "RTSBDX" 0 2 | u32 version, u32 bins, u32 sub, u32 pad | i64 n, words, fv_stride, ntiles,
//   nb, nblocks | u32 data_max, u32 pad | u64 digests: host arrays, sorted_val, sorted_pos,
//   fvs, bent, the indexed column (0 when the index had none) |
//   starts[128] u32 | area_start[128] i64 | area_len[128] i64 | estarts[bins] u32 |
//   boff[bins + 1] u32 | block_first[nblocks] u32 | block_last[nblocks] u32 |
//   sorted_val[n] u32 | sorted_pos[n] i32 | fvs[(bins - 1) * fv_stride] u32 | bent[nb] (u32, u32)
// Device arrays stream through one page-locked staging buffer.  The tile directory is not
// stored: the load rebuilds it from the B lists.  A load checks the header, the host arrays'
// structure (areas tile the sorted column, block counts, starts non-decreasing, list offsets
// non-decreasing up to nb), every B-list entry as it passes through the staging buffer (row
// < n, rows increasing within a bin: the kernels index LDS by row), and the digest of every
// array; any mismatch refuses the file before the index is used.

namespace rts {

hipError_t bitmap_digest(const BITS *bm, int64_t n, unsigned long long *digest, hipStream_t s);

namespace {

constexpr char kSnapMagic[8] = {'R', 'T', 'S', 'B', 'D', 'X', 0, 2};
constexpr uint32_t kSnapVersion = 2;
constexpr size_t kStage = 64u << 20;

struct SnapHeader {
  char magic[8];
  uint32_t version, bins, sub, pad0;
  int64_t n, words, fv_stride, ntiles, nb, nblocks;
  uint32_t data_max, pad1;
  uint64_t dg_host, dg_val, dg_pos, dg_fvs, dg_bent;
  uint64_t dg_col;  // digest of the indexed column at save time (0: not known)
};

bool put(FILE *f, const void *p, size_t bytes) { return fwrite(p, 1, bytes, f) == bytes; }
bool get(FILE *f, void *p, size_t bytes) { return fread(p, 1, bytes, f) == bytes; }

// FNV-1a over host arrays, 8 bytes at a time (a few KB per index).
struct HostDigest {
  uint64_t h = 0xCBF29CE484222325ull;
  void add(const void *p, size_t bytes) {
    const unsigned char *c = static_cast<const unsigned char *>(p);
    for (size_t i = 0; i < bytes; i++) h = (h ^ c[i]) * 0x100000001B3ull;
  }
};

uint64_t host_digest(const rts_bindex_dev *d) {
  HostDigest g;
  g.add(d->starts, sizeof(d->starts));
  g.add(d->area_start, sizeof(d->area_start));
  g.add(d->area_len, sizeof(d->area_len));
  g.add(d->estarts.data(), d->estarts.size() * sizeof(CODE));
  g.add(d->boff_host.data(), d->boff_host.size() * sizeof(uint32_t));
  g.add(d->block_first.data(), d->block_first.size() * sizeof(CODE));
  g.add(d->block_last.data(), d->block_last.size() * sizeof(CODE));
  return g.h;
}

// Digest of a device array of `words` 32-bit words (the checker's bitmap digest over all
// bits of every word).
hipError_t device_digest(const void *p, int64_t words, uint64_t *out) {
  if (words == 0) {
    *out = 0;
    return hipSuccess;
  }
  unsigned long long dg = 0;
  hipError_t e = bitmap_digest(static_cast<const BITS *>(p), words * 32, &dg, ref_stream());
  *out = dg;
  return e;
}

hipError_t put_device(FILE *f, const void *dev, size_t bytes, void *stage) {
  for (size_t off = 0; off < bytes; off += kStage) {
    const size_t len = std::min(kStage, bytes - off);
    hipError_t e = hipMemcpy(stage, (const char *)dev + off, len, hipMemcpyDeviceToHost);
    if (e != hipSuccess) return e;
    if (!put(f, stage, len)) return hipErrorUnknown;
  }
  return hipSuccess;
}

// check(stage, offset, len) sees every chunk on the host before it is uploaded.
template <class Check>
hipError_t get_device(FILE *f, void *dev, size_t bytes, void *stage, Check check) {
  for (size_t off = 0; off < bytes; off += kStage) {
    const size_t len = std::min(kStage, bytes - off);
    if (!get(f, stage, len)) return hipErrorInvalidValue;
    if (!check(stage, off, len)) return hipErrorInvalidValue;
    hipError_t e = hipMemcpy((char *)dev + off, stage, len, hipMemcpyHostToDevice);
    if (e != hipSuccess) return e;
  }
  return hipSuccess;
}

const auto kNoCheck = [](const void *, size_t, size_t) { return true; };

int blocks_of(int64_t len) {
  return (int)(len <= RTS_BLOCK_INIT_SIZE ? 1 : (len + RTS_BLOCK_INIT_SIZE - 1) / RTS_BLOCK_INIT_SIZE);
}

// Structure of the host arrays read from a snapshot.
bool host_arrays_valid(const rts_bindex_dev *d, int64_t nblocks) {
  int64_t slot = 0, blocks = 0;
  for (int k = 0; k < kAreas; k++) {
    if (d->area_start[k] != slot || d->area_len[k] < 1) return false;
    slot += d->area_len[k];
    blocks += blocks_of(d->area_len[k]);
    if (k && d->starts[k] < d->starts[k - 1]) return false;
  }
  if (slot != d->n || blocks != nblocks) return false;
  for (int b = 0; b < d->bins; b++) {
    if (b && d->estarts[b] < d->estarts[b - 1]) return false;
    if (b % d->sub == 0 && d->estarts[b] != d->starts[b / d->sub]) return false;
  }
  if (d->boff_host[0] != 0 || d->boff_host[d->bins] != (uint32_t)d->nb) return false;
  for (int b = 0; b < d->bins; b++)
    if (d->boff_host[b + 1] < d->boff_host[b]) return false;
  return true;
}

}  // namespace

hipError_t bindex_save(const BinDex *bx, const char *path) {
  if (!bx || !bx->dev || !path) return hipErrorInvalidValue;
  const rts_bindex_dev *d = bx->dev;
  SnapHeader h{};
  memcpy(h.magic, kSnapMagic, 8);
  h.version = kSnapVersion;
  h.bins = (uint32_t)d->bins;
  h.sub = (uint32_t)d->sub;
  h.n = d->n;
  h.words = d->words;
  h.fv_stride = d->fv_stride;
  h.ntiles = d->ntiles;
  h.nb = d->nb;
  h.nblocks = (int64_t)d->block_first.size();
  h.data_max = bx->data_max;
  h.dg_host = host_digest(d);
  const size_t fv_words = (size_t)(d->bins - 1) * d->fv_stride;
  hipError_t e = device_digest(d->sorted_val, d->n, &h.dg_val);
  if (e == hipSuccess) e = device_digest(d->sorted_pos, d->n, &h.dg_pos);
  if (e == hipSuccess) e = device_digest(d->fvs, (int64_t)fv_words, &h.dg_fvs);
  if (e == hipSuccess) e = device_digest(d->bent, 2 * d->nb, &h.dg_bent);
  if (e == hipSuccess && bx->rawDataInGPU) e = device_digest(bx->rawDataInGPU, d->n, &h.dg_col);
  if (e != hipSuccess) return e;
  FILE *f = fopen(path, "wb");
  if (!f) return hipErrorInvalidValue;
  void *stage = nullptr;
  e = hipHostMalloc(&stage, kStage, hipHostMallocDefault);
  bool ok = e == hipSuccess && put(f, &h, sizeof(h)) && put(f, d->starts, sizeof(d->starts)) &&
            put(f, d->area_start, sizeof(d->area_start)) && put(f, d->area_len, sizeof(d->area_len)) &&
            put(f, d->estarts.data(), d->bins * sizeof(CODE)) &&
            put(f, d->boff_host.data(), (d->bins + 1) * sizeof(uint32_t)) &&
            put(f, d->block_first.data(), h.nblocks * sizeof(CODE)) &&
            put(f, d->block_last.data(), h.nblocks * sizeof(CODE));
  if (ok) e = put_device(f, d->sorted_val, d->n * sizeof(CODE), stage);
  if (ok && e == hipSuccess) e = put_device(f, d->sorted_pos, d->n * sizeof(int32_t), stage);
  if (ok && e == hipSuccess) e = put_device(f, d->fvs, fv_words * sizeof(BITS), stage);
  if (ok && e == hipSuccess) e = put_device(f, d->bent, d->nb * sizeof(uint2), stage);
  if (stage) (void)hipHostFree(stage);
  if (fclose(f) != 0) ok = false;
  if (e != hipSuccess) return e;
  return ok ? hipSuccess : hipErrorUnknown;
}

hipError_t bindex_load(BinDex *bx, const char *path, const CODE *col) {
  if (!bx || !path) return hipErrorInvalidValue;
  FILE *f = fopen(path, "rb");
  if (!f) return hipErrorInvalidValue;
  SnapHeader h{};
  rts_bindex_dev *d = nullptr;
  void *stage = nullptr;
  hipError_t e = hipErrorInvalidValue;
  size_t fv_words = 0;
  uint64_t dg = 0;
  int64_t bin = 0;        // bin of the next B-list entry to check
  uint32_t prev_row = 0;  // row of the previous entry of that bin
  auto check_entries = [&](const void *p, size_t off, size_t len) {
    if (off % sizeof(uint2) || len % sizeof(uint2)) return false;
    const uint2 *ent = static_cast<const uint2 *>(p);
    for (size_t i = 0, e0 = off / sizeof(uint2); i < len / sizeof(uint2); i++) {
      const uint64_t e = e0 + i;
      while (bin < d->bins && e >= d->boff_host[bin + 1]) bin++;
      if (bin >= d->bins || ent[i].x >= (uint64_t)d->n) return false;
      if (e > d->boff_host[bin] && ent[i].x <= prev_row) return false;  // row order in a bin
      prev_row = ent[i].x;
    }
    return true;
  };
  if (!get(f, &h, sizeof(h)) || memcmp(h.magic, kSnapMagic, 8) != 0 || h.version != kSnapVersion ||
      (h.sub != 1 && h.sub != 2 && h.sub != 4 && h.sub != 8) || h.bins != (uint32_t)kAreas * h.sub ||
      h.n < kAreas || h.n > 0x7FFFFFFFll || h.words != (h.n + 31) / 32 || h.fv_stride < h.words ||
      h.fv_stride % kFvStrideAlign != 0 || h.fv_stride > h.words + kFvStrideAlign ||
      h.ntiles != (h.n + kTileRows - 1) / kTileRows || h.nb < 0 || h.nb > h.n || h.nblocks < kAreas ||
      h.nblocks > h.n)
    goto done;
  d = new rts_bindex_dev();
  d->n = h.n;
  d->words = h.words;
  d->fv_stride = h.fv_stride;
  d->ntiles = h.ntiles;
  d->nb = h.nb;
  d->sub = (int)h.sub;
  d->bins = (int)h.bins;
  d->estarts.resize(d->bins);
  d->boff_host.resize(d->bins + 1);
  d->block_first.resize(h.nblocks);
  d->block_last.resize(h.nblocks);
  if (!get(f, d->starts, sizeof(d->starts)) || !get(f, d->area_start, sizeof(d->area_start)) ||
      !get(f, d->area_len, sizeof(d->area_len)) || !get(f, d->estarts.data(), d->bins * sizeof(CODE)) ||
      !get(f, d->boff_host.data(), (d->bins + 1) * sizeof(uint32_t)) ||
      !get(f, d->block_first.data(), h.nblocks * sizeof(CODE)) ||
      !get(f, d->block_last.data(), h.nblocks * sizeof(CODE)))
    goto done;
  if (host_digest(d) != h.dg_host || !host_arrays_valid(d, h.nblocks)) goto done;
  fv_words = (size_t)(d->bins - 1) * h.fv_stride;
  e = hipGetDevice(&d->device);
  if (e == hipSuccess) e = hipHostMalloc(&stage, kStage, hipHostMallocDefault);
  if (e == hipSuccess) e = pool_alloc(&d->sorted_val, h.n * sizeof(CODE));
  if (e == hipSuccess) e = pool_alloc(&d->sorted_pos, h.n * sizeof(int32_t));
  if (e == hipSuccess) e = pool_alloc(&d->fvs, fv_words * sizeof(BITS));
  if (e == hipSuccess) e = pool_alloc(&d->bent, std::max<int64_t>(h.nb, 1) * sizeof(uint2));
  if (e == hipSuccess) e = pool_alloc(&d->boff, (d->bins + 1) * sizeof(uint32_t));
  if (e == hipSuccess) e = pool_alloc(&d->bdir, (size_t)d->bins * (h.ntiles + 1) * sizeof(uint32_t));
  if (e == hipSuccess) e = get_device(f, d->sorted_val, h.n * sizeof(CODE), stage, kNoCheck);
  if (e == hipSuccess) e = get_device(f, d->sorted_pos, h.n * sizeof(int32_t), stage, kNoCheck);
  if (e == hipSuccess) e = get_device(f, d->fvs, fv_words * sizeof(BITS), stage, kNoCheck);
  if (e == hipSuccess) e = get_device(f, d->bent, h.nb * sizeof(uint2), stage, check_entries);
  // the arrays as uploaded must carry the digests the saved index had
  if (e == hipSuccess) e = device_digest(d->sorted_val, h.n, &dg);
  if (e == hipSuccess && dg != h.dg_val) e = hipErrorInvalidValue;
  if (e == hipSuccess) e = device_digest(d->sorted_pos, h.n, &dg);
  if (e == hipSuccess && dg != h.dg_pos) e = hipErrorInvalidValue;
  if (e == hipSuccess) e = device_digest(d->fvs, (int64_t)fv_words, &dg);
  if (e == hipSuccess && dg != h.dg_fvs) e = hipErrorInvalidValue;
  if (e == hipSuccess) e = device_digest(d->bent, 2 * h.nb, &dg);
  if (e == hipSuccess && dg != h.dg_bent) e = hipErrorInvalidValue;
  // the column given with the snapshot must be the one that was indexed
  if (e == hipSuccess && col && h.dg_col) {
    e = device_digest(col, h.n, &dg);
    if (e == hipSuccess && dg != h.dg_col) e = hipErrorInvalidValue;
  }
  if (e == hipSuccess)
    e = hipMemcpy(d->boff, d->boff_host.data(), (d->bins + 1) * sizeof(uint32_t), hipMemcpyHostToDevice);
  if (e == hipSuccess) e = launch_tile_directory(d, d->ntiles, kTileRows, d->bdir, ref_stream());
  if (e == hipSuccess) e = hipStreamSynchronize(ref_stream());
  if (e == hipSuccess) e = rank_samples(d, ref_stream());
  if (e == hipSuccess) {
    // which bins' lists hold every row of the bin (a snapshot of an index built without
    // the start rows in its lists has none)
    std::vector<int64_t> rk;
    e = start_ranks(d, rk, ref_stream());
    if (e == hipSuccess) mark_complete_bins(d, rk);
  }
  if (e == hipSuccess) {
    memset(bx, 0, sizeof(*bx));
    bx->data_max = h.data_max;
    describe(bx, d, col);
    d = nullptr;
  }
done:
  if (stage) (void)hipHostFree(stage);
  if (d) free_dev(d);
  fclose(f);
  return e;
}

}  // namespace rts
