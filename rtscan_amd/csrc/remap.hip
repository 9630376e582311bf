// remap.hip -- value encoding of a column (the reference's remap surface, remap.cpp:110-291).
//
// Both encodings replace each value by a code that keeps the order of distinct values and
// gives every distinct value a code range proportional to its frequency:
//   rank form (remap.cpp:110-203): the row at sorted index i gets encode_min + i * I with
//     I = (int)((encode_max - encode_min) / n) in double; a value's map entry is the code of
//     its first sorted row.
//   dispersed form (remap.cpp:205-241): value v with c rows owns the codes
//     [start(v), start(v) + step(v) - 1) with step(v) = (int)(D * c), D = (max - min) / n in
//     double, start(v) = encode_min + sum of step(u) over u < v; each row draws an offset
//     inside its value's range (the reference uses rand(); here a counter hash of the row
//     index and a seed, so the result does not depend on thread timing).
// All code arithmetic is 32-bit wrap-around, as the reference's int/CODE mix is on x86.
//
// Device pipeline per column: stable radix sort of (value, row) -> runs of equal values per
// tile -> codes and map entries in sorted order -> codes to row order through groups of rows
// (k_runs).
#include <hip/hip_runtime.h>
#include <hipcub/hipcub.hpp>

#include <stdint.h>
#include <string.h>

#include <algorithm>

#include "common.h"
#include "sort_rows.h"
#define RTS_REMAP_NO_CXX
#include "rts_remap.h"

namespace rts {
namespace {

constexpr int kRemapBlock = 256;

unsigned grid_for(int64_t items) { return (unsigned)((items + kRemapBlock - 1) / kRemapBlock); }

__device__ __forceinline__ uint32_t row_hash(uint64_t seed, uint32_t row) {
  uint64_t z = seed + 0x9E3779B97F4A7C15ull * ((uint64_t)row + 1);
  z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
  z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
  return (uint32_t)(z ^ (z >> 31));
}

// Runs of equal values in the sorted column.  No array of run heads or run numbers is kept:
// the heads of each tile of kRunTile sorted rows are counted (k_run_heads), the counts
// scanned, and every later pass finds its rows' run numbers again from its tile's base
// and ballots of the heads, which it needs the sorted values for in any case.
constexpr int kRunThreads = 512;
constexpr int kRunWaves = kRunThreads / kWave;
constexpr int kRunSteps = 4;                             // uint4 of sorted rows per lane
constexpr int kRunTile = kRunThreads * 4 * kRunSteps;  // 8192

// Sorted rows i .. i + 3 of a lane and the bits of those that start a run (bit j: row i + j),
// rows past n none.  The wave's lanes hold consecutive rows.
__device__ __forceinline__ uint32_t run_heads4(const CODE *sval, int64_t i, int64_t n, int lane, uint4 *v) {
  if (i + 4 <= n) {
    *v = *reinterpret_cast<const uint4 *>(sval + i);
  } else {
    v->x = i < n ? sval[i] : 0;
    v->y = i + 1 < n ? sval[i + 1] : 0;
    v->z = i + 2 < n ? sval[i + 2] : 0;
    v->w = 0;
  }
  uint32_t before = __shfl_up(v->w, 1, kWave);
  if (lane == 0) before = i > 0 && i < n ? sval[i - 1] : ~v->x;  // the first row starts a run
  uint32_t h = (v->x != before) | (v->y != v->x) << 1 | (v->z != v->y) << 2 | (v->w != v->z) << 3;
  if (i + 4 > n) h &= i < n ? (1u << (n - i)) - 1 : 0;
  return h;
}

__global__ __launch_bounds__(kRunThreads) void k_run_heads(const CODE *sval, int64_t n, int64_t ntiles, uint32_t *heads) {
  __shared__ uint32_t part[kRunWaves];
  const int lane = threadIdx.x & (kWave - 1), wv = threadIdx.x / kWave;
  const int64_t i0 = (int64_t)blockIdx.x * kRunTile + wv * (kRunTile / kRunWaves) + 4 * lane;
  uint32_t c = 0;
#pragma unroll
  for (int s = 0; s < kRunSteps; s++) {
    uint4 v;
    c += __popc(run_heads4(sval, i0 + s * 4 * kWave, n, lane, &v));
  }
  c = wave_total(c);
  if (lane == 0) part[wv] = c;
  __syncthreads();
  if (threadIdx.x == 0) {
    uint32_t t = 0;
    for (int w = 0; w < kRunWaves; w++) t += part[w];
    heads[blockIdx.x] = t;
    if (blockIdx.x == 0) heads[ntiles] = 0;  // the scan's last value: all runs
  }
}

enum RunPass : int { kRankCodes, kRunFirsts, kDisperse };

struct RunArgs {
  const CODE *sval;
  const uint32_t *spos;
  const uint32_t *base;  // runs that start before each tile
  int64_t n;
  CODE *codes, *map_values, *map_starts;
  // rank form: the row at sorted index i gets encode_min + i * interval
  uint32_t encode_min, interval;
  CODE *sorted_codes;
  // dispersed form: first sorted index and step of each run
  uint32_t *first;
  const uint32_t *step;
  uint64_t seed;
  // rows in groups of group_windows windows (see k_runs)
  uint2 *pairs;
  uint32_t *cursor;
  uint32_t group_windows, group_mul;
};

// Row groups: a window is the rows whose codes fit an LDS tile (k_place_codes), a group
// `group_windows` windows, at most kRowGroups groups.  Window w is in group w / group_windows,
// by a multiplication that is exact for w < 2^13 and up to kGroupWindows windows.
constexpr int kWindowBits = 15, kWindowRows = 1 << kWindowBits;
constexpr int kRowGroups = 512;
constexpr int kGroupWindows = 16;
constexpr int kGroupShift = 18;
__device__ __forceinline__ uint32_t row_group(const RunArgs &a, uint32_t row) {
  return (row >> kWindowBits) * a.group_mul >> kGroupShift;
}
// Shorter columns write codes[row] directly: their codes stay in the caches (2e6 uniform rows
// 252 us against 250 for a whole encode, 4.2e6 335 against 302, one value 272 against 304).
// Longer ones too, where a group's windows would be read too often.
constexpr int64_t kGroupRowsMin = (int64_t)1 << 22;
constexpr int64_t kGroupRowsMax = (int64_t)kRowGroups * kGroupWindows * kWindowRows;

// One pass over the sorted rows with their run numbers.
//   kRankCodes  codes in sorted order, to row order and (optional) to sorted_codes, and the map
//               entries at the heads
//   kRunFirsts  distinct values and first sorted index of every run
//   kDisperse   code(row) = start(v) + (step(v) >= 2 ? hash(row) % (step(v) - 1) : 0)
// To row order: codes[row] = code is a random 4-byte write a row, which costs far more than
// its bytes (2.1 ms at 1e8 skewed rows, 1.5 with the rows grouped so that the codes being
// written stay in an L2).  GROUP therefore writes (row, code) pairs by groups of rows: a
// tile's pairs are laid out by group in LDS and go to memory in runs, each where an atomic
// on the group's cursor says (a row occurs once, so a group's pairs fill the places of its
// rows; their order inside it does not matter).  k_place_codes then gathers each window's
// codes in LDS.
template <int PASS, bool GROUP>
__global__ __launch_bounds__(kRunThreads) void k_runs(RunArgs a) {
  constexpr bool kCodes = PASS != kRunFirsts;
  __shared__ uint32_t part[kRunWaves];
  __shared__ uint2 stage[GROUP ? kRunTile : 1];
  __shared__ uint32_t cnt[GROUP ? kRowGroups : 1], delta[GROUP ? kRowGroups : 1];
  const int lane = threadIdx.x & (kWave - 1), wv = threadIdx.x / kWave;
  const int64_t i0 = (int64_t)blockIdx.x * kRunTile + wv * (kRunTile / kRunWaves) + 4 * lane;
  uint4 v[kRunSteps], p[kRunSteps];
  uint32_t h[kRunSteps], before[kRunSteps];
  const bool vec = ((uintptr_t)a.spos & 15) == 0;  // the caller's sorted_pos may not be
#pragma unroll
  for (int s = 0; s < kRunSteps; s++) {
    const int64_t i = i0 + s * 4 * kWave;
    h[s] = run_heads4(a.sval, i, a.n, lane, &v[s]);
    if (kCodes) {
      if (vec && i + 4 <= a.n) {
        p[s] = *reinterpret_cast<const uint4 *>(a.spos + i);
      } else {
        p[s].x = i < a.n ? a.spos[i] : 0;
        p[s].y = i + 1 < a.n ? a.spos[i + 1] : 0;
        p[s].z = i + 2 < a.n ? a.spos[i + 2] : 0;
        p[s].w = i + 3 < a.n ? a.spos[i + 3] : 0;
      }
    }
  }
  if (GROUP && threadIdx.x < kRowGroups) cnt[threadIdx.x] = 0;
  // heads before each lane's rows in its wave
  uint32_t seen = 0;
#pragma unroll
  for (int s = 0; s < kRunSteps; s++) {
    uint32_t c = seen;
#pragma unroll
    for (int j = 0; j < 4; j++) {
      const uint64_t b = __ballot((h[s] >> j) & 1);
      c = __builtin_amdgcn_mbcnt_hi((uint32_t)(b >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)b, c));
      seen += (uint32_t)__popcll(b);
    }
    before[s] = c;
  }
  if (lane == 0) part[wv] = seen;
  __syncthreads();
  uint32_t base = a.base[blockIdx.x];
  for (int w = 0; w < wv; w++) base += part[w];
  uint32_t code[kRunSteps][4], place[kRunSteps][4];
#pragma unroll
  for (int s = 0; s < kRunSteps; s++) {
    const uint32_t val[4] = {v[s].x, v[s].y, v[s].z, v[s].w}, row[4] = {p[s].x, p[s].y, p[s].z, p[s].w};
    uint32_t run = base + before[s] - 1;  // of the row before
#pragma unroll
    for (int j = 0; j < 4; j++) {
      const int64_t i = i0 + s * 4 * kWave + j;
      const bool head = (h[s] >> j) & 1;
      run += head;
      if (PASS == kRankCodes) {
        const uint32_t c = a.encode_min + (uint32_t)i * a.interval;
        code[s][j] = c;
        if (head) {
          a.map_values[run] = val[j];
          a.map_starts[run] = c;
        }
        if (a.sorted_codes && i < a.n) a.sorted_codes[i] = c;
      } else if (PASS == kRunFirsts) {
        if (head) {
          a.map_values[run] = val[j];
          a.first[run] = (uint32_t)i;
        }
      } else if (i < a.n) {
        const int32_t st = (int32_t)a.step[run];
        code[s][j] = a.map_starts[run] + (st >= 2 ? row_hash(a.seed, row[j]) % (uint32_t)(st - 1) : 0u);
      }
      if (kCodes && i < a.n) {
        if (GROUP) place[s][j] = atomicAdd(&cnt[row_group(a, row[j])], 1u);
        else a.codes[row[j]] = code[s][j];
      }
    }
  }
  if (!GROUP) return;
  __syncthreads();
  // groups in order: their slots of the tile, and their places in memory
  uint32_t c = 0, upto = 0;
  if (threadIdx.x < kRowGroups) {
    c = upto = cnt[threadIdx.x];
#pragma unroll
    for (int o = 1; o < kWave; o <<= 1) {
      const uint32_t u = __shfl_up(upto, o, kWave);
      if (lane >= o) upto += u;
    }
    if (lane == kWave - 1) part[wv] = upto;
  }
  __syncthreads();
  if (threadIdx.x < kRowGroups) {
    uint32_t slot = upto - c;
    for (int w = 0; w < wv; w++) slot += part[w];
    cnt[threadIdx.x] = slot;
    delta[threadIdx.x] = (c ? atomicAdd(&a.cursor[threadIdx.x], c) : 0u) - slot;
  }
  __syncthreads();
#pragma unroll
  for (int s = 0; s < kRunSteps; s++) {
    const uint32_t row[4] = {p[s].x, p[s].y, p[s].z, p[s].w};
#pragma unroll
    for (int j = 0; j < 4; j++)
      if (i0 + s * 4 * kWave + j < a.n) stage[cnt[row_group(a, row[j])] + place[s][j]] = make_uint2(row[j], code[s][j]);
  }
  __syncthreads();
  const uint32_t rows = (uint32_t)min((int64_t)kRunTile, a.n - (int64_t)blockIdx.x * kRunTile);
  for (uint32_t e = threadIdx.x; e < rows; e += kRunThreads) {
    const uint2 x = stage[e];
    a.pairs[delta[row_group(a, x.x)] + e] = x;
  }
}

__global__ void k_group_cursors(uint32_t *cursor, uint32_t group_rows) { cursor[threadIdx.x] = threadIdx.x * group_rows; }

// codes[row] = code of the pairs (0.4 ms at 1e8 rows): a workgroup reads its window's whole group and keeps the
// window's codes in LDS, then writes them in order.  A group's windows run on one XCD one
// after another (workgroup b runs on XCD b % 8), so that the group (1.6 MB at 1e8 rows, six
// windows) comes from memory once and from the L2 otherwise.
constexpr unsigned kPlaceXcds = 8;
constexpr int kPlaceThreads = 1024;
constexpr int kPlaceLoads = 8;  // 16-byte loads in flight per thread (4: 4116 us for the whole encode, 8: 4035, 16: 4023)
__global__ __launch_bounds__(kPlaceThreads) void k_place_codes(const uint2 *pairs, int64_t n, uint32_t group_windows,
                                                               CODE *codes) {
  __shared__ alignas(16) CODE tile[kWindowRows];
  const uint32_t j = blockIdx.x / kPlaceXcds;
  const int64_t g = (int64_t)(j / group_windows) * kPlaceXcds + blockIdx.x % kPlaceXcds;
  const int64_t r0 = (g * group_windows + j % group_windows) * kWindowRows;
  if (r0 >= n) return;
  const uint32_t window = (uint32_t)(r0 >> kWindowBits);
  const int64_t e0 = g * group_windows * kWindowRows, e1 = min(n, e0 + (int64_t)group_windows * kWindowRows);
  const uint4 *src = reinterpret_cast<const uint4 *>(pairs + e0);  // two pairs each
  const int64_t whole = (e1 - e0) / 2;
  const int64_t rounds = whole / (kPlaceLoads * kPlaceThreads) * (kPlaceLoads * kPlaceThreads);
  for (int64_t e = threadIdx.x; e < rounds; e += kPlaceLoads * kPlaceThreads) {
    uint4 v[kPlaceLoads];
#pragma unroll
    for (int k = 0; k < kPlaceLoads; k++) v[k] = src[e + k * kPlaceThreads];
#pragma unroll
    for (int k = 0; k < kPlaceLoads; k++) {
      if (v[k].x >> kWindowBits == window) tile[v[k].x & (kWindowRows - 1)] = v[k].y;
      if (v[k].z >> kWindowBits == window) tile[v[k].z & (kWindowRows - 1)] = v[k].w;
    }
  }
  for (int64_t e = rounds + threadIdx.x; e < whole; e += kPlaceThreads) {
    const uint4 v = src[e];
    if (v.x >> kWindowBits == window) tile[v.x & (kWindowRows - 1)] = v.y;
    if (v.z >> kWindowBits == window) tile[v.z & (kWindowRows - 1)] = v.w;
  }
  if (((e1 - e0) & 1) && threadIdx.x == 0) {
    const uint2 v = pairs[e1 - 1];
    if (v.x >> kWindowBits == window) tile[v.x & (kWindowRows - 1)] = v.y;
  }
  __syncthreads();
  const int rows = (int)min((int64_t)kWindowRows, n - r0);
  if (rows == kWindowRows && ((uintptr_t)codes & 15) == 0) {
    for (int i = threadIdx.x; i < kWindowRows / 4; i += kPlaceThreads)
      reinterpret_cast<uint4 *>(codes + r0)[i] = reinterpret_cast<const uint4 *>(tile)[i];
  } else {
    for (int i = threadIdx.x; i < rows; i += kPlaceThreads) codes[r0 + i] = tile[i];
  }
}

// Pass 2: step(v) = (int)(D * count(v)); kept as the 32-bit pattern of that int.
__global__ void k_run_steps(const uint32_t *first, int64_t m, int64_t n, double per_row,
                            uint32_t *step) {
  const int64_t r = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (r >= m) return;
  const int64_t end = r + 1 < m ? (int64_t)first[r + 1] : n;
  const double w = per_row * (double)(end - (int64_t)first[r]);
  step[r] = (uint32_t)(int64_t)w;  // truncation toward zero, then the low 32 bits
}

// Pass 3: start(v) = encode_min + exclusive prefix sum of the steps (mod 2^32).
__global__ void k_run_starts(const uint32_t *excl, int64_t m, uint32_t encode_min, CODE *map_starts) {
  const int64_t r = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (r < m) map_starts[r] = encode_min + excl[r];
}

#define RTS_TRY(x)                      \
  do {                                  \
    err = (x);                          \
    if (err != hipSuccess) goto fail;   \
  } while (0)

// Shared front half: stable sort and the runs before each tile.  On success sval, spos
// (maybe the caller's buffer) and base are allocated, m holds the number of distinct values
// and no work is queued.
struct Runs {
  CODE *sval = nullptr;
  uint32_t *spos = nullptr;
  uint32_t *base = nullptr;
  bool own_spos = false;
  int64_t m = 0, tiles = 0;
  // idle: no queued work uses them any more
  void release(bool idle) {
    pool_free(sval, idle);
    if (own_spos) pool_free(spos, idle);
    pool_free(base, idle);
  }
};

hipError_t sorted_runs(const CODE *data, int64_t n, POSTYPE *caller_spos, Runs &R, hipStream_t s) {
  hipError_t err = hipSuccess;
  uint32_t *heads = nullptr;
  void *sort_tmp = nullptr, *tmp = nullptr;
  size_t need = 0;
  uint32_t last = 0;

  R.tiles = (n + kRunTile - 1) / kRunTile;
  RTS_TRY(pool_alloc(&R.sval, n * sizeof(CODE)));
  if (caller_spos) {
    R.spos = (uint32_t *)caller_spos;
  } else {
    RTS_TRY(pool_alloc(&R.spos, n * sizeof(uint32_t)));
    R.own_spos = true;
  }
  RTS_TRY(pool_alloc(&heads, (R.tiles + 1) * sizeof(uint32_t)));
  RTS_TRY(pool_alloc(&R.base, (R.tiles + 1) * sizeof(uint32_t)));
  RTS_TRY(pool_alloc(&sort_tmp, sort_rows_workspace(n)));
  RTS_TRY(hipcub::DeviceScan::ExclusiveSum(nullptr, need, heads, R.base, (int)R.tiles + 1, s));
  RTS_TRY(pool_alloc(&tmp, need));
  RTS_TRY(sort_rows(data, n, R.sval, R.spos, sort_tmp, s));
  hipLaunchKernelGGL(k_run_heads, dim3((unsigned)R.tiles), dim3(kRunThreads), 0, s, R.sval, n, R.tiles, heads);
  RTS_TRY(hipGetLastError());
  RTS_TRY(hipcub::DeviceScan::ExclusiveSum(tmp, need, heads, R.base, (int)R.tiles + 1, s));
  RTS_TRY(hipMemcpyAsync(&last, R.base + R.tiles, sizeof(uint32_t), hipMemcpyDeviceToHost, s));
  RTS_TRY(hipStreamSynchronize(s));
  R.m = last;

fail:
  pool_free(sort_tmp, err == hipSuccess);
  pool_free(heads, err == hipSuccess);
  pool_free(tmp, err == hipSuccess);
  return err;
}

// The pass that writes the codes to row order, directly or through groups of rows.
template <int PASS>
hipError_t codes_to_rows(RunArgs &a, int64_t tiles, hipStream_t s) {
  hipError_t err = hipSuccess;
  if (a.n < kGroupRowsMin || a.n > kGroupRowsMax) {
    hipLaunchKernelGGL((k_runs<PASS, false>), dim3((unsigned)tiles), dim3(kRunThreads), 0, s, a);
    err = hipGetLastError();
    return err == hipSuccess ? hipStreamSynchronize(s) : err;
  }
  const int64_t windows = (a.n + kWindowRows - 1) / kWindowRows;
  a.group_windows = (uint32_t)((windows + kRowGroups - 1) / kRowGroups);
  a.group_mul = ((1u << kGroupShift) + a.group_windows - 1) / a.group_windows;
  const int64_t groups = (windows + a.group_windows - 1) / a.group_windows;
  const unsigned grid = (unsigned)((groups + kPlaceXcds - 1) / kPlaceXcds * kPlaceXcds * a.group_windows);
  RTS_TRY(pool_alloc(&a.pairs, a.n * sizeof(uint2)));
  RTS_TRY(pool_alloc(&a.cursor, kRowGroups * sizeof(uint32_t)));
  hipLaunchKernelGGL(k_group_cursors, dim3(1), dim3(kRowGroups), 0, s, a.cursor, a.group_windows * (uint32_t)kWindowRows);
  RTS_TRY(hipGetLastError());
  hipLaunchKernelGGL((k_runs<PASS, true>), dim3((unsigned)tiles), dim3(kRunThreads), 0, s, a);
  RTS_TRY(hipGetLastError());
  hipLaunchKernelGGL(k_place_codes, dim3(grid), dim3(kPlaceThreads), 0, s, a.pairs, a.n, a.group_windows, a.codes);
  RTS_TRY(hipGetLastError());
  RTS_TRY(hipStreamSynchronize(s));
fail:
  pool_free(a.pairs, err == hipSuccess);
  pool_free(a.cursor, err == hipSuccess);
  return err;
}

bool valid_column(const CODE *data, int64_t n, const CODE *codes, const CODE *mv, const CODE *ms) {
  return data && codes && mv && ms && n >= 1 && n <= 0x7FFFFFFFll;
}

}  // namespace

hipError_t encode_rank(const CODE *data, int64_t n, CODE encode_min, CODE encode_max, CODE *codes,
                       POSTYPE *sorted_pos, CODE *sorted_codes, CODE *map_values, CODE *map_starts,
                       int64_t *map_size, hipStream_t s) {
  if (!valid_column(data, n, codes, map_values, map_starts) || !map_size) return hipErrorInvalidValue;
  hipError_t err = hipSuccess;
  Runs R;
  RunArgs a{};
  // remap.cpp:158: int intervalPerObject = (double(max) - double(min)) / double(n)
  const double q = ((double)encode_max - (double)encode_min) / (double)n;
  const uint32_t interval = (uint32_t)(int64_t)q;
  RTS_TRY(sorted_runs(data, n, sorted_pos, R, s));
  a.sval = R.sval;
  a.spos = R.spos;
  a.base = R.base;
  a.n = n;
  a.codes = codes;
  a.map_values = map_values;
  a.map_starts = map_starts;
  a.encode_min = encode_min;
  a.interval = interval;
  a.sorted_codes = sorted_codes;
  RTS_TRY(codes_to_rows<kRankCodes>(a, R.tiles, s));
  *map_size = R.m;
fail:
  R.release(err == hipSuccess);
  return err;
}

hipError_t encode_dispersed(const CODE *data, int64_t n, CODE encode_min, CODE encode_max, uint64_t seed,
                            CODE *codes, CODE *map_values, CODE *map_starts, int64_t *map_size,
                            hipStream_t s) {
  if (!valid_column(data, n, codes, map_values, map_starts) || !map_size) return hipErrorInvalidValue;
  hipError_t err = hipSuccess;
  Runs R;
  RunArgs a{};
  uint32_t *first = nullptr, *step = nullptr, *excl = nullptr;
  void *tmp = nullptr;
  size_t need = 0;
  // remap.cpp:222: double intervalPerObject = (double(max) - double(min)) / double(n)
  const double per_row = ((double)encode_max - (double)encode_min) / (double)n;
  RTS_TRY(sorted_runs(data, n, nullptr, R, s));
  RTS_TRY(pool_alloc(&first, R.m * sizeof(uint32_t)));
  RTS_TRY(pool_alloc(&step, R.m * sizeof(uint32_t)));
  RTS_TRY(pool_alloc(&excl, R.m * sizeof(uint32_t)));
  a.sval = R.sval;
  a.spos = R.spos;
  a.base = R.base;
  a.n = n;
  a.codes = codes;
  a.map_values = map_values;
  a.map_starts = map_starts;
  a.first = first;
  a.step = step;
  a.seed = seed;
  hipLaunchKernelGGL((k_runs<kRunFirsts, false>), dim3((unsigned)R.tiles), dim3(kRunThreads), 0, s, a);
  RTS_TRY(hipGetLastError());
  hipLaunchKernelGGL(k_run_steps, dim3(grid_for(R.m)), dim3(kRemapBlock), 0, s, first, R.m, n, per_row, step);
  RTS_TRY(hipGetLastError());
  RTS_TRY(hipcub::DeviceScan::ExclusiveSum(nullptr, need, step, excl, (int)R.m, s));
  RTS_TRY(pool_alloc(&tmp, need));
  RTS_TRY(hipcub::DeviceScan::ExclusiveSum(tmp, need, step, excl, (int)R.m, s));
  hipLaunchKernelGGL(k_run_starts, dim3(grid_for(R.m)), dim3(kRemapBlock), 0, s, excl, R.m, encode_min,
                     map_starts);
  RTS_TRY(hipGetLastError());
  RTS_TRY(codes_to_rows<kDisperse>(a, R.tiles, s));
  *map_size = R.m;
fail:
  for (void *p : {(void *)first, (void *)step, (void *)excl, tmp}) pool_free(p, err == hipSuccess);
  R.release(err == hipSuccess);
  return err;
}

#undef RTS_TRY

}  // namespace rts

// ------------------------------------------------------------------------------- C ABI

extern "C" hipError_t rts_encode_column(const CODE *data, int64_t n, CODE encode_min, CODE encode_max,
                                        CODE *codes, POSTYPE *sorted_pos, CODE *sorted_codes,
                                        CODE *map_values, CODE *map_starts, int64_t *map_size,
                                        hipStream_t stream) {
  return rts::set_error(rts::encode_rank(data, n, encode_min, encode_max, codes, sorted_pos, sorted_codes,
                                         map_values, map_starts, map_size, stream),
                        "rts_encode_column");
}

extern "C" hipError_t rts_encode_column_dispersed(const CODE *data, int64_t n, CODE encode_min,
                                                  CODE encode_max, uint64_t seed, CODE *codes,
                                                  CODE *map_values, CODE *map_starts, int64_t *map_size,
                                                  hipStream_t stream) {
  return rts::set_error(rts::encode_dispersed(data, n, encode_min, encode_max, seed, codes, map_values,
                                              map_starts, map_size, stream),
                        "rts_encode_column_dispersed");
}

namespace {
int64_t first_not_below(const CODE *v, int64_t m, CODE q, bool strictly_above) {
  int64_t lo = 0, hi = m;
  while (lo < hi) {
    const int64_t mid = lo + (hi - lo) / 2;
    const bool go_right = strictly_above ? v[mid] <= q : v[mid] < q;
    if (go_right) lo = mid + 1; else hi = mid;
  }
  return lo;
}
}  // namespace

extern "C" hipError_t rts_encode_lookup(const CODE *map_values, const CODE *map_starts, int64_t m,
                                        CODE old_query, enum OPERATOR op, CODE sentinel, CODE *code) {
  if ((m > 0 && (!map_values || !map_starts)) || m < 0 || !code) return hipErrorInvalidValue;
  int64_t i;
  switch (op) {
    case LT:  // first value >= q (remap.cpp:244-249)
    case GE:  // remap.cpp:262-267
      i = first_not_below(map_values, m, old_query, false);
      *code = i == m ? sentinel : map_starts[i];
      return hipSuccess;
    case LE:  // first value > q, its start minus one (remap.cpp:250-255)
      i = first_not_below(map_values, m, old_query, true);
      *code = i == m ? sentinel : map_starts[i] - 1u;
      return hipSuccess;
    case GT:  // first value > q (remap.cpp:256-261)
      i = first_not_below(map_values, m, old_query, true);
      *code = i == m ? sentinel : map_starts[i];
      return hipSuccess;
    default:  // eq and bt are rejected (remap.cpp:268-271 exits)
      return hipErrorInvalidValue;
  }
}

extern "C" CODE rts_encode_key_of(const CODE *map_values, const CODE *map_starts, int64_t m, CODE code) {
  // findKeyByValue (remap.cpp:274-283): the key of the last entry whose start is <= code,
  // provided a later entry starts above code; 0 otherwise (also past the last entry).
  CODE last = 0;
  for (int64_t i = 0; i < m; i++) {
    if (map_starts[i] > code) return last;
    last = map_values[i];
  }
  return 0;
}
