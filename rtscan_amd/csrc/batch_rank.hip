// batch_rank.hip -- a batch's queries evaluated together from the columns' values.
//
// The bounds of up to 256 queries cut a column's values into at most 255 ranges whose rows
// satisfy the same queries' predicates.  A row's range is found by a binary search in LDS,
// the ranges' query masks of all columns are looked up and ANDed, and 32 rows' masks are
// transposed in registers into words of 32 queries' bitmaps, as k_scan_ranked does for the
// ranges of one column.  A query without a predicate on a column has its bit set in all of
// the column's ranges; an empty query has it in none.
//
// k_batch reads two filter-vector words (8 bytes) and two list slices for every word of every
// query-column, 16 KB a query-column and tile through the L2: that is its bound (1024 queries
// on 4 columns of 1e8 rows: 7.2 ms, 11-13 TB/s from L2).  Here a row costs, per 256 queries,
// a search of every column (24 VALU instructions, 6 LDS reads at 254 bounds) and per 32
// queries 17 VALU instructions for four columns (8 lookups and ANDs, 8 the transpose), and
// memory moves the columns and the bitmaps alone.  Launches, k_batch against this, us: 1e8
// rows x 4, 1024 queries 7180 / 5250; 2^26 x 2, 64 queries 374 / 226 (its memory traffic
// alone 210); 2e7 x 3, 333 queries 530 / 327; queries that no index serves, 1e8 x 4, 256:
// 15500 / 1400.  A batch takes the faster of the two by its estimates (plan_us, batch_us).
#include <string.h>

#include <algorithm>
#include <type_traits>

#include "batch_rank.h"
#include "device_ptr.h"
#include "transpose.h"

namespace rts {

// Two workgroups of 256 a compute unit, one searching while the other stores (one of 512, with 2
// KB a store: 1024 queries on 1e8 rows x 4 6280 us against 5270).
constexpr int kRankThreads = 256, kRankWaves = kRankThreads / kWave, kRankPerCu = 2;  // workgroups
constexpr int kRankTileRows = 2048;  // of a wave: lane l makes word l
constexpr int kRankStepRows = kRankWaves * kRankTileRows, kRankStepWords = kRankStepRows / 32;
constexpr int kRankStaged = 8;       // queries whose words pass through LDS at once
constexpr uint32_t kNoRange = 255;   // of rows past the end

// Work items between one of a workgroup and its next: a multiple of the groups, unless that
// leaves more than one of the XCD's `per_xcd` workgroups in sixteen without work.
__host__ __device__ __forceinline__ uint32_t rank_stride(uint32_t ngroups, uint32_t per_xcd) {
  const uint32_t even = per_xcd / ngroups * ngroups;
  return 16 * even >= 15 * per_xcd ? even : per_xcd;
}

// 2 i + (v > t), in two instructions.
static __device__ __forceinline__ uint32_t descend_above(uint32_t i, uint32_t v, uint32_t t) {
  asm("v_cmp_gt_u32 vcc, %1, %2\n\tv_addc_co_u32 %0, vcc, %0, %0, vcc" : "+v"(i) : "v"(v), "v"(t) : "vcc");
  return i;
}

// 62 KB: two workgroups a compute unit.
struct RankLds {
  uint64_t mask[kRankBlocks][kRankCols][256];
  alignas(16) uint32_t xch[kRankWaves][kRankTileRows / 4];
  alignas(16) uint32_t words[2][kRankStaged][kRankStepWords];  // of as many queries
  uint32_t tree[kRankCols][256];
  uint32_t count[kRankQueries];
};

// Rows of the wave's 64 words of each of 32 queries (word 31 - q: query q): lane l gets query
// l / 4's in its low and query l / 4 + 16's in its high 16 bits.  Halving steps: lanes of
// two registers are exchanged and added, so that each step leaves half the registers.
__device__ __forceinline__ uint32_t wave_counts32(const uint32_t (&words)[32], int lane) {
  uint32_t v[16];
#pragma unroll
  for (int q = 0; q < 16; q++) v[q] = (uint32_t)__popc(words[31 - q]) | (uint32_t)__popc(words[15 - q]) << 16;
#pragma unroll
  for (int q = 0; q < 8; q++) {
    const auto r = __builtin_amdgcn_permlane32_swap(v[q], v[q + 8], false, false);
    v[q] = r[0] + r[1];
  }
#pragma unroll
  for (int q = 0; q < 4; q++) {
    const auto r = __builtin_amdgcn_permlane16_swap(v[q], v[q + 4], false, false);
    v[q] = r[0] + r[1];
  }
#pragma unroll
  for (int q = 0; q < 4; q++) v[q] += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v[q], 0x128, 0xF, 0xF, true);  // row_ror:8
#pragma unroll
  for (int q = 0; q < 2; q++) {
    const uint32_t v0 = v[q], v1 = v[q + 2];
    v[q] = lane & 8 ? v1 : v0;
    v[q] += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v[q], 0x141, 0xF, 0xF, true);  // row_half_mirror
  }
  const uint32_t v0 = v[0], v1 = v[1];
  uint32_t x = lane & 4 ? v1 : v0;
  x += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, 0xB1, 0xF, 0xF, true);  // quad_perm [1,0,3,2]
  x += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, 0x4E, 0xF, 0xF, true);  // quad_perm [2,3,0,1]
  return x;
}

// Work item = (chunk of rows, group): chunk c runs on XCD c % 8 (workgroup b runs on XCD
// b % 8), its groups one after another, so that the workgroups of the groups read the chunk
// from the XCD's L2 at about the same time.  While the groups fit, a workgroup stays with
// one group, whose tables it then loads once.
//
// Bound by the vector ALU (busy half the time) and the LDS (40%), which the waves' phases do
// not overlap fully, and, where the bitmaps do not start on cache lines, by their writes.
// - Writes: lines that two stores fill in part are what a long batch waits for.  Stored
//   straight from the transposed registers (256 bytes a wave and query) bitmaps of 12.5 MB,
//   which start 32 bytes past a line, are written at 2.7 TB/s, aligned ones at 5.4; passed
//   through LDS, 1 KB a workgroup and query, at 3.9 (1e8 rows x 4, 1024 queries: 7.2 ms / 5.6),
//   and non-temporal, which leaves the caches to the columns that the other groups read
//   again, at 4.2 (5.49 ms / 5.25; 2e7 rows x 3, 333 queries 358 us / 327).  Two buffers: one
//   barrier for every 8 queries.
// - 256 registers a lane: the next column's 32 rows are loaded during the search of this
//   one's, and the next step's before this one's stores, which later loads would wait for
//   (5.8 -> 5.6 ms); 64 queries' masks come with one address each.  With 128 registers (twice
//   the waves) the lookups leave no registers to overlap in: 10-15% slower.
// - The upper two levels of a search are compares with registers, two instructions a level.
template <bool COUNT>
__global__ __launch_bounds__(kRankThreads) __attribute__((amdgpu_waves_per_eu(kRankPerCu))) void k_batch_ranked(
    const RankGroup *__restrict__ groups, const RankHeader *__restrict__ header, int64_t n, BITS *out,
    int64_t out_stride, unsigned long long *counts) {
  __shared__ RankLds lds;
  const uint32_t ngroups = (uint32_t)header->ngroups;
  if (ngroups == 0) return;
  const uint32_t run = (uint32_t)header->steps;
  const uint64_t place0 = header->own_outs ? 0 : (uint64_t)out, place1 = header->own_outs ? 1 : (uint64_t)out_stride * 4;
  const int lane = threadIdx.x & (kWave - 1), wv = (int)uniform_u32(threadIdx.x / kWave);
  const uint32_t nsteps = (uint32_t)((n + kRankStepRows - 1) / kRankStepRows), runs = (nsteps + run - 1) / run;
  const uint32_t xcd = blockIdx.x % kXcds, stride = rank_stride(ngroups, gridDim.x / kXcds);
  // units of the XCD: (run of steps, group)
  const uint32_t units = runs > xcd ? ((runs - 1 - xcd) / kXcds + 1) * ngroups : 0;
  uint32_t u = blockIdx.x / kXcds, k = 0, gi, at;  // step k of unit u: group gi, step `at` of the rows
  if (u >= stride || u >= units) return;
  auto place_at = [&](uint32_t u, uint32_t &gi, uint32_t &at) {
    const uint32_t ri = uniform_u32(u / ngroups);
    gi = u - ri * ngroups;
    at = (ri * kXcds + xcd) * run;
  };
  place_at(u, gi, at);
  const int64_t words = (n + 31) / 32;
  uint32_t *const xw = lds.xch[wv];
  uint32_t v[32];  // the column that is searched next: of row 256 j + 4 lane + i, in v[4 j + i]
  auto load = [&](uint32_t(&x)[32], uint64_t rows) {
    const RTS_GLOBAL u32x4 *src = (const RTS_GLOBAL u32x4 *)rows + lane;
#pragma unroll
    for (int j = 0; j < 8; j++) {
      const u32x4 y = src[64 * j];
      x[4 * j] = y.x, x[4 * j + 1] = y.y, x[4 * j + 2] = y.z, x[4 * j + 3] = y.w;
    }
  };
  // a step that is not whole is loaded where it is searched; `load` then reads the first rows,
  // if there are as many
  auto first_rows = [&](uint32_t gi, uint32_t at) -> uint64_t {
    const int64_t row0 = (int64_t)at * kRankStepRows + wv * kRankTileRows;
    return (uint64_t)(const CODE *)(cmem(groups) + gi)->col[0] +
           (((int64_t)at + 1) * kRankStepRows <= n ? row0 : wv * kRankTileRows) * sizeof(CODE);
  };
  const bool any_whole = n >= kRankStepRows;
  if (any_whole) load(v, first_rows(gi, at));
  uint32_t cur = ~0u;
  auto flush = [&]() {
    __syncthreads();
    if (!COUNT || cur == ~0u) return;
    const RankGroup *g = groups + cur;
    if (threadIdx.x < g->nq && lds.count[threadIdx.x])
      atomicAdd(&counts[g->id[threadIdx.x]], (unsigned long long)lds.count[threadIdx.x]);
  };
  while (true) {
    const RTS_CONST RankGroup *g = cmem(groups) + gi;
    const int ncols = (int)g->ncols, nq = (int)g->nq;
    if (gi != cur) {
      flush();
      const int nblocks = (nq + 63) / 64;
      for (int c = 0; c < ncols; c++) {
        lds.tree[c][threadIdx.x] = groups[gi].tree[c][threadIdx.x];
        for (int b = 0; b < nblocks; b++) lds.mask[b][c][threadIdx.x] = groups[gi].mask[b][c][threadIdx.x];
      }
      if (COUNT) lds.count[threadIdx.x] = 0;
      __syncthreads();
      cur = gi;
    }
    uint32_t nu = u, nk = k + 1, ngi = gi, nat = at + 1;  // the next position
    if (nk == run || nat >= nsteps) {
      nu += stride;
      nk = 0;
      if (nu < units) place_at(nu, ngi, nat);
    }
    const bool more = nu < units;
    if (!more) nat = 0;
    const int64_t row0 = (int64_t)at * kRankStepRows + wv * kRankTileRows;
    auto tile = [&](auto whole_tile) __attribute__((always_inline)) {
      constexpr bool kWhole = decltype(whole_tile)::value;
      uint32_t rank4[kRankCols][8];  // the lane's 32 ranges of each column, four a word
#pragma unroll
      for (int c = 0; c < kRankCols; c++) {
        if (c < ncols) {
          // the next column's loads, or the next step's, go out before this column's search:
          // loads wait for the stores issued before them
          uint32_t vn[32];
          const uint64_t next = c + 1 < kRankCols && c + 1 < ncols
                                    ? (uint64_t)(const CODE *)g->col[c + 1 < kRankCols ? c + 1 : 0] + row0 * sizeof(CODE)
                                    : first_rows(ngi, nat);
          if (kWhole) {
            load(vn, next);
          } else {
            const RTS_GLOBAL CODE *col = gmem((const CODE *)g->col[c]);
#pragma unroll
            for (int j = 0; j < 32; j++) {
              v[j] = col[min(row0 + 256 * (j / 4) + 4 * lane + j % 4, n - 1)];
              asm volatile("" : "+v"(v[j]));
            }
          }
          const uint32_t *tree = lds.tree[c];
          const uint32_t root = uniform_u32(tree[1]), node2 = tree[2], node3 = tree[3];
          const int levels = (int)g->levels[c];
          uint32_t i[32];
#pragma unroll
          for (int j = 0; j < 32; j++) {
            const bool up = v[j] > root;
            i[j] = descend_above(up ? 3 : 2, v[j], up ? node3 : node2);
          }
          for (int l = 2; l < levels; l++) {
#pragma unroll
            for (int j = 0; j < 32; j++) i[j] = descend_above(i[j], v[j], tree[i[j]]);
          }
          // range = leaf less 2^levels: no byte of four borrows, and at 8 levels the low byte is it
          const uint32_t leaf0 = levels < 8 ? 0x01010101u << levels : 0u;
#pragma unroll
          for (int j = 0; j < 8; j++) {
            uint32_t r = (__builtin_amdgcn_perm(i[4 * j + 1], i[4 * j], 0x0C0C0400) |
                          __builtin_amdgcn_perm(i[4 * j + 3], i[4 * j + 2], 0x04000C0C)) - leaf0;
            if (!kWhole) {
              const int64_t left = n - row0 - (256 * j + 4 * lane);
              r |= left >= 4 ? 0u : left <= 0 ? ~0u : ~0u << (8 * left);
            }
            xw[64 * j + lane] = r;
          }
          __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");  // the wave's own exchange: LDS keeps its order
          __builtin_amdgcn_wave_barrier();
          const uint4 ra = *reinterpret_cast<const uint4 *>(xw + 8 * lane), rb = *reinterpret_cast<const uint4 *>(xw + 8 * lane + 4);
          __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
          __builtin_amdgcn_wave_barrier();
          rank4[c][0] = ra.x, rank4[c][1] = ra.y, rank4[c][2] = ra.z, rank4[c][3] = ra.w;
          rank4[c][4] = rb.x, rank4[c][5] = rb.y, rank4[c][6] = rb.z, rank4[c][7] = rb.w;
          if (kWhole)
#pragma unroll
            for (int j = 0; j < 32; j++) v[j] = vn[j];
        }
      }
      if (!kWhole && any_whole) load(v, first_rows(ngi, nat));
      const int64_t w0 = (int64_t)at * kRankStepWords + 4 * lane;  // of the lane's four words of a query
#pragma unroll 1
      for (int q0 = 0; q0 < nq; q0 += 64) {
        const uint32_t cols = g->cols_of[q0 / 64];
        uint32_t w[2][32];
#pragma unroll
        for (int r = 0; r < 32; r++) w[0][r] = w[1][r] = ~0u;
        // without this the ranges' 128 addresses would be kept in registers
#pragma unroll
        for (int c = 0; c < kRankCols; c++)
#pragma unroll
          for (int r = 0; r < 8; r++) asm volatile("" : "+v"(rank4[c][r]));
        // two columns at a time: three ANDed by one instruction
#pragma unroll
        for (int c = 0; c < kRankCols; c += 2) {
          const uint32_t use = cols >> c & 3;
          const uint64_t *m0 = lds.mask[q0 / 64][c], *m1 = lds.mask[q0 / 64][c + 1];
          if (use == 3) {
#pragma unroll
            for (int r = 0; r < 32; r++) {
              const uint64_t x = m0[rank4[c][r / 4] >> (8 * (r & 3)) & 0xFF], y = m1[rank4[c + 1][r / 4] >> (8 * (r & 3)) & 0xFF];
              w[0][r] = __builtin_amdgcn_bitop3_b32(w[0][r], (uint32_t)x, (uint32_t)y, 0x80);
              w[1][r] = __builtin_amdgcn_bitop3_b32(w[1][r], (uint32_t)(x >> 32), (uint32_t)(y >> 32), 0x80);
              if (r % 16 == 15) __builtin_amdgcn_sched_barrier(0);
            }
          } else if (use == 1) {
#pragma unroll
            for (int r = 0; r < 32; r++) {
              const uint64_t x = m0[rank4[c][r / 4] >> (8 * (r & 3)) & 0xFF];
              w[0][r] &= (uint32_t)x;
              w[1][r] &= (uint32_t)(x >> 32);
              if (r % 16 == 15) __builtin_amdgcn_sched_barrier(0);
            }
          } else if (use == 2) {
#pragma unroll
            for (int r = 0; r < 32; r++) {
              const uint64_t x = m1[rank4[c + 1][r / 4] >> (8 * (r & 3)) & 0xFF];
              w[0][r] &= (uint32_t)x;
              w[1][r] &= (uint32_t)(x >> 32);
              if (r % 16 == 15) __builtin_amdgcn_sched_barrier(0);
            }
          }
        }
#pragma unroll
        for (int h = 0; h < 2; h++) {
          const int q1 = q0 + 32 * h;
          if (q1 >= nq) break;
          transpose32(w[h]);
          if (COUNT) {
            const uint32_t x = wave_counts32(w[h], lane);
            if ((lane & 2) == 0) atomicAdd(&lds.count[q1 + lane / 4 + 16 * (lane & 1)], lane & 1 ? x >> 16 : x & 0xFFFF);
          }
          // the step's words of a query, 1 KB, by one wave: the fewest partial cache lines of
          // bitmaps that do not start on one
          const RTS_CONST uint64_t *place = g->place + q1 + wv;
#pragma unroll
          for (int p = 0; p < 32; p += kRankStaged) {
#pragma unroll
            for (int q = 0; q < kRankStaged; q++) lds.words[p / kRankStaged % 2][q][64 * wv + lane] = w[h][31 - p - q];
            __syncthreads();
#pragma unroll
            for (int q = 0; q < kRankStaged; q += kRankWaves) {
              if (q1 + p + q + wv < nq) {
                const u32x4 x = *reinterpret_cast<const u32x4 *>(&lds.words[p / kRankStaged % 2][q + wv][4 * lane]);
                RTS_GLOBAL BITS *o = (RTS_GLOBAL BITS *)(place0 + place[p + q] * place1) + w0;
                if (kWhole || w0 + 4 <= words) {
                  __builtin_nontemporal_store(x, (RTS_GLOBAL u32x4 *)o);
                } else {
#pragma unroll
                  for (int j = 0; j < 3; j++)
                    if (w0 + j < words) o[j] = x[j];
                }
              }
            }
          }
        }
      }
    };
    if (((int64_t)at + 1) * kRankStepRows <= n)
      tile(std::true_type{});
    else
      tile(std::false_type{});
    if (!more) break;
    u = nu, k = nk, gi = uniform_u32(ngi), at = uniform_u32(nat);
  }
  flush();
}

// ------------------------------------------------------------------------------ planner

// The models are off by a few per cent.  Where other queries of the batch keep to their columns'
// forms (rest_us), their kernel is one more, and it costs more for each query the fewer there are.
// Of 99 such batches (2e4 to 6.7e7 rows, 2 and 4 columns, 16 to 1024 queries, 1, 4 and 7 of 8 kept
// apart) those taken here save 3 to 23 per cent; with the whole of bindex_us charged to the
// queries in question, 1e5 rows x 4 with 8 of 16 took 49 us for 29, 4.2e6 x 4 with 128 of 256 186 for
// 139, 2e7 x 4 with 32 of 64 249 for 192.
constexpr double kBesideUs = 8;
static bool rank_cheaper(double rank_us, double rest_us, double bindex_us) {
  return rest_us > 0 ? rank_us + rest_us + kBesideUs < bindex_us : rank_us < 0.9 * bindex_us;
}

namespace {

unsigned rank_grid() {
  return std::max<unsigned>(kXcds, (unsigned)kRankPerCu * (unsigned)std::max(1, device_cu_count()) / kXcds * kXcds);
}

struct Column {
  const CODE *ptr;
  std::vector<uint32_t> bound;  // of the batch, less one; distinct and sorted
};

// A query's predicates as numbers of columns and of their bounds (-1: none on that side).
struct Predicates {
  int ncols = 0;
  int col[kRankCols], lo[kRankCols], hi[kRankCols];
};

// A group in the making: its queries, and of its columns the bounds that they use.
struct GroupPlan {
  std::vector<int> query;
  int ncols = 0;
  int col[kRankCols];
  int nbounds[kRankCols] = {};
  std::vector<uint64_t> uses[kRankCols];  // a bit for each of the column's bounds

  bool has(int c, int b) const { return b < 0 || (uses[c][b / 64] >> (b % 64) & 1); }
  // 2^levels - 1 nodes hold the bounds; the kernel takes the upper two levels for granted
  int levels(int c) const {
    int l = 2;
    while ((1 << l) <= nbounds[c]) l++;
    return l;
  }
  // Adds query number i if the group can take it.
  bool add(const Predicates &q, int i, const std::vector<Column> &columns) {
    if (query.size() == (size_t)kRankQueries) return false;
    int at[kRankCols], cols = ncols;
    for (int k = 0; k < q.ncols; k++) {
      int c = 0;
      while (c < cols && col[c] != q.col[k]) c++;
      if (c == kRankCols) return false;
      if (c == cols) {
        col[cols++] = q.col[k];
        nbounds[c] = 0;
        uses[c].assign((columns[q.col[k]].bound.size() + 63) / 64, 0);
      }
      if (nbounds[c] + !has(c, q.lo[k]) + !has(c, q.hi[k]) > kRankBounds) return false;
      at[k] = c;
    }
    for (int k = 0; k < q.ncols; k++)
      for (const int b : {q.lo[k], q.hi[k]})
        if (!has(at[k], b)) {
          uses[at[k]][b / 64] |= 1ull << (b % 64);
          nbounds[at[k]]++;
        }
    ncols = cols;
    query.push_back(i);
    return true;
  }
  // Columns that queries [i, i + 64) have predicates on, a bit each.
  uint32_t cols_of(size_t i, const std::vector<Predicates> &q) const {
    uint32_t used = 0;
    for (size_t j = i; j < std::min(i + 64, query.size()); j++)
      for (int k = 0; k < q[query[j]].ncols; k++)
        for (int c = 0; c < ncols; c++) used |= (uint32_t)(col[c] == q[query[j]].col[k]) << c;
    return used;
  }
  // Microseconds for 1e8 rows by all workgroups: the bitmaps' writes and, beside them, the
  // columns' reads (`memory`: they don't fit the caches) or half of the instructions.
  double us(const std::vector<Predicates> &q, bool memory) const {
    double compute = 0;
    for (int c = 0; c < ncols; c++) compute += 14 * levels(c);
    for (size_t i = 0; i < query.size(); i += 64)
      compute += (52 + 7 * __builtin_popcount(cols_of(i, q))) * (i + 32 < query.size() ? 2 : 1);
    return 2.9 * query.size() + std::max(memory ? 82.0 * ncols : 0.0, compute / 2);
  }
};

void fill_group(RankGroup &g, const GroupPlan &gp, const std::vector<RankQuery> &in, const std::vector<Predicates> &q,
                const std::vector<Column> &columns) {
  memset(&g, 0, sizeof(g));
  const int nq = (int)gp.query.size();
  g.nq = (uint32_t)nq;
  g.ncols = (uint32_t)gp.ncols;
  std::vector<uint8_t> range[kRankCols];  // that begins at a bound of the column
  for (int c = 0; c < gp.ncols; c++) {
    const std::vector<uint32_t> &all = columns[gp.col[c]].bound;
    std::vector<uint32_t> b;
    range[c].resize(all.size());
    for (size_t w = 0; w < gp.uses[c].size(); w++)
      for (uint64_t m = gp.uses[c][w]; m; m &= m - 1) {
        const size_t i = 64 * w + __builtin_ctzll(m);
        b.push_back(all[i]);
        range[c][i] = (uint8_t)b.size();
      }
    g.col[c] = columns[gp.col[c]].ptr;
    g.levels[c] = (uint32_t)gp.levels(c);
    for (uint32_t &v : g.tree[c]) v = 0xFFFFFFFFu;
    for (uint32_t l = 0; l < g.levels[c]; l++)  // node i of level l: the bound in the middle of its span
      for (uint32_t i = 0; i < 1u << l; i++) {
        const size_t at = ((2 * (size_t)i + 1) << (g.levels[c] - 1 - l)) - 1;
        if (at < b.size()) g.tree[c][(1u << l) + i] = b[at];
      }
  }
  for (int i = 0; i < nq; i++) {
    const RankQuery &Q = in[gp.query[i]];
    const Predicates &P = q[gp.query[i]];
    const uint64_t bit = 1ull << (i % 64);
    g.id[i] = (uint32_t)Q.id;
    g.place[i] = Q.own ? (uint64_t)Q.own : (uint64_t)Q.id;
    if (Q.empty) continue;
    for (int c = 0; c < gp.ncols; c++) {
      uint64_t *const m = g.mask[i / 64][c];  // the ranges where the query's bit changes, for now
      int k = 0;
      while (k < P.ncols && P.col[k] != gp.col[c]) k++;
      m[k < P.ncols && P.lo[k] >= 0 ? range[c][P.lo[k]] : 0] ^= bit;
      if (k < P.ncols && P.hi[k] >= 0) m[range[c][P.hi[k]]] ^= bit;
    }
  }
  for (int b = 0; 64 * b < nq; b++) {
    g.cols_of[b] = gp.cols_of(64 * b, q);
    for (int c = 0; c < gp.ncols; c++) {
      for (uint32_t r = 1; r < kNoRange; r++) g.mask[b][c][r] ^= g.mask[b][c][r - 1];
      g.mask[b][c][kNoRange] = 0;
    }
  }
}

using Plan = std::vector<GroupPlan>;

// The queries in order, a group filled as far as it goes before the next: few columns a group
// where queries of the same columns follow each other.
Plan groups_in_order(const std::vector<Predicates> &q, const std::vector<int> &order, const std::vector<Column> &columns) {
  Plan p(1);
  for (const int i : order)
    if (!p.back().add(q[i], i, columns)) {
      p.emplace_back();
      p.back().add(q[i], i, columns);
    }
  return p;
}

// The queries dealt out in turn to the fewest groups that take them, at most `most`: like
// numbers of queries, columns and bounds in each.
Plan groups_dealt(const std::vector<Predicates> &q, const std::vector<int> &order, const std::vector<Column> &columns,
                  size_t most) {
  size_t n = (q.size() + kRankQueries - 1) / kRankQueries;
  for (const Column &c : columns) n = std::max(n, (c.bound.size() + kRankBounds - 1) / kRankBounds);
  for (; n <= most; n++) {
    Plan p(n);
    size_t i = 0;
    while (i < order.size() && p[i % n].add(q[order[i]], order[i], columns)) i++;
    if (i == order.size()) return p;
  }
  return {};
}

// Time of a plan in microseconds.  A workgroup that stays with its group waits for those of the
// longest.  Measured (1e8 rows, 4 columns / 2 columns, mixed queries, us): 32 queries 440 / 271,
// 64 550 / 377, 128 764 / 608, 256 1420 / 1230, 1024 5250 / -; 2e7 rows, 4 columns: 32 121, 64
// 147, 128 191; 1e6 rows, 4 columns: 16 25, 64 31.
double plan_us(const Plan &p, const std::vector<Predicates> &q, int64_t n) {
  const uint32_t steps = (uint32_t)((n + kRankStepRows - 1) / kRankStepRows), grid = rank_grid();
  const uint32_t stride = rank_stride((uint32_t)p.size(), grid / kXcds);
  const uint32_t rounds = ((steps + kXcds - 1) / kXcds * (uint32_t)p.size() + stride - 1) / stride;
  const double round = (double)grid * kRankStepRows / 1e8;
  double worst = 0;
  for (const GroupPlan &g : p) worst = std::max(worst, g.us(q, rounds > 1));
  // less than a round: the workgroups have more of the compute units each
  return (rounds > 1 ? 25 : 15) + worst * round * (2 * steps * p.size() <= grid ? 0.7 : rounds);
}

// plan_us is no less than this, which takes no planning: the bitmaps are written and, in more
// than a round, the columns read.
double least_us(const std::vector<RankQuery> &in, int64_t n) {
  if (n <= (int64_t)rank_grid() * kRankStepRows) return 0.7 * 2.9 * in.size() * n / 1e8;
  const CODE *seen[kRankCols];
  int ncols = 0;
  for (const RankQuery &q : in)
    for (int c = 0; c < q.ncols && ncols < kRankCols; c++)
      if (std::find(seen, seen + ncols, q.col[c]) == seen + ncols) seen[ncols++] = q.col[c];
  return 25 + (2.9 * in.size() + 82.0 * ncols) * n / 1e8;
}

}  // namespace

int max_rank_groups(int max_queries) { return std::min(max_queries / kRankMinQueries, kRankMaxGroups); }

bool plan_rank_groups(const std::vector<RankQuery> &in, int64_t n, int max_groups, double bindex_us, double rest_us,
                      std::vector<RankGroup> &groups, RankHeader *header) {
  groups.clear();
  header->ngroups = 0;
  header->steps = 1;
  if (in.size() < (size_t)kRankMinQueries || in.size() > (size_t)max_groups * kRankQueries) return false;
  if (!rank_cheaper(least_us(in, n), rest_us, bindex_us)) return false;
  std::vector<Column> columns;
  std::vector<std::vector<std::pair<uint32_t, int *>>> bounds;  // (bound less one, where its number goes)
  std::vector<Predicates> q(in.size());
  std::vector<std::pair<uint64_t, int>> key(in.size());
  for (size_t i = 0; i < in.size(); i++) {
    q[i].ncols = in[i].empty ? 1 : in[i].ncols;  // an empty query: zeros by some column's masks
    for (int k = 0; k < q[i].ncols; k++) {
      int c = 0;
      while (c < (int)columns.size() && columns[c].ptr != in[i].col[k]) c++;
      if (c == (int)columns.size()) {
        columns.push_back({in[i].col[k], {}});
        bounds.emplace_back();
      }
      q[i].col[k] = c;
      q[i].lo[k] = q[i].hi[k] = -1;
      if (!in[i].empty) {
        if (in[i].lo[k]) bounds[c].emplace_back(in[i].lo[k] - 1, &q[i].lo[k]);
        if (in[i].hi[k] != 0xFFFFFFFFu) bounds[c].emplace_back(in[i].hi[k], &q[i].hi[k]);
      }
      key[i].first |= 1ull << std::min(c, 63);
    }
    key[i].second = (int)i;
  }
  for (size_t c = 0; c < columns.size(); c++) {
    std::sort(bounds[c].begin(), bounds[c].end(), [](const auto &a, const auto &b) { return a.first < b.first; });
    for (const auto &b : bounds[c]) {
      if (columns[c].bound.empty() || columns[c].bound.back() != b.first) columns[c].bound.push_back(b.first);
      *b.second = (int)columns[c].bound.size() - 1;
    }
  }
  // queries with the same columns next to each other: a block of 64 then looks up fewer columns
  std::sort(key.begin(), key.end());
  std::vector<int> order(in.size());
  for (size_t i = 0; i < in.size(); i++) order[i] = key[i].second;
  Plan plan = groups_in_order(q, order, columns);
  double us = plan_us(plan, q, n);
  if (plan.size() > 1) {
    Plan dealt = groups_dealt(q, order, columns, plan.size());
    const double dealt_us = dealt.empty() ? us : plan_us(dealt, q, n);
    if (dealt_us < us) {
      plan.swap(dealt);
      us = dealt_us;
    }
  }
  if ((int)plan.size() > max_groups || !rank_cheaper(us, rest_us, bindex_us)) return false;
  groups.resize(plan.size());
  for (size_t g = 0; g < plan.size(); g++) fill_group(groups[g], plan[g], in, q, columns);
  header->ngroups = (int)groups.size();
  // a workgroup that changes its group with every item loads the group's tables for it
  header->steps = rank_stride((uint32_t)groups.size(), rank_grid() / kXcds) % groups.size() ? 4 : 1;
  return true;
}

hipError_t launch_rank_groups(const RankGroup *groups, const RankHeader *header, int64_t n, BITS *out,
                              int64_t out_stride, unsigned long long *counts, hipStream_t s) {
  const dim3 grid(rank_grid());
  if (counts)
    hipLaunchKernelGGL(k_batch_ranked<true>, grid, dim3(kRankThreads), 0, s, groups, header, n, out, out_stride, counts);
  else
    hipLaunchKernelGGL(k_batch_ranked<false>, grid, dim3(kRankThreads), 0, s, groups, header, n, out, out_stride, counts);
  return hipGetLastError();
}

}  // namespace rts
