// batch_rank.h -- batched queries evaluated from the columns' values, many queries a row at
// once (batch_rank.hip).
#pragma once

#include <vector>

#include "batch.h"

namespace rts {

constexpr int kRankQueries = 256;                 // queries of a group
constexpr int kRankCols = 4;                      // columns of a group
constexpr int kRankBlocks = kRankQueries / 64;    // its queries' masks, 64 a word
constexpr int kRankBounds = 254;                  // of a column: ranges 0 .. 254, and 255 for rows past the end
constexpr int kRankMinQueries = 8;                // a batch of fewer is not evaluated together
constexpr int kRankMaxGroups = 64;                // of a plan

// A group of queries evaluated together, as k_batch_ranked reads it.
struct alignas(16) RankGroup {
  uint32_t nq, ncols;
  uint32_t cols_of[kRankBlocks];  // bit c: one of the block's queries has a predicate on column c
  uint32_t levels[kRankCols];     // of the column's search: 2^levels - 1 nodes
  const CODE *col[kRankCols];
  uint64_t place[kRankQueries];  // the query's own bitmap, or its index in the launch's bitmaps
  uint32_t id[kRankQueries];     // the query's index in the caller's order
  // [1, 2^levels) breadth-first: a row goes right when its value is above the node's (a
  // bound less one; padding 2^32 - 1, which no value is above)
  uint32_t tree[kRankCols][256];
  uint64_t mask[kRankBlocks][kRankCols][256];  // bit q: range r satisfies the block's query q
};

// What a launch does, read from device memory so that a captured launch follows the queries
// that are set later.
struct RankHeader {
  int ngroups;
  int steps;          // of kRankStepRows rows, that a workgroup takes of a group at a time
  int own_outs;       // the queries have their own bitmaps
  int bindex_groups;  // groups of k_batch for the queries that are not evaluated together
  int apart_groups;   // and for all, where a captured launch may need them
  int nq;             // queries that are set
  int pad[2];
};

// A query as the planner sees it: distinct columns (by address), no empty range unless `empty`.
struct RankQuery {
  int id = 0, ncols = 0;
  bool empty = false;
  const CODE *col[kRankCols];
  CODE lo[kRankCols], hi[kRankCols];
  BITS *own = nullptr;
};

// Groups a plan of max_queries queries has room for; 0: it never has any.
int max_rank_groups(int max_queries);

// All queries of `in` in groups, at most max_groups, if that is faster than the columns' forms
// (else false, and none): by those the whole batch takes bindex_us microseconds, and its queries
// that are not in `in` rest_us (0: none), which a second kernel then takes beside the groups.
bool plan_rank_groups(const std::vector<RankQuery> &in, int64_t n, int max_groups, double bindex_us, double rest_us,
                      std::vector<RankGroup> &groups, RankHeader *header);

// counts (zero between launches): the queries' rows are added.  nullptr: not counted.
hipError_t launch_rank_groups(const RankGroup *groups, const RankHeader *header, int64_t n, BITS *out,
                              int64_t out_stride, unsigned long long *counts, hipStream_t s);

}  // namespace rts
