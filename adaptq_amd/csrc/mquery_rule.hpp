// mquery_rule.hpp -- when a decode of many queries per head takes the matrix-core
// kernel (mquery.hip), and how that splits its work.  Host code only, of sizes.
#pragma once

#include <algorithm>

namespace aq {

constexpr int kMqWaves = 4;
constexpr int kMqQueries = 16;  // queries per wave
constexpr int kMqTile = 16;     // tokens per wave step

struct MqPlan {
  int splits, chunk, qgroups;
  int qg;       // query groups a block
  int qblocks;  // blocks over the query groups
};

inline MqPlan mq_plan(int n_heads, int nq, int max_n) {
  MqPlan mp;
  mp.qgroups = (nq + kMqQueries - 1) / kMqQueries;
  mp.qg = mp.qgroups >= 3 ? 4 : mp.qgroups;
  mp.qblocks = (mp.qgroups + mp.qg - 1) / mp.qg;
  const int max1 = max_n > 0 ? max_n : 1;
  // two blocks a CU (256 CUs), of at least 128 tokens each.  Measured, 64
  // queries of 8 heads d128 K4/V4 x 32,768 tokens, the whole call: one block a
  // CU 147 us, two 129, three (as many as the registers allow) 130 with half
  // as much finalize work again.
  const int step = kMqTile * (kMqWaves / mp.qg);
  const int blocks = n_heads * mp.qblocks;
  const int splits = std::max(1, std::min(512 / blocks, (max1 + 127) / 128));
  int chunk = (max1 + splits - 1) / splits;
  chunk = ((chunk + step - 1) / step) * step;
  mp.chunk = chunk;
  mp.splits = (max1 + chunk - 1) / chunk;
  return mp;
}

// Whether the matrix-core kernel takes nq queries of n_heads heads over max_n
// tokens, rather than the LUT kernel as nq * n_heads items.  The LUT kernel
// pays for each query, about 4.5 M values of K a microsecond, in one launch
// or two; this one for groups of 16 queries, about 11 M values a microsecond,
// and 10 us more for its rotation and finalize launches.  Measured (whole
// call, LUT and matrix cores): 8 heads d128 K4/V4 x 32,768 tokens, 4 queries
// 41 and 51 us, 8 queries 68 and 51, 12 queries 116 and 52; 16 heads d64 K4/V2
// x 16,384, 8 queries 26 and 31, 12 queries 36 and 32; 2 heads d128 K3/V3 x
// 32,768, 12 queries 39 and 38; 12 heads d128 x 512, 12 queries 9 and 18; 4
// heads d64 x 1,024, 12 queries 7 and 14.
constexpr int kMqMinQueries = 8;

inline bool mq_pays(int n_heads, int nq, int max_n, int padded) {
  if (nq < kMqMinQueries) return false;
  const double per_query = (double)n_heads * (max_n > 0 ? max_n : 1) * padded;
  const int padded_nq = (nq + kMqQueries - 1) / kMqQueries * kMqQueries;
  return nq * per_query / 4.5e6 > 10.0 + padded_nq * per_query / 1.1e7;
}

}  // namespace aq
