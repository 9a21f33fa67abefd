// The attention's split of the queries over workgroups (host code, no HIP).
#pragma once

#include <cstdint>

namespace wf {

constexpr int kQueriesWide = 256;  // queries of a workgroup whose eight waves all compute
constexpr int kTileKeys = 64;

// Queries per workgroup: the split whose rounds of workgroups (one per CU) take least.  A round costs its tiles, plus
// a fixed part (Q in, O out, the first stage) that short contexts feel; both in tile times of the 128-query split,
// about 0.96 us.  Per tile: 256 queries 1.6 (fp8 scores 1.65), 96 queries 0.95, 64 and 32 queries 0.94 and 0.92
// (fewer query waves contend for LDS).  The fixed part, 2.5 with bf16 scores and 0.5 with fp8 ones, is where the rule
// goes wrong least over 1-9360 queries, 12 and 40 heads, 64-10920 keys: its split is within 4 % of the fastest of the
// five and never slower than 256 queries.  Without it short contexts of many heads went into more, smaller rounds
// (us, 256 / 128 queries: dense 3120 x 40 heads over 64 keys 21.4 / 24.7, exact 2400 x 40 over 256 28.7 / 30.2).
// 4680 x 12 heads: 228 workgroups of 256 in one round (23.3 us over 512 keys) against 444 of 128 in two (27.1 us);
// 1560 x 40 over 4680 keys: 280 of 256 in two rounds 264 us, 520 of 128 in three 229, 680 of 96 in three 222.
inline int pick_queries(int64_t lq, int64_t n_heads, int64_t n_kv, bool fp8_scores, int64_t cus) {
  // the finer splits' staging waves index up to four tiles past the last
  if (n_kv >= (1ll << 31) - 8 * kTileKeys) return kQueriesWide;
  const struct {
    int queries;
    double tile;
  } splits[] = {{kQueriesWide, fp8_scores ? 1.65 : 1.6}, {128, 1.0}, {96, 0.95}, {64, 0.94}, {32, 0.92}};
  const double fixed = fp8_scores ? 0.5 : 2.5;
  const double tiles = static_cast<double>((n_kv + kTileKeys - 1) / kTileKeys);
  int best = kQueriesWide;
  double best_cost = 0;
  for (const auto& sp : splits) {
    const int64_t items = (lq + sp.queries - 1) / sp.queries * n_heads;
    const double cost = static_cast<double>((items + cus - 1) / cus) * (fixed + sp.tile * tiles);
    if (sp.queries == kQueriesWide || cost < best_cost) {
      best = sp.queries;
      best_cost = cost;
    }
  }
  return best;
}

}  // namespace wf
