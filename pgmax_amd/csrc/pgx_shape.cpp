// Host rules that choose how a run is executed (pgx_shape.h).

#include "pgx_shape.h"

#include <algorithm>

namespace pgx {

std::pair<int64_t, int64_t> converge_shape(const Plan& P, int32_t kinds_mask, int32_t batch,
                                           int32_t n_it, bool t0) {
  if (P.tasks.empty()) return {1, 256};
  const Task& big = P.tasks[0];  // ordered by descending work
  int64_t total = 0, factors = 0;
  for (const Task& t : P.tasks) total += t.work;
  for (int32_t bi = big.b0; bi < big.b1; ++bi) factors += P.blocks[bi].count;
  const bool bin2 = kinds_mask == kKindsBin2;
  const double ns = (bin2 ? 0.65 : 1.3) * (t0 ? 0.45 : 1.0);
  const double us_iter =
      1e-3 * ns * double(std::max(big.work, total * batch / 256));
  if (us_iter >= 20.0 && 20.0 * us_iter >= 2.7 * n_it) return {2, 0};
  const int64_t wgs = int64_t(P.tasks.size()) * batch;
  if (bin2 && factors >= 512) return {1, wgs <= 512 ? 1024 : 512};
  if ((kinds_mask & ~kKindsPairwise) == 0 && factors >= 256) return {1, 512};
  return {1, 256};
}

const RunCfg& tuned_shape(const Tuned& tuned, bool converge, const Plan& plan, int32_t kinds_mask,
                          int32_t batch, int32_t n_it, bool t0) {
  const bool other = converge && tuned.best.mode != 1 &&
                     converge_shape(plan, kinds_mask, batch, n_it, t0).first != 2;
  return other ? tuned.task_loop : tuned.best;
}

std::vector<RunCfg> tune_candidates(const TuneInput& in) {
  std::vector<RunCfg> c;
  const bool can_fuse = in.fusable || in.bipartite || in.wide;
  for (const int64_t fuse : {1, 0}) {
    if (fuse && !can_fuse) continue;
    if (!in.converge && in.bipartite && fuse) {  // k_bipartite tiles: (columns, threads)
      for (const auto& ct : {std::make_pair(64, 256), std::make_pair(64, 512),
                             std::make_pair(32, 256), std::make_pair(32, 512),
                             std::make_pair(128, 512)})
        c.push_back(RunCfg{2, ct.second, 1, 3, ct.first});
    } else if (!in.converge) {
      for (const int64_t t : {64, 128, 256}) c.push_back(RunCfg{2, 0, fuse, 3, t});
      c.push_back(RunCfg{2, 0, fuse, 0, 256});
      // square pairwise tables: also thread per factor instead of S lanes
      if (!fuse && in.square)
        for (const int64_t t : {128, 256}) c.push_back(RunCfg{2, 0, 0, 3, t, 0});
      // runs of consecutive tiles per XCD (enough tiles for several rounds)
      if (!fuse && in.tiles >= 64 * 8)
        for (const int64_t x : {4, 16})
          for (const int64_t ln : {1, 0}) c.push_back(RunCfg{2, 0, 0, 3, 256, ln, x});
      if (!fuse && in.logical) c.push_back(RunCfg{2, 0, 0, 3, 256, 1, 8});
      // fused lane groups: also one factor per thread, and XCD runs
      if (fuse && in.lane_tiles) {
        if (in.short_lane_tiles)
          for (const int64_t t : {16, 32}) c.push_back(RunCfg{2, 0, 1, 3, t});
        c.push_back(RunCfg{2, 0, 1, 3, 256, 0, 0});
        for (const int64_t x : {4, 16}) c.push_back(RunCfg{2, 0, 1, 3, 256, 1, x});
      }
    } else if (in.per_phase_converge && (in.fusable || !fuse)) {
      // per-phase launches that skip the tasks that are done, where untuned runs
      // of few enough iterations take them (tuned_shape looks at each run's count)
      if (fuse && in.short_lane_tiles)
        for (const int64_t t : {16, 32}) c.push_back(RunCfg{2, 0, 1, 3, t});
      for (const int64_t t : {64, 128, 256}) c.push_back(RunCfg{2, 0, fuse, 3, t});
    }
  }
  if (!in.converge && in.patches) c.push_back(RunCfg{4, 0, 1, 3, 256});
  if (!in.converge && in.fusable)
    for (const int64_t t : {64, 256}) c.push_back(RunCfg{3, 0, 1, 3, t});
  c.push_back(RunCfg{0, 0, 1, 3, 0});
  for (const int64_t fuse : {1, 0})
    for (const int64_t b : {256, 512, 1024})
      if (can_fuse || !fuse) c.push_back(RunCfg{1, b, fuse, 3, 256});
  return c;
}

}  // namespace pgx
