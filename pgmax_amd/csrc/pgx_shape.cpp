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

}  // namespace pgx
