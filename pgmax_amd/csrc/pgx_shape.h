// Host rules that choose how a run is executed: plain functions of the plan
// and the call's sizes, so they can be tested without a GPU.
#ifndef PGX_SHAPE_H_
#define PGX_SHAPE_H_

#include <utility>
#include <vector>

#include "pgx_plan.h"

namespace pgx {

// Execution shape of one run: mode 1 task loop / 2 phased / 3 cooperative / 4
// patches, workgroup size of the task loop and of the bipartite tiles,
// factor-side variable sums, vector accesses. mode 0: the untuned rules choose,
// under the options in force.
struct RunCfg {
  int64_t mode = 0, bs = 0, fuse = 1, vec = 3, tile = 256, lanes = 1, xcd = 0;
};

// Untuned shape of a convergence run: {mode, threads per task-loop workgroup}.
// The task loop (1) stops each task's workgroup at its convergence, but an
// iteration takes one CU the whole task: about 0.65 ns per edge or variable
// state of 2x2 graphs at T > 0, 1.3 ns with larger tables, under half of it
// at T = 0 (us_iter: the largest task, or the CUs' share of all tasks). The
// per-phase launches (2) spread every iteration over the chip, but all n_it
// of them are launched, 2.7 us each also after the last task is done. They
// are taken where an iteration of the task loop is long (20 us) and the idle
// launches cost at most about 20 of them. Measured, 300 iterations allowed:
// 100 x 100 torus 46.5 ms (task loop, 256 threads) -> 2.0 ms; 300 Potts grids
// 40 x 40 x 8, done after 26 on average, 10.3 -> 4.6; 10 x 10 torus, done
// after 69, stays in the task loop (0.24 ms against 1.3). Workgroups of the
// task loop: 30 x 30 torus 1,416 us with 256 threads, 634 with 1,024; 16 x 16
// Potts grid of 8 states 328 with 256, 281 with 512, 323 with 1,024; 4,096
// 10 x 10 tori 1.8 ms with 256, 2.8 with 512.
// A graph without factors has no tasks, and its runs launch no iterations.
std::pair<int64_t, int64_t> converge_shape(const Plan& plan, int32_t kinds_mask, int32_t batch,
                                           int32_t n_it, bool t0);

// The autotuner's choice for a batch size and temperature class. Convergence
// runs also keep their fastest task-loop shape.
struct Tuned {
  RunCfg best, task_loop;
};
// The shape a tuned run of at most n_it iterations takes. Probes are short and
// no task finishes in them, so they do not show what per-phase launches that
// outlast every task cost: a convergence run takes them only where
// converge_shape lets an untuned run of n_it iterations take them, and the
// task loop elsewhere.
const RunCfg& tuned_shape(const Tuned& tuned, bool converge, const Plan& plan, int32_t kinds_mask,
                          int32_t batch, int32_t n_it, bool t0);

// What the autotuner's shapes depend on.
struct TuneInput {
  bool converge = false;
  bool bipartite = false;           // complete bipartite binary graph
  bool fusable = false;             // factor side may form the variable sums
  bool wide = false;                // pairwise tables above 8 states that may
  bool logical = false;             // OR or AND factors
  bool patches = false;
  bool square = false;              // square pairwise tables of 3..8 states
  bool lane_tiles = false;          // fused lane-group tiles
  bool short_lane_tiles = false;    // those of one and two passes, at this batch size
  bool per_phase_converge = false;  // converge_shape takes per-phase launches for some n_it
  int32_t tiles = 0;                // per-phase tiles of 64 factors
};
// The shapes the autotuner times, the task loop's last so that their probes can
// stop early against the best of the others. The untuned rules' own choice is
// always among them (RunCfg{} with tile 0): they also take shapes no list names
// for every graph, and a tuned graph must not run slower than an untuned one.
std::vector<RunCfg> tune_candidates(const TuneInput& in);

}  // namespace pgx

#endif  // PGX_SHAPE_H_
