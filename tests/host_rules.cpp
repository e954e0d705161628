// Test doors into the library's host rules (pgx_plan.cpp, pgx_shape.cpp), built
// with the host compiler by test_host_rules.py: no GPU, no HIP.

#include "../pgmax_amd/csrc/pgx_plan.h"
#include "../pgmax_amd/csrc/pgx_shape.h"

using namespace pgx;

namespace {

int plan_of(const pgx_wiring* w, Plan* P, int32_t* kinds) {
  std::string err;
  const int rc = build_plan(*w, P, &err, 4096, true);
  *kinds = 0;
  for (const Block& b : P->blocks) *kinds |= 1 << b.kind;
  return rc;
}

}  // namespace

extern "C" {

// Untuned shape of a convergence run: [tasks, mode, threads].
int rules_converge_shape(const pgx_wiring* w, int32_t batch, int32_t n_it, int32_t t0,
                         int64_t* out) {
  Plan P;
  int32_t kinds;
  const int rc = plan_of(w, &P, &kinds);
  if (rc) return rc;
  const auto shape = converge_shape(P, kinds, batch, n_it, t0 != 0);
  out[0] = int64_t(P.tasks.size());
  out[1] = shape.first;
  out[2] = shape.second;
  return 0;
}

// Mode a convergence run takes that was tuned to per-phase launches.
int rules_tuned_mode(const pgx_wiring* w, int32_t batch, int32_t n_it, int32_t t0,
                     int32_t converge) {
  Plan P;
  int32_t kinds;
  if (plan_of(w, &P, &kinds)) return -1;
  Tuned tuned;
  tuned.best.mode = 2;
  tuned.task_loop.mode = 1;
  return int(tuned_shape(tuned, converge != 0, P, kinds, batch, n_it, t0 != 0).mode);
}

// The autotuner's shapes, 7 numbers each (as pgx_autotune returns them), at
// most `most` of them; flags: TuneInput's in order, bit by bit. Returns their
// number.
int rules_candidates(int32_t flags, int32_t tiles, int64_t* out, int32_t most) {
  TuneInput in;
  bool* const f[] = {&in.converge, &in.bipartite, &in.fusable,    &in.wide,
                     &in.logical,  &in.patches,   &in.square,     &in.lane_tiles,
                     &in.short_lane_tiles,        &in.per_phase_converge};
  for (int k = 0; k < 10; ++k) *f[k] = (flags >> k) & 1;
  in.tiles = tiles;
  const std::vector<RunCfg> c = tune_candidates(in);
  for (int i = 0; i < int(c.size()) && i < most; ++i) {
    const int64_t v[] = {c[i].mode, c[i].bs, c[i].fuse, c[i].vec, c[i].tile, c[i].lanes, c[i].xcd};
    for (int k = 0; k < 7; ++k) out[7 * i + k] = v[k];
  }
  return int(c.size());
}

// Patches of a graph: [patches, depth], or of one that only states its size
// (w null): num_edges / 2 factors, and a task with none of them.
int rules_patches(const pgx_wiring* w, int64_t num_edges, int64_t* out) {
  Plan P;
  int32_t kinds;
  if (w) {
    const int rc = plan_of(w, &P, &kinds);
    if (rc) return rc;
  } else {
    P.num_edges = int32_t(num_edges);
    P.num_factors = int32_t(num_edges / 2);
    P.max_degree = 4;
    P.tasks.push_back(Task{});
  }
  const Patches p = build_patches(P);
  out[0] = p.count;
  out[1] = p.depth;
  return 0;
}

int rules_patch_edges_fit(int64_t num_edges) { return patch_edges_fit(num_edges) ? 1 : 0; }

}  // extern "C"
