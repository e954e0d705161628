"""GPU parity of specialised kernels at the sizes where they can go wrong
(edges of lane groups, tiles and dispatch rules), against the FP32 oracle,
which states the same operations in the same order: equal bits."""

import numpy as np
import pytest

from oracle import lbp
from pgmax_amd import _lib
from pgmax_amd import fgraph
from pgmax_amd import fgroup
from pgmax_amd import infer
from pgmax_amd import vgroup

pytestmark = pytest.mark.gpu


def _np(x):
  return x.detach().cpu().numpy()


def _bipartite_tables(n0, s0, n1, s1):
  """n0 variables of s0 states, each joined to each of n1 variables of s1."""
  a = vgroup.NDVarArray(num_states=s0, shape=(n0,))
  b = vgroup.NDVarArray(num_states=s1, shape=(n1,))
  fg = fgraph.FactorGraph(variable_groups=[a, b])
  fg.add_factors(fgroup.PairwiseFactorGroup(
      variables_for_factors=[[a[i], b[j]] for i in range(n0) for j in range(n1)],
      log_potential_matrix=np.zeros((n0 * n1, s0, s1))))
  return fg


@pytest.mark.parametrize("temperature", [0.0, 0.4, 1.0])
@pytest.mark.parametrize("n0,s0,n1,s1", [
    (5, 9, 7, 9),      # three factors per wavefront, lanes left over
    (6, 16, 5, 16),    # two factors per wavefront
    (3, 32, 4, 32),    # the whole wavefront, 1,024 configs
    (4, 31, 3, 33),    # odd sizes
    (3, 63, 2, 1),     # one column
    (2, 1, 9, 12),     # one row
    (3, 10, 4, 2),     # a wide and a binary variable
    (3, 40, 3, 40),    # 80 edge states: the general kernel
    (1, 11, 70, 3),    # a wide variable of 70 edges (summed in chunks)
])
def test_pairwise_tables_above_8_states(gpu, n0, s0, n1, s1, temperature):
  fg = _bipartite_tables(n0, s0, n1, s1)
  bp = infer.BP(fg.bp_state, temperature=temperature)
  arrays = bp.init()
  rng = np.random.default_rng(s0 * 100 + s1)
  lp = rng.normal(size=arrays.log_potentials.shape[0]).astype(np.float32)
  lp[:3] = [1e7, -1e7, -np.inf]
  ev = rng.normal(size=arrays.evidence.shape[0]).astype(np.float32)
  ft = rng.normal(size=arrays.ftov_msgs.shape[0]).astype(np.float32)
  g = lbp.graph_from_context(bp.context)
  _lib.set_option("mode", 2)
  for bad in (None, np.nan, np.inf):
    if bad is not None:
      lp[lp.size // 2] = bad
    out, deltas = bp.run_with_diffs(infer.BPArrays(lp.copy(), ft.copy(), ev.copy()), 5)
    ref, ref_d = lbp.run_with_diffs(g, lp, ft, ev, 5, 0.5, temperature)
    np.testing.assert_array_equal(_np(out.ftov_msgs), ref)
    np.testing.assert_array_equal(_np(deltas), ref_d)
  np.testing.assert_array_equal(_np(bp.context.get_flat_beliefs(out)),
                                lbp.get_flat_beliefs(g, ref, ev))


def _uneven_union(kind):
  """Connected graphs of different sizes, layouts and factor kinds, and their
  inputs as one union."""
  from pgmax_amd import batch
  rng = np.random.default_rng(5)
  if kind == "binary":  # one float per message in the per-phase shape
    ws = [batch.grid_wiring(n, n, 2, torus=True, full_tables=True) for n in (3, 9, 30)]
  elif kind == "mixed":  # planar and plain blocks, lane-group tiles
    ws = [batch.grid_wiring(n, n, s, full_tables=True)
          for n, s in ((2, 2), (7, 5), (20, 2), (3, 8), (12, 3))]
  elif kind == "heavy":  # stars: centres of 5 and 40 edges, two-kernel iterations
    ws = [batch.pairwise_wiring(n + 1, s, np.stack([np.zeros(n, int), np.arange(1, n + 1)], 1),
                                full_tables=True) for n, s in ((5, 3), (40, 2), (40, 4))]
  elif kind == "bipartite":  # complete, binary: the plan of k_bipartite
    ws = [batch.pairwise_wiring(33 + 35, 2, np.array([[i, 33 + j] for i in range(33)
                                                      for j in range(35)]), full_tables=True)]
  else:  # 12 states: general Enum blocks
    ws = [batch.grid_wiring(n, n, 12, full_tables=True) for n in (2, 5)]
  bb = batch.BatchedBP(ws, temperature=1.0)
  lp = rng.normal(0, 0.4, size=bb.layout.num_lp).astype(np.float32)
  ev = rng.normal(size=bb.layout.num_vs).astype(np.float32)
  return bb, lp, ev


@pytest.mark.parametrize("temperature", [0.0, 1.0])
@pytest.mark.parametrize("kind", ["binary", "mixed", "heavy", "general", "bipartite"])
@pytest.mark.parametrize("iters,tol", [(1, 1e-3), (40, 1e-3), (41, 1e-3), (25, 0.0), (7, -1.0),
                                       (9, 1e30)])
def test_per_phase_convergence_equals_task_loop(gpu, kind, temperature, iters, tol):
  """Per-phase convergence runs stop every task where the task loop does, with
  the same messages, deltas and counts, whichever buffer a task stopped in (a
  task that stops early in a run of 40 iterations stops in the other buffer in
  one of 41)."""
  import torch
  bb, lp, ev = _uneven_union(kind)
  ft = np.random.default_rng(6).normal(size=bb.layout.num_es).astype(np.float32)
  got = {}
  for mode in (1, 2):
    for fuse in (0, 1):
      _lib.set_option("mode", mode)
      _lib.set_option("fuse", fuse)
      got[mode, fuse] = bb.run_converge(lp, ft, ev, iters, tol, 0.5, temperature)
  _lib.set_option("mode", 0)
  got["auto"] = bb.run_converge(lp, ft, ev, iters, tol, 0.5, temperature)
  ref = got[1, 0]
  for key, res in got.items():
    for a, b in zip(res, ref):
      assert torch.equal(a, b), key
  n = ref[2].cpu().numpy()
  assert (n == (1 if tol == 1e30 else iters)).all() or tol in (1e-3, 0.0)
  if tol == 1e-3 and iters > 1:
    assert (n < iters).any()
  bb.close()


@pytest.mark.parametrize("tile", [0, 16, 32])
@pytest.mark.parametrize("temperature", [0.0, 1.0])
def test_short_lane_tiles_match_oracle(gpu, tile, temperature):
  """Lane-group tiles of one and two passes (and the untuned choice) on grids
  whose factors fill no tile, exactly one, and one and a bit, with shared and
  with own tables."""
  from pgmax_amd import batch
  # 64 / S factors per wavefront and pass, four wavefronts: 256 / S a tile
  ws = [batch.grid_wiring(h, w, s, full_tables=True)
        for h, w, s in ((2, 2, 3), (1, 33, 8), (1, 34, 8), (1, 49, 5), (1, 50, 5), (9, 13, 2),
                        (6, 7, 7), (17, 16, 4))]
  bb = batch.BatchedBP(ws, temperature=temperature)
  rng = np.random.default_rng(3)
  shared = np.concatenate([np.tile(rng.normal(size=s * s), nf) for nf, s in (
      (4, 3), (32, 8), (33, 8), (48, 5), (49, 5), (9 * 12 + 8 * 13, 2), (71, 7), (511, 4))])
  own = rng.normal(size=shared.size)
  ev = rng.normal(size=bb.layout.num_vs).astype(np.float32)
  ft = rng.normal(size=bb.layout.num_es).astype(np.float32)
  _lib.set_option("tile", tile)
  for lp in (shared.astype(np.float32), own.astype(np.float32)):
    assert lp.size == bb.layout.num_lp
    out, d = bb.run(lp, ft, ev, 9, 0.5, temperature)
    ref, ref_d = lbp.run_with_diffs(lbp.graph_from_flat(bb.union), lp, ft, ev, 9, 0.5,
                                    temperature)
    np.testing.assert_array_equal(_np(out), ref)
    np.testing.assert_array_equal(_np(d), ref_d)
  bb.close()


@pytest.mark.parametrize("kind", ["torus", "bipartite", "unary", "mixed"])
@pytest.mark.parametrize("offset", [0, 1, 3])
@pytest.mark.parametrize("iters", [1, 2])
def test_entry_messages_at_any_alignment(gpu, kind, offset, iters):
  """Messages enter normalised and clipped in each engine layout, from buffers
  at any float alignment, with non-finite states."""
  import torch
  from pgmax_amd import batch
  from pgmax_amd import engine
  if kind == "torus":
    w = batch.grid_wiring(5, 7, 2, torus=True, full_tables=True)
  elif kind == "mixed":  # 2, 3, 9 and 12 states
    w = batch.BatchedBP([batch.grid_wiring(3, 3, s, full_tables=True) for s in (2, 3, 9, 12)],
                        temperature=1.0).union
  else:
    h, v = vgroup.NDVarArray(num_states=2, shape=(33,)), vgroup.NDVarArray(num_states=2, shape=(35,))
    fg = fgraph.FactorGraph(variable_groups=[h, v])
    if kind == "unary":
      for g, n in ((h, 33), (v, 35)):
        fg.add_factors(fgroup.EnumFactorGroup(variables_for_factors=[[g[i]] for i in range(n)],
                                              factor_configs=np.arange(2)[:, None]))
    fg.add_factors(fgroup.PairwiseFactorGroup(
        variables_for_factors=[[h[i], v[j]] for i in range(33) for j in range(35)]))
    w = None
    eng = infer.BP(fg.bp_state, temperature=1.0).context
    graph = lbp.graph_from_context(eng)
    eng = eng.engine
  if w is not None:
    eng, graph = engine.Engine.from_wiring(w.to_engine_wiring()), lbp.graph_from_flat(w)
  g, rng = eng.graph, np.random.default_rng(11)
  ft = rng.normal(0, 3, size=(3, g.num_es)).astype(np.float32)
  ft[0, ::7] = -3e38
  ft[1, 1::11] = -np.inf
  ft[2, 2::13] = np.inf
  ft[2, 5::17] = np.nan
  lp = rng.normal(size=(3, g.num_lp)).astype(np.float32)
  ev = rng.normal(size=g.num_vs).astype(np.float32)
  buf = torch.zeros(ft.size + offset, device="cuda")
  buf[offset:] = torch.as_tensor(ft.reshape(-1), device="cuda")
  out, d = eng.run(lp, buf[offset:].view(3, -1), ev, iters, 0.5, 1.0)
  for b in range(3):
    ref, ref_d = lbp.run_with_diffs(graph, lp[b], ft[b], ev, iters, 0.5, 1.0)
    np.testing.assert_array_equal(_np(out)[b], ref)
    np.testing.assert_array_equal(_np(d)[b], ref_d)


def _binary_graph(kind):
  from pgmax_amd import batch
  grid = lambda h, w, torus: batch.grid_wiring(h, w, 2, torus=torus, full_tables=True)
  if kind == "tiny":
    return grid(1, 2, False)
  if kind == "whole":  # 512 factors: a workgroup's last
    return grid(16, 16, True)
  if kind == "rings":  # 544: the first with rings
    return grid(17, 16, True)
  if kind == "open":
    return grid(41, 30, False)
  if kind == "chain":
    return grid(1, 801, False)
  if kind == "union":  # components of a workgroup each, merged and not
    return batch.BatchedBP([grid(n, n, True) for n in (3, 9, 3, 16, 12)], temperature=1.0).union
  if kind == "slots":  # rings, 18,432 factors: deltas fold into several slots each
    return grid(96, 96, True)
  if kind == "slots union":  # the same without rings, 16,896 factors
    return batch.BatchedBP([grid(16, 16, True)] * 33, temperature=1.0).union
  if kind == "parallel":  # two factors on every other pair
    pairs = [[i, i + 1] for i in range(799)] + [[i, i + 1] for i in range(0, 799, 2)]
    return batch.pairwise_wiring(800, 2, np.array(pairs), full_tables=True)
  rng = np.random.default_rng(0)  # rings grow past a workgroup: no patches
  pairs = np.concatenate([np.sort(rng.permutation(900).reshape(-1, 2), 1) for _ in range(3)])
  return batch.pairwise_wiring(900, 2, np.unique(pairs, axis=0), full_tables=True)


@pytest.mark.parametrize("kind", ["tiny", "whole", "rings", "open", "chain", "union", "parallel",
                                  "slots", "slots union", "random"])
@pytest.mark.parametrize("temperature", [0.0, 0.35, 1.0])
@pytest.mark.parametrize("iters", [1, 4, 7])
def test_patches_match_oracle(gpu, kind, temperature, iters):
  """Several iterations per launch on patches: the oracle's messages and
  deltas, with fewer, exactly and more iterations than rings, batched, from
  buffers at an odd float offset, with non-finite tables and evidence."""
  import torch
  from pgmax_amd import engine
  w = _binary_graph(kind)
  eng, graph = engine.Engine.from_wiring(w.to_engine_wiring()), lbp.graph_from_flat(w)
  g, rng = eng.graph, np.random.default_rng(13)
  def shifted(x):
    buf = torch.zeros(x.size + 1, device="cuda")
    buf[1:] = torch.as_tensor(x.reshape(-1), device="cuda")
    return buf[1:].view(x.shape)
  ft = rng.normal(size=(2, g.num_es)).astype(np.float32)
  lp = rng.normal(size=(2, g.num_lp)).astype(np.float32)
  ev = rng.normal(size=(2, g.num_vs)).astype(np.float32)
  lp[1, 1] = np.inf
  lp[1, -1] = np.nan
  ev[1, g.num_vs // 2] = -np.inf
  _lib.set_option("mode", 4)
  out, d = eng.run(shifted(lp), shifted(ft), shifted(ev), iters, 0.5, temperature)
  _lib.set_option("mode", 0)
  auto, auto_d = eng.run(lp, ft, ev, iters, 0.5, temperature)
  for b in range(2):
    ref, ref_d = lbp.run_with_diffs(graph, lp[b], ft[b], ev[b], iters, 0.5, temperature)
    for o, od in ((out, d), (auto, auto_d)):
      np.testing.assert_array_equal(_np(o)[b], ref)
      np.testing.assert_array_equal(_np(od)[b], ref_d)


@pytest.mark.parametrize("kind,iters,launches", [("whole", 9, 1), ("rings", 4, 1),
                                                 ("rings", 5, 2), ("rings", 9, 3)])
def test_patch_launches_are_counted(gpu, kind, iters, launches):
  """The per-kernel record holds every launch of a run on patches."""
  from pgmax_amd import engine
  eng = engine.Engine.from_wiring(_binary_graph(kind).to_engine_wiring())
  g = eng.graph
  zeros = [np.zeros(n, np.float32) for n in (g.num_lp, g.num_es, g.num_vs)]
  _lib.profile_kernels()
  _lib.set_option("mode", 4)
  _lib.set_option("profile", 2)
  eng.run(*zeros, iters, 0.5, 1.0)
  kernels = _lib.profile_kernels()
  _lib.profile_read()
  assert {k: n for k, (_, n) in kernels.items()} == {"fac_fused": launches}


@pytest.mark.parametrize("kind", ["parents 1", "parents 2", "parents 3", "mixed", "wave"])
@pytest.mark.parametrize("logical", ["or", "and"])
@pytest.mark.parametrize("temperature", [0.0, 0.7])
def test_logical_blocks_match_oracle(gpu, kind, logical, temperature):
  """OR / AND blocks whose factors all have as many parents and whose do not,
  and the row chunks of a variable that is the same slot of 41 and of 65
  consecutive factors (positions 4, 6 and 8 floats apart, whole and partial
  chunks, a lone edge), in the per-phase and the automatic shape."""
  group = {"or": fgroup.ORFactorGroup, "and": fgroup.ANDFactorGroup}[logical]
  rng = np.random.default_rng(23)
  v = vgroup.NDVarArray(num_states=2, shape=(700,))
  if kind == "wave":
    facs = [[v[i] for i in rng.choice(700, size=n + 1, replace=False)]
            for n in (33, 64, 128, 255, 256)]
  else:
    sizes = [2] * 106 if kind == "mixed" else [int(kind[-1])] * 106
    if kind == "mixed":
      sizes[3], sizes[50], sizes[90] = 1, 3, 3
    rest, facs = iter(range(2, 700)), []
    for i, n in enumerate(sizes):  # variable 0 in 41 factors, then variable 1 in 65
      facs.append([v[0] if i < 41 else v[1]] + [v[next(rest)] for _ in range(n)])
  fg = fgraph.FactorGraph(variable_groups=v)
  fg.add_factors(group(variables_for_factors=facs))
  bp = infer.BP(fg.bp_state, temperature=temperature)
  graph = lbp.graph_from_context(bp.context)
  ev = rng.normal(size=1400).astype(np.float32)
  ft = rng.normal(size=bp.init().ftov_msgs.shape[0]).astype(np.float32)
  lp = np.zeros((0,), np.float32)
  ref, ref_d = lbp.run_with_diffs(graph, lp, ft, ev, 5, 0.5, temperature)
  for mode in (0, 2):
    _lib.set_option("mode", mode)
    out, d = bp.run_with_diffs(infer.BPArrays(log_potentials=lp, ftov_msgs=ft, evidence=ev), 5)
    np.testing.assert_array_equal(_np(out.ftov_msgs), ref)
    np.testing.assert_array_equal(_np(d), ref_d)
  np.testing.assert_array_equal(_np(bp.context.get_flat_beliefs(out)),
                                lbp.get_flat_beliefs(graph, ref, ev))


@pytest.mark.parametrize("sizes", [(2,), (1, 2, 8), (9, 16), (7, 17, 40)])
def test_map_and_marginals_at_register_sizes(gpu, sizes):
  """Variables of states that stay in registers and that do not, mixed in a
  graph, with ties, infinite and NaN beliefs in each: the oracle's first maximal
  state and softmax, bit for bit."""
  groups = [vgroup.NDVarArray(num_states=s, shape=(70,)) for s in sizes]
  fg = fgraph.FactorGraph(variable_groups=groups)
  for g in groups:
    n = g.num_states.reshape(-1)[0]
    fg.add_factors(fgroup.EnumFactorGroup(variables_for_factors=[[g[i]] for i in range(70)],
                                          factor_configs=np.arange(n)[:, None]))
  bp = infer.BP(fg.bp_state, temperature=1.0)
  eng = bp.context.engine
  rng = np.random.default_rng(3)
  ev = rng.integers(-3, 3, size=eng.graph.num_vs).astype(np.float32)  # (ties)
  at = 0
  for n in sizes:  # of every size: a NaN, a -inf, a +inf, and only -inf
    ev[at + n // 2], ev[at + n], ev[at + 3 * n - 1] = np.nan, -np.inf, np.inf
    ev[at + 3 * n:at + 4 * n] = -np.inf
    at += 70 * n
  ft = np.zeros(eng.graph.num_es, np.float32)
  bel, dec, marg = (_np(x) for x in eng.beliefs_decode(ev, ft))
  np.testing.assert_array_equal(bel, ev)
  vs0 = np.concatenate([[0], np.cumsum(np.repeat(sizes, 70))])
  ref_dec, ref_marg = lbp.map_and_marginals(bel, vs0)
  np.testing.assert_array_equal(dec, ref_dec)
  np.testing.assert_array_equal(marg, ref_marg)  # NaN where the oracle has NaN
  assert np.isnan(marg).any() and np.isfinite(marg).any()
