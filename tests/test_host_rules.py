"""The library's host rules (plans and execution shapes) as plain functions,
built with the host compiler: no GPU needed."""

import ctypes
import os
import subprocess

import pytest

from pgmax_amd import batch

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, "..", "pgmax_amd", "csrc")


@pytest.fixture(scope="module")
def rules(tmp_path_factory):
  lib = str(tmp_path_factory.mktemp("rules") / "rules.so")
  subprocess.run(["g++", "-std=c++17", "-O1", "-fPIC", "-shared",
                  os.path.join(HERE, "host_rules.cpp"), os.path.join(CSRC, "pgx_plan.cpp"),
                  os.path.join(CSRC, "pgx_shape.cpp"), "-o", lib], check=True)
  return ctypes.CDLL(lib)


def _converge_shape(rules, flat, n_it, batch_size=1, t0=False):
  w = flat.to_engine_wiring()
  out = (ctypes.c_int64 * 3)()
  assert rules.rules_converge_shape(ctypes.byref(w.struct), batch_size, n_it, int(t0), out) == 0
  return tuple(out)


def test_convergence_shape_of_a_graph_without_factors(rules):
  """No factors, no tasks: the rule answers (any shape, nothing is launched)."""
  lone = batch.grid_wiring(1, 1, 3, full_tables=True)
  assert lone.num_edge_states == 0 and lone.num_var_states == 3
  assert _converge_shape(rules, lone, 10) == (0, 1, 256)


@pytest.mark.parametrize("side,n_it,want", [
    (10, 300, (1, 256)),    # iterations of microseconds: task loop
    (30, 300, (1, 1024)),
    (100, 300, (2, 0)),     # long iterations, few idle launches
    (100, 5000, (1, 1024)),  # too many launches that might be idle
])
def test_convergence_shape_by_iterations_allowed(rules, side, n_it, want):
  torus = batch.grid_wiring(side, side, 2, torus=True, full_tables=True)
  assert _converge_shape(rules, torus, n_it)[1:] == want


@pytest.mark.parametrize("n_it", [1, 10, 300, 480, 485, 5000])
@pytest.mark.parametrize("side", [30, 100])
def test_tuned_convergence_runs_follow_the_iterations_allowed(rules, side, n_it):
  """Per-phase launches chosen by short probes run only where untuned runs of
  as many iterations may take them; runs of a fixed count take them always."""
  torus = batch.grid_wiring(side, side, 2, torus=True, full_tables=True)
  w = torus.to_engine_wiring()
  mode = lambda converge: rules.rules_tuned_mode(ctypes.byref(w.struct), 1, n_it, 0, converge)
  assert mode(1) == _converge_shape(rules, torus, n_it)[1]
  assert mode(0) == 2


_FLAGS = ("converge", "bipartite", "fusable", "wide", "logical", "patches", "square",
          "lane_tiles", "short_lane_tiles", "per_phase_converge")


def _candidates(rules, *names, tiles=100):
  out = (ctypes.c_int64 * (7 * 64))()
  n = rules.rules_candidates(sum(1 << _FLAGS.index(k) for k in names), tiles, out, 64)
  assert n <= 64
  return [tuple(out[7 * i:7 * i + 7]) for i in range(n)]


def test_autotuner_times_what_untuned_runs_take(rules):
  """(mode, threads, fuse, vec, tile, lanes, xcd): mode 0 is the untuned rules'
  own choice, in every list; the shapes those rules take by name are listed too,
  and task loops come last."""
  for flags in range(1 << len(_FLAGS)):
    names = [k for i, k in enumerate(_FLAGS) if flags >> i & 1]
    got = _candidates(rules, *names, tiles=(0, 600)[flags & 1])
    assert got.count((0, 0, 1, 3, 0, 1, 0)) == 1
    assert len(set(got)) == len(got)
    modes = [c[0] for c in got]
    assert modes.count(1) == modes[::-1].index(next(m for m in modes[::-1] if m != 1)) >= 3
    if "converge" in names:
      assert set(modes) <= {0, 1, 2} and (2 in modes) == ("per_phase_converge" in names)
  assert (2, 512, 1, 3, 32, 1, 0) in _candidates(rules, "bipartite")
  assert (2, 0, 0, 3, 256, 1, 8) in _candidates(rules, "logical", tiles=8)
  for t in (16, 32):
    assert (2, 0, 1, 3, t, 1, 0) in _candidates(rules, "converge", "fusable", "lane_tiles",
                                                "short_lane_tiles", "per_phase_converge")


def test_patches_take_edge_numbers_of_28_bits(rules):
  """A patch's threads hold their edge in 28 bits under its ring: graphs with
  more edges have no patches, whatever their components' size."""
  out = (ctypes.c_int64 * 2)()
  for flat in (batch.grid_wiring(16, 16, 2, torus=True, full_tables=True),
               batch.grid_wiring(17, 16, 2, torus=True, full_tables=True)):
    w = flat.to_engine_wiring()
    assert rules.rules_patches(ctypes.byref(w.struct), ctypes.c_int64(0), out) == 0
    assert out[0] > 0
  fit = lambda n: rules.rules_patch_edges_fit(ctypes.c_int64(n))
  assert fit(0) and fit(2) and fit(2**28 - 2) and fit(2**28)
  assert not fit(2**28 + 1) and not fit(2**28 + 2) and not fit(2**31 - 2)
  assert rules.rules_patches(None, ctypes.c_int64(2**28 + 2), out) == 0
  assert out[0] == 0
