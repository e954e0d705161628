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
