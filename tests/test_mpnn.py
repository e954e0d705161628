"""Warm-start network: FP64 oracle pinned by finite differences (CPU); GPU
forward / backward kernels against the oracle; training gain (GPU)."""

import numpy as np
import pytest

from oracle import mpnn as omp
from pgmax_amd import batch


def _spin_glass(side, seed, torus=True):
  rng = np.random.default_rng(seed)
  w = batch.grid_wiring(side, side, 2, torus=torus, full_tables=True)
  nf = w.num_log_potentials // 4
  J = rng.normal(size=nf)
  lp = np.stack([J, -J, -J, J], 1).reshape(-1)
  ev = rng.normal(0, 0.5, size=w.num_var_states)
  return w, lp, ev


def _graph(w):
  return omp.pairwise_binary_graph(w.var_states_for_edge_states, w.evidence_to_vars)


def test_features_orientation():
  """The second edge of a factor sees the transposed table."""
  w, lp, ev = _spin_glass(3, 0)
  ev_var, pos, lp0, nv = _graph(w)
  lp = np.arange(lp.size, dtype=np.float64) ** 1.5  # asymmetric tables
  x = omp.features(ev_var, pos, lp0, lp, ev)
  t = lp[:4]
  assert x[0, 2] == pytest.approx((t[0] + t[3] - t[1] - t[2]) / 4)
  assert x[0, 3] == pytest.approx((t[2] + t[3] - t[0] - t[1]) / 2)  # field on the first var
  assert x[1, 3] == pytest.approx((t[1] + t[3] - t[0] - t[2]) / 2)  # field on the second var
  assert x[0, 4] == pytest.approx(x[1, 3]) and x[1, 4] == pytest.approx(x[0, 3])
  evd = ev.reshape(-1, 2)
  assert x[0, 0] == pytest.approx(evd[ev_var[0], 1] - evd[ev_var[0], 0])
  assert x[0, 1] == pytest.approx(x[1, 0])


def test_oracle_gradients_match_finite_differences():
  w, lp, ev = _spin_glass(3, 1)
  ev_var, pos, lp0, nv = _graph(w)
  x = omp.features(ev_var, pos, lp0, lp, ev)
  p = omp.init_params(3)
  for k in p:  # move biases off zero so every ReLU is away from its kink
    if k.startswith("b"):
      p[k] = p[k] + 0.05
  target = np.random.default_rng(2).normal(size=x.shape[0])
  y, cache = omp.forward(p, x, ev_var, nv)
  g = omp.backward(p, cache, y, target, ev_var, nv)
  rng = np.random.default_rng(4)
  h = 1e-6
  for k in p:
    flat = p[k].reshape(-1)
    for idx in rng.choice(flat.size, size=min(6, flat.size), replace=False):
      old = flat[idx]
      flat[idx] = old + h
      lp_ = omp.loss(omp.forward(p, x, ev_var, nv)[0], target)
      flat[idx] = old - h
      lm_ = omp.loss(omp.forward(p, x, ev_var, nv)[0], target)
      flat[idx] = old
      fd = (lp_ - lm_) / (2 * h)
      an = g[k].reshape(-1)[idx]
      assert an == pytest.approx(fd, rel=1e-5, abs=1e-9), (k, idx)


def test_oracle_planted_mistake_fails_finite_differences():
  """Dropping the -h_e term of the variable aggregate breaks the check."""
  w, lp, ev = _spin_glass(3, 5)
  ev_var, pos, lp0, nv = _graph(w)
  x = omp.features(ev_var, pos, lp0, lp, ev)
  p = omp.init_params(6)
  target = np.zeros(x.shape[0])
  y, cache = omp.forward(p, x, ev_var, nv)
  g = omp.backward(p, cache, y, target, ev_var, nv)
  # a wrong backward that forgets the self-exclusion of the variable sum
  E = x.shape[0]
  other = np.arange(E) ^ 1
  dy = 2.0 * (y - target) / E
  dh = np.outer(dy, p["wh"])
  for l in range(omp.LAYERS, 0, -1):
    dpre = dh * (cache["h"][l] > 0)
    dz = dpre @ p[f"W{l}"].T
    tv = np.zeros((nv, omp.HIDDEN))
    np.add.at(tv, ev_var, dz[:, 64:128])
    dh = dz[:, :64] + tv[ev_var] + dz[:, 128:][other]  # missing "- d_var"
  wrong_b0 = (dh * (cache["h"][0] > 0)).sum(0)
  assert not np.allclose(wrong_b0, g["b0"], rtol=1e-3)


def test_message_ratio_round_trip():
  y = np.array([-2.0, 0.0, 3.5])
  m = omp.messages_from_ratio(y)
  assert np.all(m.reshape(-1, 2).max(1) == 0)
  np.testing.assert_allclose(omp.ratio_from_messages(m), y)


def test_flat_layout_round_trip():
  p = omp.init_params(1)
  flat = omp.to_flat(p)
  assert flat.size == 37697  # PGX_MPNN_NUM_PARAMS
  q = omp.from_flat(flat)
  for k in p:
    np.testing.assert_array_equal(p[k], q[k])


def test_bf16_rounding():
  x = np.array([1.0, 1.00390625, 1.005859375, -3.14159, 0.0, 1e-30])
  r = omp.bf16(x)
  assert r[0] == 1.0 and r[1] == 1.0  # tie rounds to even
  assert r[2] == 1.0078125
  assert abs(r[3] + 3.140625) < 1e-12
  assert r[4] == 0.0 and r[5] > 0


# ---------------------------------------------------------------------------
# GPU
# ---------------------------------------------------------------------------


def _batch_inputs(side, batch, seed):
  rng = np.random.default_rng(seed)
  w = batch_mod_grid(side)
  nf = w.num_log_potentials // 4
  J = rng.normal(size=(batch, nf))
  lp = np.stack([J, -J, -J, J], -1).reshape(batch, -1)
  ev = rng.normal(0, 0.5, size=(batch, w.num_var_states))
  return w, lp, ev


def batch_mod_grid(side):
  return batch.grid_wiring(side, side, 2, torus=True, full_tables=True)


def _oracle_rows(w, lp, ev, p, target=None, emulate=True):
  ev_var, pos, lp0, nv = _graph(w)
  ys, grads, losses = [], [], []
  B = lp.shape[0]
  xs = [omp.features(ev_var, pos, lp0, lp[b], ev[b]) for b in range(B)]
  # one batched graph: B disjoint copies
  x = np.concatenate(xs)
  E = ev_var.size
  ev_all = np.concatenate([ev_var + b * nv for b in range(B)])
  y, cache = omp.forward(p, x, ev_all, nv * B, emulate_bf16=emulate)
  if target is None:
    return y, None, None
  t = np.concatenate([omp.ratio_from_messages(target[b]) for b in range(B)])
  g = omp.backward(p, cache, y, t, ev_all, nv * B, emulate_bf16=emulate)
  return y, g, omp.loss(y, t)


@pytest.mark.gpu
@pytest.mark.parametrize("side,batch", [(6, 3), (3, 5), (17, 2)])
def test_gpu_forward_matches_oracle(gpu, side, batch):
  """Prediction against the BF16-emulating oracle. The layer kernels work on
  tiles of 16 edge rows: 3x3 tori (36 edges) put several batch elements in
  one tile, 17x17 ones (1,156 edges) end a batch element inside a tile."""
  import torch
  from pgmax_amd import engine, warmstart
  w, lp, ev = _batch_inputs(side, batch, 11)
  graph = engine.Graph(w.to_engine_wiring())
  net = warmstart.WarmStart(graph, seed=2)
  p = omp.from_flat(net.params.cpu().numpy())
  lp_t = torch.as_tensor(lp, dtype=torch.float32)
  ev_t = torch.as_tensor(ev, dtype=torch.float32)
  out = net.predict(lp_t, ev_t).cpu().numpy()
  # every batch element alone gives the same bits
  for b in range(batch):
    np.testing.assert_array_equal(net.predict(lp_t[b], ev_t[b]).cpu().numpy(), out[b])
  y_gpu = np.concatenate([omp.ratio_from_messages(out[b]) for b in range(batch)])
  y_ref, _, _ = _oracle_rows(w, lp.astype(np.float32), ev.astype(np.float32), p)
  y_64, _, _ = _oracle_rows(w, lp.astype(np.float32), ev.astype(np.float32), p, emulate=False)
  scale = max(1.0, np.abs(y_ref).max())
  d = np.abs(y_gpu - y_ref) / scale
  err = d.max()
  print(f"forward: max |gpu - bf16-emulating oracle| / scale = {err:.2e} "
        f"(99th percentile {np.quantile(d, 0.99):.2e}); "
        f"vs pure FP64 {np.abs(y_gpu - y_64).max() / scale:.2e}")
  # The GPU and the emulating oracle round to BF16 at the same places but
  # accumulate in different orders, so a value within an FP32 rounding of a
  # BF16 tie can round the other way and move its row by up to a BF16 step
  # (2^-8) of one activation. Measured: max 3.6e-7 on the 6x6 and 3x3 batches;
  # at 17x17, one row of 2,312 at 7.4e-5 and the 99th percentile 2.7e-7
  # (at 40x40 x 9: 348 rows of 57,600 above 4e-6, max 2.6e-3). Bars: 4e-6 for
  # all but 1 % of the rows, 1e-2 for every row.
  assert np.quantile(d, 0.99) < 4e-6
  assert (d > 4e-6).mean() < 0.01
  assert err < 1e-2
  if side <= 6:  # no row of these two batches sits at such a tie
    assert err < 4e-6
  assert np.all(out.reshape(batch, -1, 2).max(-1) == 0)  # normalised messages


def _row_order_cases():
  rng = np.random.default_rng(21)
  cases = {"torus 12x12": batch.grid_pairs(12, 12, True)}
  # uneven degrees (1 .. about 12), 60 variables
  pairs = set()
  while len(pairs) < 150:
    a, b = (int(v) for v in rng.integers(0, 60, 2))
    if a != b:
      pairs.add((min(a, b), max(a, b)))
  cases["random 60 vars"] = np.array(sorted(pairs), np.int64)
  # a variable of 20 edges: prediction keeps the edge-major rows
  star = [(0, k) for k in range(1, 21)] + [(k, k + 1) for k in range(1, 20)]
  cases["star of 20"] = np.array(star, np.int64)
  return cases


@pytest.mark.gpu
@pytest.mark.parametrize("case", ["torus 12x12", "random 60 vars", "star of 20"])
def test_gpu_predict_row_orders_agree(gpu, case):
  """Prediction in variable-major rows (each variable's sum over its edges
  taken inside its tile) against edge-major rows with the separate sum pass:
  the same bits, batch of 3."""
  import torch
  from pgmax_amd import _lib, engine, warmstart
  pairs = _row_order_cases()[case]
  nv = int(pairs.max()) + 1
  w = batch.pairwise_wiring(nv, 2, pairs, full_tables=True)
  rng = np.random.default_rng(5)
  J = rng.normal(size=(3, pairs.shape[0]))
  lp = torch.as_tensor(np.stack([J, -J, -J, J], -1).reshape(3, -1), dtype=torch.float32)
  ev = torch.as_tensor(rng.normal(0, 0.5, size=(3, w.num_var_states)), dtype=torch.float32)
  net = warmstart.WarmStart(engine.Graph(w.to_engine_wiring()), seed=3)
  vm = net.predict(lp, ev).cpu().numpy()
  prev = _lib.set_option("mpnn_rows", 0)
  try:
    em = net.predict(lp, ev).cpu().numpy()
  finally:
    _lib.set_option("mpnn_rows", prev)
  np.testing.assert_array_equal(vm, em)
  assert np.all(np.isfinite(vm)) and np.all(vm.reshape(3, -1, 2).max(-1) == 0)


@pytest.mark.gpu
def test_gpu_gradients_match_oracle(gpu):
  import torch
  from pgmax_amd import engine, warmstart
  w, lp, ev = _batch_inputs(6, 2, 12)
  graph = engine.Graph(w.to_engine_wiring())
  flat = omp.to_flat(omp.init_params(5))
  rng = np.random.default_rng(3)
  flat = flat + np.where(np.arange(flat.size) >= 0, 0.02 * rng.normal(size=flat.size), 0)
  net = warmstart.WarmStart(graph, params=flat.astype(np.float32))
  p = omp.from_flat(net.params.cpu().numpy())
  target = np.stack([omp.messages_from_ratio(rng.normal(size=w.num_edge_states // 2))
                     for _ in range(2)])
  loss, grads = net.loss_and_grad(torch.as_tensor(lp, dtype=torch.float32),
                                  torch.as_tensor(ev, dtype=torch.float32),
                                  torch.as_tensor(target, dtype=torch.float32))
  g_gpu = omp.from_flat(grads.cpu().numpy())
  _, g_ref, l_ref = _oracle_rows(w, lp.astype(np.float32), ev.astype(np.float32), p, target)
  print(f"loss: gpu {float(loss.cpu()):.8g} oracle {l_ref:.8g} "
        f"rel err {abs(float(loss.cpu()) - l_ref) / abs(l_ref):.2e}")
  assert float(loss.cpu()) == pytest.approx(l_ref, rel=1e-6)  # measured 3.3e-8
  for k in g_ref:
    num = np.linalg.norm(g_gpu[k] - g_ref[k])
    den = np.linalg.norm(g_ref[k]) + 1e-12
    print(f"grad {k}: rel err {num / den:.2e}")
    assert num / den < 7e-5, k  # measured <= 6.8e-6 per tensor; bar ten times that


@pytest.mark.gpu
@pytest.mark.parametrize("num,pairs,batch_size", [
    (2, "pair", 1),     # 2 rows: most of a tile empty
    (2, "pair", 37),    # variables' rows cross tiles of 16 and 64
    (21, "star", 3),    # 20 edges on a variable, 120 rows
    (9, "chain", 8),    # 128 rows: two whole tiles of 64
    (9, "chain", 9),    # and 16 rows more
])
def test_gpu_gradients_at_tile_edges(gpu, num, pairs, batch_size):
  """Backward tiles of 16 and 64 rows that are empty, full and cut by a batch
  element's end, against the oracle; the bar of the test above."""
  import torch
  from pgmax_amd import engine, warmstart
  pairs = {"pair": [[0, 1]], "star": [[0, i] for i in range(1, num)],
           "chain": [[i, i + 1] for i in range(num - 1)]}[pairs]
  w = batch.pairwise_wiring(num, 2, np.array(pairs), full_tables=True)
  rng = np.random.default_rng(num + batch_size)
  j = rng.normal(size=(batch_size, len(pairs)))
  lp = np.stack([j, -j, -j, j], -1).reshape(batch_size, -1).astype(np.float32)
  ev = rng.normal(0, 0.5, size=(batch_size, 2 * num)).astype(np.float32)
  target = np.stack([omp.messages_from_ratio(rng.normal(size=2 * len(pairs)))
                     for _ in range(batch_size)]).astype(np.float32)
  graph = engine.Graph(w.to_engine_wiring())
  flat = omp.to_flat(omp.init_params(5))
  net = warmstart.WarmStart(graph, params=(flat + 0.02 * rng.normal(size=flat.size)).astype(
      np.float32))
  loss, grads = net.loss_and_grad(*(torch.as_tensor(x) for x in (lp, ev, target)))
  got = omp.from_flat(grads.cpu().numpy())
  _, want, loss_ref = _oracle_rows(w, lp, ev, omp.from_flat(net.params.cpu().numpy()), target)
  assert float(loss.cpu()) == pytest.approx(loss_ref, rel=1e-6)
  for k in want:
    assert np.linalg.norm(got[k] - want[k]) <= 7e-5 * np.linalg.norm(want[k]) + 1e-12, k
  net.close()
  graph.close()


@pytest.mark.gpu
@pytest.mark.parametrize("side,copies", [(3, 2), (5, 64), (33, 64), (40, 128)])
def test_gpu_gradients_of_repeated_graph(gpu, side, copies):
  """A batch of 2^k copies of one graph has its loss and gradients: the mean
  over rows does not change, every per-row term is scaled by a power of two
  (so BF16 rounds it the same way), and only the FP32 sums over up to 409,600
  rows run over more partials. Their rounding is at most about
  sqrt(rows) * 2^-24 of the summed magnitudes, which the gradient's norm is a
  few per cent of: 1e-4 covers it."""
  from pgmax_amd import engine
  from pgmax_amd import warmstart
  torch = pytest.importorskip("torch")
  w, lp, ev = _spin_glass(side, 17)
  g = engine.Graph(w.to_engine_wiring())
  net = warmstart.WarmStart(g, seed=3)
  rng = np.random.default_rng(18)
  t = np.stack([np.zeros(w.num_edge_states // 2), rng.normal(size=w.num_edge_states // 2)], 1)
  args = [torch.as_tensor(np.asarray(a, np.float32).reshape(1, -1), device="cuda")
          for a in (lp, ev, t)]
  loss1, g1 = net.loss_and_grad(*args)
  loss2, g2 = net.loss_and_grad(*[a.repeat(copies, 1) for a in args])
  assert float((loss2 - loss1).abs()) <= 1e-5 * float(loss1)
  assert float((g2 - g1).norm()) <= 1e-4 * float(g1.norm())
  net.close()
  g.close()


@pytest.mark.gpu
def test_gpu_gradients_deterministic(gpu):
  import torch
  from pgmax_amd import engine, warmstart
  w, lp, ev = _batch_inputs(5, 2, 13)
  graph = engine.Graph(w.to_engine_wiring())
  net = warmstart.WarmStart(graph, seed=1)
  target = torch.zeros((2, w.num_edge_states), device="cuda")
  a = net.loss_and_grad(torch.as_tensor(lp, dtype=torch.float32), torch.as_tensor(ev, dtype=torch.float32), target)[1]
  b = net.loss_and_grad(torch.as_tensor(lp, dtype=torch.float32), torch.as_tensor(ev, dtype=torch.float32), target)[1]
  assert torch.equal(a, b)


@pytest.mark.gpu
def test_gpu_rejects_non_binary_graph(gpu):
  from pgmax_amd import engine, warmstart
  graph = engine.Graph(batch.grid_wiring(4, 4, 3, full_tables=True).to_engine_wiring())
  with pytest.raises(ValueError, match="binary"):
    warmstart.WarmStart(graph)


def _converged_samples(eng, w, n_batches, batch_size, seed, iters=600):
  """(lp, ev, converged ftov) batches; graphs not converged to 1e-6 are dropped."""
  import torch
  out = []
  for k in range(n_batches):
    _, lp, ev = _batch_inputs_w(w, batch_size, seed + k)
    lp_t = torch.as_tensor(lp, dtype=torch.float32, device="cuda")
    ev_t = torch.as_tensor(ev, dtype=torch.float32, device="cuda")
    zero = torch.zeros((batch_size, w.num_edge_states), device="cuda")
    ft, deltas = eng.run(lp_t, zero, ev_t, iters, 0.5, 1.0)
    keep = (deltas[:, -1] < 1e-6).nonzero().reshape(-1)
    if keep.numel():
      out.append((lp_t[keep], ev_t[keep], ft[keep]))
  return out


def _batch_inputs_w(w, batch_size, seed):
  rng = np.random.default_rng(seed)
  nf = w.num_log_potentials // 4
  J = rng.normal(size=(batch_size, nf))
  lp = np.stack([J, -J, -J, J], -1).reshape(batch_size, -1)
  ev = rng.normal(0, 0.5, size=(batch_size, w.num_var_states))
  return w, lp, ev


@pytest.mark.gpu
def test_gpu_trained_warm_start(gpu):
  """Trained on converged messages of 10x10 spin glasses, the network predicts
  held-out converged messages far better than the zero start; BP from its
  prediction reaches the same fixed point; the iteration counts of both
  starts are reported (on these frustrated grids BP's slowest mode, not the
  start, sets the count, so no speed-up is asserted)."""
  import torch
  from pgmax_amd import engine, warmstart
  w = batch_mod_grid(10)
  eng = engine.Engine.from_wiring(w.to_engine_wiring())
  train = _converged_samples(eng, w, 24, 32, seed=100)
  net = warmstart.WarmStart(eng, seed=0)
  losses = net.fit(train, steps=400, lr=3e-3)
  print(f"loss: first {losses[:5].mean():.4f} last {losses[-20:].mean():.4f}")
  assert losses[-20:].mean() < 0.6 * losses[:5].mean()
  held = _converged_samples(eng, w, 2, 32, seed=999)
  lp_t = torch.cat([h[0] for h in held])
  ev_t = torch.cat([h[1] for h in held])
  target = torch.cat([h[2] for h in held])
  pred = net.predict(lp_t, ev_t)
  ratio = lambda m: (m.reshape(m.shape[0], -1, 2)[..., 1] - m.reshape(m.shape[0], -1, 2)[..., 0])
  mse_net = float(((ratio(pred) - ratio(target)) ** 2).mean())
  mse_zero = float((ratio(target) ** 2).mean())
  print(f"held-out log-ratio MSE: network {mse_net:.4f}, zero start {mse_zero:.4f}")
  assert mse_net < 0.8 * mse_zero
  n = lp_t.shape[0]
  cold = warmstart.solve(eng, None, lp_t, ev_t, max_iters=2000, tol=1e-4)
  warm = warmstart.solve(eng, net, lp_t, ev_t, max_iters=2000, tol=1e-4)
  ci = cold.iterations.float().cpu().numpy()
  wi = warm.iterations.float().cpu().numpy()
  print(f"iterations to 1e-4 on {n} converging graphs: zero start {ci.mean():.1f}, "
        f"warm start {wi.mean():.1f}, fallbacks {int(warm.fell_back.sum())}")
  bc = eng.beliefs(ev_t, cold.ftov).cpu().numpy().reshape(n, -1, 2)
  bw = eng.beliefs(ev_t, warm.ftov).cpu().numpy().reshape(n, -1, 2)
  diff = np.abs((bc[..., 1] - bc[..., 0]) - (bw[..., 1] - bw[..., 0])).max()
  print(f"max belief log-ratio difference: {diff:.2e}")
  assert diff < 1e-2


@pytest.mark.gpu
def test_gpu_warm_start_fallback_reruns_from_zero(gpu):
  """A start that misses the budget is rerun from zeros: the result equals
  the zero-start run and the iterations of both runs are counted."""
  import torch
  from pgmax_amd import engine, warmstart
  w = batch_mod_grid(6)
  eng = engine.Engine.from_wiring(w.to_engine_wiring())
  _, lp, ev = _batch_inputs_w(w, 4, 5)
  lp_t = torch.as_tensor(lp, dtype=torch.float32, device="cuda")
  ev_t = torch.as_tensor(ev, dtype=torch.float32, device="cuda")
  net = warmstart.WarmStart(eng, seed=0)
  cold = warmstart.solve(eng, None, lp_t, ev_t, max_iters=3, tol=0.0)
  warm = warmstart.solve(eng, net, lp_t, ev_t, max_iters=3, tol=0.0)
  assert bool(warm.fell_back.all())
  assert torch.equal(warm.ftov, cold.ftov)
  assert torch.equal(warm.iterations, cold.iterations + 3)


@pytest.mark.gpu
def test_gpu_warm_start_has_no_gain_in_the_spin_glass_regime(gpu):
  """The evaluation regime (toroidal spin glasses, J ~ N(0,1), fields
  ~ N(0,0.5), T = 1, damping 0.5), at reduced size: a network trained on the
  converged plain-BP messages of 2,000 32x32 tori (the only side where any
  converge) is no help on 64 held-out 64x64 tori. Plain BP from zeros
  reaches max |change| <= 1e-4 within 1,000 iterations on almost none of
  them; the warm start converges on no more, and every graph it misses is
  rerun from zeros, so its final messages equal plain BP's bit for bit and
  it takes longer. The absence of a gain is what is asserted."""
  import torch
  from pgmax_amd import engine, warmstart, workloads
  w32, lp, ev = workloads.spin_glass_batch(32, 2000, seed=1000)
  eng32 = engine.Engine.from_wiring(w32.to_engine_wiring())
  lp_t = torch.as_tensor(lp, device="cuda")
  ev_t = torch.as_tensor(ev, device="cuda")
  out, deltas, iters = eng32.run_converge(lp_t, torch.zeros((2000, w32.num_edge_states), device="cuda"),
                                          ev_t, 1000, 1e-4, 0.5, 1.0)
  last = deltas[:, 0].gather(-1, (iters[:, 0].long() - 1).clamp(min=0)[:, None])[:, 0]
  keep = torch.nonzero(last <= 1e-4).reshape(-1)
  print(f"{keep.numel()} of 2000 32x32 training tori converge")
  assert 0 < keep.numel() < 200
  net32 = warmstart.WarmStart(eng32, seed=0)
  batches = [(lp_t[keep[i:i + 16]], ev_t[keep[i:i + 16]], out[keep[i:i + 16]])
             for i in range(0, int(keep.numel()), 16)]
  losses = net32.fit(batches, steps=200, lr=3e-3)
  assert losses[-10:].mean() < losses[:10].mean()
  w64, lp, ev = workloads.spin_glass_batch(64, 64, seed=99)
  eng64 = engine.Engine.from_wiring(w64.to_engine_wiring())
  net64 = warmstart.WarmStart(eng64, params=net32.params)
  lp_t = torch.as_tensor(lp, device="cuda")
  ev_t = torch.as_tensor(ev, device="cuda")
  plain = warmstart.solve(eng64, None, lp_t, ev_t, max_iters=1000, tol=1e-4)
  warm = warmstart.solve(eng64, net64, lp_t, ev_t, max_iters=1000, tol=1e-4)
  plain_it = plain.iterations.cpu().numpy().reshape(-1)
  fell = warm.fell_back.cpu().numpy().reshape(-1)
  plain_conv = int((plain_it < 1000).sum())
  warm_conv = int((~fell).sum())
  print(f"64x64 held out: plain converges on {plain_conv} of 64, warm on {warm_conv} "
        f"(fallbacks {int(fell.sum())}); mean iterations plain {plain_it.mean():.0f}, "
        f"warm {warm.iterations.float().mean().item():.0f}")
  assert plain_conv <= 3
  assert warm_conv <= plain_conv
  sel = torch.as_tensor(fell, device="cuda")
  assert torch.equal(warm.ftov[sel], plain.ftov[sel])
  assert float(warm.iterations.float().mean()) >= float(plain.iterations.float().mean())
