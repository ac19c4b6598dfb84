"""TRWP's reverse scan for 21 labels and a 2-D table with four wavefronts per chain (MPL_OPT_TEAM_SCANS)
against the fp64 oracle: chains around a block of six pixels, both kinds of dcontext, gradients that are left
out, argmin labels that crowd on one target, terms that are not finite; both soft-weighted scans."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

L = 21


def _problem(n_dir, n_iter, B, H, W, seed, crowd=False):
  rng = np.random.default_rng(seed)
  ctx = np.triu(rng.random((L, L)), 1).astype(np.float32)
  ew = (rng.random((n_dir, B, 1, H, W)) - 0.2).astype(np.float32)
  dcost = rng.standard_normal((B, 1, H, W, L)).astype(np.float32)
  imin = rng.integers(0, L, (n_iter, n_dir, B, 1, H, W, L)).astype(np.uint8)
  if crowd:
    imin[...] = rng.integers(0, L, imin.shape[:-1] + (1,))
  inorm = rng.integers(0, L, (n_iter, n_dir, B, 1, H, W)).astype(np.uint8)
  return ctx, ew, dcost, imin, inorm


def _backward(gpu, problem, option=2, **kw):
  from mplayers_amd import _lib
  ctx, ew, dcost, imin, inorm = problem
  _lib.set_option(_lib.OPT_TEAM_SCANS, option)
  try:
    return gpu.gpu_backward("TRWP", ctx, ew, dcost, imin, inorm, 0.5, **kw)
  finally:
    _lib.set_option(_lib.OPT_TEAM_SCANS, 1)


@pytest.mark.parametrize("n_dir,B,H,W", [(2, 1, 1, 1), (4, 1, 2, 5), (4, 2, 6, 7), (8, 1, 12, 13), (4, 1, 3, 50),
                                         (16, 1, 9, 11)])
@pytest.mark.parametrize("crowd", [False, True])
def test_backward_against_the_oracle(gpu, oracle, n_dir, B, H, W, crowd):
  from mplayers_amd import _lib
  problem = _problem(n_dir, 2, B, H, W, 100 * H + W, crowd)
  ctx, ew, dcost, imin, inorm = problem
  for same, flags in ((False, 0), (True, _lib.F_DCONTEXT_SAME_LABEL), (False, _lib.F_FUSED_PAIRS_OFF)):
    print("case", n_dir, B, H, W, crowd, same, flags, flush=True)
    ref = oracle.backward("TRWP", ctx.astype(np.float64), ew.astype(np.float64), dcost.astype(np.float64), imin,
                          inorm, 0.5, same_label=same)
    got = _backward(gpu, problem, flags=flags | _lib.F_PACKED_OFF)
    for a, b, what in zip(got, ref, ("dunary", "dcontext", "dedge_weights")):
      # sums of at most a few thousand products: 1e-4 of the largest entry, as everywhere
      assert np.abs(a - b).max() <= 1e-4 * max(1.0, float(np.abs(b).max())), what
    for want_dctx, want_dedge in ((False, False), (True, False), (False, True)):
      part = _backward(gpu, problem, flags=flags | _lib.F_PACKED_OFF, want_dctx=want_dctx, want_dedge=want_dedge)
      assert np.array_equal(part[0], got[0])
      if want_dedge:
        assert np.array_equal(part[2], got[2])


def _same_where_not_finite(four, one):
  for a, b, what in zip(four, one, ("dunary", "dcontext", "dedge_weights")):
    assert np.array_equal(np.isnan(a), np.isnan(b)), what
    assert np.array_equal(np.isposinf(a), np.isposinf(b)) and np.array_equal(np.isneginf(a), np.isneginf(b)), what
    ok = np.isfinite(b)
    assert np.abs(a[ok] - b[ok]).max() <= 1e-4 * max(1.0, float(np.abs(b[ok]).max())), what


@pytest.mark.parametrize("value", [np.inf, -np.inf, np.nan])
def test_terms_that_are_not_finite(gpu, value):
  """They reach the entries they reach with one wavefront per chain, and the others are what they are there."""
  problem = _problem(4, 1, 1, 9, 14, 3)
  problem[2][0, 0, 4, 5, 7] = value
  _same_where_not_finite(_backward(gpu, problem, 2), _backward(gpu, problem, 0))


@pytest.mark.parametrize("value", [np.inf, -np.inf, np.nan, 1e38])
@pytest.mark.parametrize("y,x", [(4, 5), (0, 0), (8, 13), (4, 12)])
def test_edge_weights_that_are_not_finite(gpu, value, y, x):
  """The same for an edge weight, and for one whose product with a gradient overflows: only dcontext has it as
  a factor, in the entries that the argmin labels of its pixel point at."""
  problem = _problem(4, 1, 1, 9, 14, 4)
  problem[1][:, 0, 0, y, x] = value
  if np.isfinite(value):
    problem[2][0, 0, y, x] *= 1e10
  one, four = _backward(gpu, problem, 0), _backward(gpu, problem, 2)
  bad = ~np.isfinite(one[1])
  assert bad.any() and not bad.all()
  assert np.array_equal(~np.isfinite(four[1]), bad)
  four[1][bad] = one[1][bad]  # (infinities that meet in another order)
  _same_where_not_finite(four, one)


@pytest.mark.parametrize("n_dir,B,H,W", [(4, 1, 1, 1), (4, 1, 2, 5), (4, 2, 6, 7), (8, 1, 12, 13), (4, 1, 3, 50)])
@pytest.mark.parametrize("pairs", [True, False])
def test_soft_backward_against_the_oracle(gpu, oracle, n_dir, B, H, W, pairs):
  """Soft-weighted TRWP: the same scan with the softmin's stored parts in the place of the argmin labels."""
  import torch
  from mplayers_amd import _lib, lib_stereo
  rng = np.random.default_rng(100 * H + W)
  unary = rng.random((B, 1, H, W, L)).astype(np.float32)
  ctx = np.triu(rng.random((L, L)), 1).astype(np.float32)
  ew = (0.2 + rng.random((n_dir, B, 1, H, W))).astype(np.float32)
  dcost = rng.standard_normal((B, 1, H, W, L)).astype(np.float32)
  fwd = oracle.forward_soft(unary, ctx, ew, n_dir, 2, 0.5)
  ref = oracle.backward_soft(ctx.astype(np.float64), ew.astype(np.float64), dcost.astype(np.float64),
                             fwd["msg_edge_label"].astype(np.float64), fwd["msg_norm_index"], 0.5)
  up = lambda a: torch.as_tensor(np.ascontiguousarray(a)).cuda()
  print("case", n_dir, B, H, W, pairs, flush=True)
  try:
    for option in (0, 2):
      _lib.set_option(_lib.OPT_TEAM_SCANS, option)
      g = up(dcost)
      got = g.new_zeros(B, 1, H, W, L), g.new_zeros(L, L), g.new_zeros(n_dir, B, 1, H, W)
      lib_stereo.TRWP_hard_soft.backward_soft(0.5, g, up(ctx), up(ew), up(fwd["msg_edge_label"]),
                                              up(fwd["msg_norm_index"]), *got, g.new_full((n_dir, B, 1, H, W, L), 3.5),
                                              g.new_empty(0), flags=0 if pairs else _lib.F_FUSED_PAIRS_OFF)
      for a, b, what in zip(got, ref, ("dunary", "dcontext", "dedge_weights")):
        # sums of at most a few thousand products: 1e-4 of the largest entry, as everywhere
        assert np.abs(a.cpu().numpy() - b).max() <= 1e-4 * max(1.0, float(np.abs(b).max())), (option, what)
  finally:
    _lib.set_option(_lib.OPT_TEAM_SCANS, 1)


def _soft_backward(option, dcost, ctx, ew, duals, norm, flags=0, **kw):
  import torch
  from mplayers_amd import _lib, lib_stereo
  up = lambda a: torch.as_tensor(np.ascontiguousarray(a)).cuda()
  _lib.set_option(_lib.OPT_TEAM_SCANS, option)
  try:
    g = up(dcost)
    got = g.new_zeros(dcost.shape), g.new_zeros(L, L), g.new_zeros(ew.shape)
    lib_stereo.TRWP_hard_soft.backward_soft(0.5, g, up(ctx), up(ew), up(duals), up(norm), *got,
                                            g.new_full(ew.shape + (L,), 3.5), g.new_empty(0), flags=flags)
    return [x.cpu().numpy() for x in got]
  finally:
    _lib.set_option(_lib.OPT_TEAM_SCANS, 1)


@pytest.mark.parametrize("n_dir,B,H,W", [(4, 1, 1, 1), (4, 1, 6, 7), (8, 1, 12, 13), (4, 1, 3, 50)])
@pytest.mark.parametrize("value", [np.nan, np.inf, 3e38])
def test_soft_backward_reads_no_duals_of_chain_starts(gpu, oracle, n_dir, B, H, W, value):
  """The forward scan does not write them (a chain start has no message): whatever is in that memory reaches no
  gradient, whether the scan has one wavefront per chain or four."""
  from mplayers_amd import _lib
  rng = np.random.default_rng(100 * H + W + 2)
  unary = (0.1 + rng.random((B, 1, H, W, L))).astype(np.float32)
  ctx = np.triu(rng.random((L, L)), 1).astype(np.float32)
  ew = (0.2 + rng.random((n_dir, B, 1, H, W))).astype(np.float32)
  dcost = rng.standard_normal((B, 1, H, W, L)).astype(np.float32)
  fwd = oracle.forward_soft(unary, ctx, ew, n_dir, 2, 0.5)
  duals, norm = fwd["msg_edge_label"].astype(np.float32), fwd["msg_norm_index"]
  ref = oracle.backward_soft(ctx.astype(np.float64), ew.astype(np.float64), dcost.astype(np.float64),
                             fwd["msg_edge_label"].astype(np.float64), norm, 0.5)
  starts = (duals == 0).all(axis=(-1, -2))  # (the oracle leaves them at zero; the others are positive)
  assert starts.any()
  duals[starts] = value
  duals[starts, ::2] *= -1
  for option in (0, 2):
    for flags in (0, _lib.F_FUSED_PAIRS_OFF):
      print("case", n_dir, B, H, W, value, option, flags, flush=True)
      for a, b, what in zip(_soft_backward(option, dcost, ctx, ew, duals, norm, flags), ref,
                            ("dunary", "dcontext", "dedge_weights")):
        # sums of at most a few thousand products: 1e-4 of the largest entry, as everywhere
        assert np.abs(a - b).max() <= 1e-4 * max(1.0, float(np.abs(b).max())), (option, what)


@pytest.mark.parametrize("value", [np.inf, np.nan])
def test_soft_backward_of_one_pixel(gpu, value):
  """An image of one pixel has chain starts only: its gradient, finite or not, reaches neither the table nor the
  edge weights."""
  rng = np.random.default_rng(5)
  ctx = np.triu(rng.random((L, L)), 1).astype(np.float32)
  ew = np.ones((4, 1, 1, 1, 1), np.float32)
  dcost = rng.standard_normal((1, 1, 1, 1, L)).astype(np.float32)
  dcost[..., 7] = value
  for option in (0, 2):
    print("case", value, option, flush=True)
    _, dctx, dedge = _soft_backward(option, dcost, ctx, ew, np.zeros((2, 4, 1, 1, 1, 1, L, L), np.float32),
                                    np.zeros((2, 4, 1, 1, 1, 1), np.uint8))
    assert not dctx.any() and not dedge.any()


@pytest.mark.parametrize("n_dir,B,H,W", [(4, 1, 1, 1), (4, 1, 2, 5), (4, 2, 6, 7), (8, 1, 12, 13), (4, 1, 3, 50)])
@pytest.mark.parametrize("train", [True, False])
def test_soft_forward_against_the_oracle(gpu, oracle, n_dir, B, H, W, train):
  """Soft-weighted TRWP forward, one and four wavefronts, pairs in one launch and in two."""
  import torch
  from mplayers_amd import _lib, lib_stereo
  rng = np.random.default_rng(100 * H + W + 1)
  unary = rng.random((B, 1, H, W, L)).astype(np.float32)
  ctx = np.triu(rng.random((L, L)), 1).astype(np.float32)
  ew = (0.2 + rng.random((n_dir, B, 1, H, W))).astype(np.float32)
  start = rng.random((n_dir, B, 1, H, W, L)).astype(np.float32)  # what the scans leave alone shows
  up = lambda a: torch.as_tensor(np.ascontiguousarray(a)).cuda()
  u8 = dict(dtype=torch.uint8, device="cuda")

  def forward(option, flags, u=unary, m0=start):
    u = up(u)
    msg, cost, scratch = up(m0), torch.zeros_like(u), torch.zeros_like(u)
    duals = u.new_full((2, n_dir, B, 1, H, W, L, L), 7.0) if train else torch.empty(0)
    norm = torch.full((2, n_dir, B, 1, H, W), 77, **u8) if train else torch.empty(0, dtype=torch.uint8)
    _lib.set_option(_lib.OPT_TEAM_SCANS, option)
    try:
      lib_stereo.TRWP_hard_soft.forward_soft(0.5, 2, u, up(ctx), up(ew), msg, duals, norm, cost, scratch,
                                             torch.empty(0, **u8), flags=flags)
      torch.cuda.synchronize()
    finally:
      _lib.set_option(_lib.OPT_TEAM_SCANS, 1)
    return [x.cpu().numpy() for x in ((msg, cost, duals, norm) if train else (msg, cost))]

  print("case", n_dir, B, H, W, train, flush=True)
  ref = oracle.forward_soft(unary, ctx, ew, n_dir, 2, 0.5)
  got = forward(2, 0, m0=np.zeros_like(start))
  scale = max(1.0, float(np.abs(ref["cost_final"]).max()))
  assert np.abs(got[0] - ref["msg"]).max() <= 2e-5 * scale
  assert np.abs(got[1] - ref["cost_final"]).max() <= 2e-5 * scale
  one, pairs, single = forward(0, 0), forward(2, 0), forward(2, _lib.F_FUSED_PAIRS_OFF)
  for a, b, c in zip(one, pairs, single):
    assert np.array_equal(b, c)
    if a.dtype != np.uint8:
      assert np.abs(a - b).max() <= 2e-5 * scale
    else:  # (labels whose softmin messages are closer than the tolerance aside)
      assert (a != b).mean() <= 0.02 and np.array_equal(a == 77, b == 77)
  for value in (np.inf, -np.inf, np.nan):
    bad = unary.copy()
    bad[0, 0, H // 2, W // 2, 18] = value
    for a, b in zip(forward(0, 0, bad)[:2], forward(2, 0, bad)[:2]):
      assert np.array_equal(np.isfinite(a), np.isfinite(b)), value
