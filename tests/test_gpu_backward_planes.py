"""TRWP backward: the planes the walks of a pair hand to each other and to the next pair.

The two walks of a pair of opposite directions pass on three planes, and the plane a pair reads as
A is the one the pair before it left in its even direction's slot; the number of pairs, of iterations
and the way the walks are launched decide which slot that is.  Random argmin labels (any label is a
valid one) against the fp64 oracle, scratch filled with garbage."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.usefixtures("reverse_scans")
@pytest.mark.parametrize("L", [5, 21, 40, 64, 96, 131, 192, 250])
@pytest.mark.parametrize("n_dir,n_iter", [(2, 1), (2, 3), (4, 1), (4, 2), (8, 2), (16, 1)])
def test_planes_of_the_pairs(gpu, oracle, n_dir, n_iter, L):
  from mplayers_amd import _lib
  rng = np.random.default_rng(100 * L + 10 * n_dir + n_iter)
  B, H, W = 2, 9, 37
  ctx = (np.triu(rng.random((L, L)), 1) if L == 21 else rng.random(L)).astype(np.float32)
  ew = (0.1 + 0.9 * rng.random((n_dir, B, 1, H, W))).astype(np.float32)
  dcost = rng.standard_normal((B, 1, H, W, L)).astype(np.float32)
  imin = rng.integers(0, L, (n_iter, n_dir, B, 1, H, W, L)).astype(np.uint8)
  inorm = rng.integers(0, L, (n_iter, n_dir, B, 1, H, W)).astype(np.uint8)
  ref = oracle.backward("TRWP", ctx.astype(np.float64), ew.astype(np.float64), dcost.astype(np.float64),
                        imin, inorm, 0.5)
  routes = [0, _lib.F_FUSED_PAIRS_OFF]
  if L <= 32:
    routes += [_lib.F_PACKED_ALWAYS, _lib.F_PACKED_ALWAYS | _lib.F_FUSED_PAIRS_OFF]
  for flags in routes:
    print("case", L, n_dir, n_iter, flags, flush=True)
    got = gpu.gpu_backward("TRWP", ctx, ew, dcost, imin, inorm, 0.5, flags=flags, garbage_scratch=True)
    for name, g, r in zip(("dunary", "dcontext", "dedge"), got, ref):
      # the gradient bar of the GPU tests: 1e-4 of the largest entry
      assert np.abs(g.reshape(r.shape) - r).max() <= 1e-4 * max(1.0, np.abs(r).max()), (name, flags)


@pytest.mark.parametrize("kind", ["any", "band", "one_far", "two_far"])
@pytest.mark.parametrize("mode,n_dir", [("TRWP", 4), ("TRWP", 16), ("ISGMR", 8)])
@pytest.mark.parametrize("L", [1, 2, 5, 63, 64, 65, 96, 128, 131, 191, 192, 193, 254, 256])
def test_several_wavefronts_per_chain(gpu, oracle, mode, n_dir, L, kind):
  """The reverse scan that puts four wavefronts on a chain (MPL_OPT_TEAM_SCANS; up to 64 labels one
  wavefront runs whatever the option): label counts at the edges of a lane's labels, chains of 1 to 13
  pixels (a block has six), argmin labels anywhere, in the register window or one step outside it with
  a shared far target (where the ways of scattering meet) or with two of them, all combinations of
  wanted gradients."""
  from mplayers_amd import _lib
  rng = np.random.default_rng(1000 * L + n_dir)
  B, H, W, n_iter, rho = 1, 7, 13, 2, (0.5 if mode == "TRWP" else 1.0)
  ctx = rng.random(L).astype(np.float32)
  ew = (0.1 + 0.9 * rng.random((n_dir, B, 1, H, W))).astype(np.float32)
  dcost = rng.standard_normal((B, 1, H, W, L)).astype(np.float32)
  imin = rng.integers(0, L, (n_iter, n_dir, B, 1, H, W, L))
  if kind != "any":
    reach = 3 if kind == "one_far" else 2
    near = np.clip(np.arange(L) + rng.integers(-reach, reach + 1, imin.shape), 0, L - 1)
    far = np.broadcast_to(imin[..., :1], imin.shape)
    if kind == "two_far":
      far = np.where(rng.random(imin.shape) < 0.5, far, imin[..., -1:])
    imin = np.where(rng.random(imin.shape) < 0.6, far, near)
  imin = imin.astype(np.uint8)
  inorm = rng.integers(0, L, (n_iter, n_dir, B, 1, H, W)).astype(np.uint8)
  ref = oracle.backward(mode, ctx.astype(np.float64), ew.astype(np.float64), dcost.astype(np.float64),
                        imin, inorm, rho, ctx2d=False)
  _lib.set_option(_lib.OPT_TEAM_SCANS, 2)
  try:
    for want_dctx, want_dedge in ((True, True), (False, False), (True, False), (False, True)):
      print("case", mode, n_dir, L, kind, want_dctx, want_dedge, flush=True)
      got = gpu.gpu_backward(mode, ctx, ew, dcost, imin, inorm, rho, flags=_lib.F_PACKED_OFF,
                             garbage_scratch=True, want_dctx=want_dctx, want_dedge=want_dedge)
      for name, g, r in zip(("dunary", "dcontext", "dedge"), got, ref):
        if g is not None:
          assert np.abs(g.reshape(r.shape) - r).max() <= 1e-4 * max(1.0, np.abs(r).max()), name
  finally:
    _lib.set_option(_lib.OPT_TEAM_SCANS, 1)


@pytest.mark.parametrize("L", [65, 96, 131, 192, 254, 256])
def test_kernels_of_a_call_differ_by_direction(gpu, oracle, L):
  """9 x 90 x 5 pixels: 810 rows of 5 pixels, which take one wavefront per chain and both walks of the
  pair in one launch, 45 columns of 90 pixels, which take four, and 846 diagonals; they hand their
  planes to each other."""
  rng = np.random.default_rng(L)
  B, H, W, n_dir, n_iter = 9, 90, 5, 8, 2
  ctx = rng.random(L).astype(np.float32)
  ew = (0.1 + 0.9 * rng.random((n_dir, B, 1, H, W))).astype(np.float32)
  dcost = rng.standard_normal((B, 1, H, W, L)).astype(np.float32)
  imin = rng.integers(0, L, (n_iter, n_dir, B, 1, H, W, L)).astype(np.uint8)
  inorm = rng.integers(0, L, (n_iter, n_dir, B, 1, H, W)).astype(np.uint8)
  print("case", L, flush=True)
  ref = oracle.backward("TRWP", ctx.astype(np.float64), ew.astype(np.float64), dcost.astype(np.float64),
                        imin, inorm, 0.5)
  got = gpu.gpu_backward("TRWP", ctx, ew, dcost, imin, inorm, 0.5, garbage_scratch=True)
  for name, g, r in zip(("dunary", "dcontext", "dedge"), got, ref):
    # the gradient bar of the GPU tests: 1e-4 of the largest entry
    assert np.abs(g.reshape(r.shape) - r).max() <= 1e-4 * max(1.0, np.abs(r).max()), name


@pytest.mark.parametrize("L", [65, 70, 131, 256])
def test_every_place_of_the_main_wavefront(gpu, oracle, L):
  """Which of the four wavefronts of a chain runs the recurrence changes with the workgroup's number
  over the number of compute units: 7 x 8 x 16 pixels give one ISGMR launch of 8 directions 980 chains,
  all four places on a device of 256."""
  import torch
  from mplayers_amd import _lib
  B, H, W, n_dir, n_iter = 7, 8, 16, 8, 2
  chains = sum(B * _lib.load().mpl_n_chains(d, H, W) for d in range(n_dir))
  assert chains > 3 * torch.cuda.get_device_properties(0).multi_processor_count
  rng = np.random.default_rng(L)
  ctx = rng.random(L).astype(np.float32)
  ew = (0.1 + 0.9 * rng.random((n_dir, B, 1, H, W))).astype(np.float32)
  dcost = rng.standard_normal((B, 1, H, W, L)).astype(np.float32)
  near = np.clip(np.arange(L) + rng.integers(-2, 3, (n_iter, n_dir, B, 1, H, W, L)), 0, L - 1)
  imin = np.where(rng.random(near.shape) < 0.6, near[..., :1], near).astype(np.uint8)
  inorm = rng.integers(0, L, (n_iter, n_dir, B, 1, H, W)).astype(np.uint8)
  ref = oracle.backward("ISGMR", ctx.astype(np.float64), ew.astype(np.float64), dcost.astype(np.float64),
                        imin, inorm, 1.0, ctx2d=False)
  print("case", L, chains, flush=True)
  _lib.set_option(_lib.OPT_TEAM_SCANS, 2)
  try:
    got = gpu.gpu_backward("ISGMR", ctx, ew, dcost, imin, inorm, 1.0, garbage_scratch=True)
  finally:
    _lib.set_option(_lib.OPT_TEAM_SCANS, 1)
  for name, g, r in zip(("dunary", "dcontext", "dedge"), got, ref):
    # the gradient bar of the GPU tests: 1e-4 of the largest entry
    assert np.abs(g.reshape(r.shape) - r).max() <= 1e-4 * max(1.0, np.abs(r).max()), name


@pytest.mark.parametrize("option", [0, 2])
@pytest.mark.parametrize("offset", [1, 2, 3])
@pytest.mark.parametrize("L", [70, 192, 256])
def test_table_gradient_of_a_long_chain(gpu, L, offset, option):
  """One entry of the table collects nearly every label of every pixel of a chain of 4000, all terms
  positive (rho = 0: every gradient is the upstream one; the label that the normalisation makes
  negative points elsewhere).  A scan sums them in at least a word per lane."""
  from mplayers_amd import _lib
  rng = np.random.default_rng(L + offset)
  n, n_dir = 4000, 2
  ctx = rng.random(L).astype(np.float32)
  ew = (0.1 + 0.9 * rng.random((n_dir, 1, 1, 1, n))).astype(np.float32)
  dcost = (0.5 + 0.5 * rng.random((1, 1, 1, n, L))).astype(np.float32)
  label = np.arange(L)
  target = np.where(label + offset < L, label + offset, label)
  norm = L // 2
  target[norm] = 0
  imin = np.broadcast_to(target, (1, n_dir, 1, 1, 1, n, L)).astype(np.uint8)
  inorm = np.full((1, n_dir, 1, 1, 1, n), norm, np.uint8)
  # pixels with an incoming edge: all but the first of either direction
  term = dcost[0, 0, 0].astype(np.float64)[:, (target == label + offset) & (label != norm)].sum(-1)
  exact = (ew[0, 0, 0, 0, 1:] * term[1:]).sum() + (ew[1, 0, 0, 0, :-1] * term[:-1]).sum()
  print("case", L, offset, option, flush=True)
  _lib.set_option(_lib.OPT_TEAM_SCANS, option)
  try:
    got = gpu.gpu_backward("ISGMR", ctx, ew, dcost, imin, inorm, 0.0)[1]
  finally:
    _lib.set_option(_lib.OPT_TEAM_SCANS, 1)
  # m positive additions into one word round to a relative error of about sqrt(m) * 2^-24 (each rounds
  # either way); the 64 words of a wavefront average to an eighth of that.  One wavefront adds its
  # lane's labels first (m = n), each of three helpers every label of a lane (m = n / 3 per label).  A
  # word for all labels would see m = n L.
  m = n * (-(-L // 64)) / (3 if option else 1)
  assert abs(got[offset] - exact) <= m ** 0.5 * 2.0 ** -24 * exact, (got[offset] - exact) / exact


@pytest.mark.parametrize("option", [0, 2])
@pytest.mark.parametrize("L", [128, 192, 256])
def test_two_targets_share_the_labels(gpu, L, option):
  """Half of the labels of every pixel point at one label, half at another, as either side of a slope
  under a linear table.  Chains of two pixels (and the label that the normalisation changes points
  elsewhere), so a gradient is one sum of random terms and its error shows how it was formed."""
  from mplayers_amd import _lib
  rng = np.random.default_rng(L)
  n_dir, H, W = 2, 400, 2
  ctx = rng.random(L).astype(np.float32)
  dcost = rng.standard_normal((1, 1, H, W, L)).astype(np.float32)
  low, high, norm = L // 4, 3 * L // 4, L // 2
  target = np.where(np.arange(L) < norm, low, high)
  target[norm] = norm
  imin = np.broadcast_to(target, (1, n_dir, 1, 1, H, W, L)).astype(np.uint8)
  inorm = np.full((1, n_dir, 1, 1, H, W), norm, np.uint8)
  print("case", L, option, flush=True)
  _lib.set_option(_lib.OPT_TEAM_SCANS, option)
  try:
    got = gpu.gpu_backward("ISGMR", ctx, None, dcost, imin, inorm, 1.0, want_dctx=False, want_dedge=False)[0]
  finally:
    _lib.set_option(_lib.OPT_TEAM_SCANS, 1)
  d = dcost[0, 0].astype(np.float64)
  for label, share in ((low, np.arange(L) < norm), (high, np.arange(L) > norm)):
    sums = d[:, :, share].sum(-1)
    exact = d[:, :, label] + sums[:, ::-1]  # a pixel's sum goes to its neighbour
    err = np.linalg.norm(got[0, 0, :, :, label] - exact) / np.linalg.norm(exact) * 2 ** 24
    # an addition rounds its sum by some 0.42 * 2^-24 in the root mean square.  In a tree over the lanes
    # every level's sums have the variance of the whole: nine levels (six of lanes, up to two in a lane, the
    # upstream gradient) come to 0.42 * 3 = 1.26.  One after the other, 63 to 127 additions of growing
    # sums come to 0.42 sqrt(n / 2), 2.4 to 3.4
    assert err <= 1.75, err


@pytest.mark.parametrize("value", [np.inf, -np.inf, np.nan])
@pytest.mark.parametrize("mode,L", [("TRWP", 5), ("ISGMR", 21), ("TRWP", 40), ("TRWP", 70), ("ISGMR", 96),
                                    ("TRWP", 192), ("ISGMR", 254)])
def test_gradients_that_are_not_finite(gpu, oracle, mode, L, value):
  """An upstream gradient that is not finite shows in every entry that it reaches and in no other,
  whichever kernel scans.  (The normalisation gives one label of the pixel the other sign, so a sum over
  labels may be NaN, the table's gradient among them.)"""
  from mplayers_amd import _lib
  rng = np.random.default_rng(L)
  B, H, W, n_dir, n_iter, rho = 1, 6, 11, 4, 1, (0.5 if mode == "TRWP" else 1.0)
  routes = [(0, 0), (2, 0)] if L > 64 else [(0, _lib.F_PACKED_OFF)]
  if L <= 32:
    routes.append((0, _lib.F_PACKED_ALWAYS))
  for k in range(8):
    ctx = (np.triu(rng.random((L, L)), 1) if L == 21 else rng.random(L)).astype(np.float32)
    ew = (0.1 + 0.9 * rng.random((n_dir, B, 1, H, W))).astype(np.float32)
    dcost = rng.standard_normal((B, 1, H, W, L)).astype(np.float32)
    dcost[0, 0, rng.integers(H), rng.integers(W), rng.integers(L)] = value
    imin = rng.integers(0, L, (n_iter, n_dir, B, 1, H, W, L))
    near = np.clip(np.arange(L) + rng.integers(-2, 3, imin.shape), 0, L - 1)
    imin = np.where(rng.random(imin.shape) < (0.6 if k % 2 else 1.0), imin if k % 4 == 0 else imin[..., :1], near)
    imin = imin.astype(np.uint8)
    inorm = rng.integers(0, L, (n_iter, n_dir, B, 1, H, W)).astype(np.uint8)
    ref = oracle.backward(mode, ctx.astype(np.float64), ew.astype(np.float64), dcost.astype(np.float64),
                          imin, inorm, rho)
    for option, flags in routes:
      print("case", mode, L, value, k, option, flags, flush=True)
      _lib.set_option(_lib.OPT_TEAM_SCANS, option)
      try:
        got = gpu.gpu_backward(mode, ctx, ew, dcost, imin, inorm, rho, flags=flags, garbage_scratch=True)
      finally:
        _lib.set_option(_lib.OPT_TEAM_SCANS, 1)
      for name, g, r in zip(("dunary", "dcontext", "dedge"), got, ref):
        assert np.array_equal(np.isfinite(g), np.isfinite(r.reshape(g.shape))), (name, option, flags)
