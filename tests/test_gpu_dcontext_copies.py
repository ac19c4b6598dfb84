"""dcontext through tables that the chains of a launch take turns on (MPL_F_DCONTEXT_COPIES): every reverse scan, on
both sides of the number of chains from which the library wants them."""
import numpy as np
import pytest
import torch

from mplayers_amd import _lib


def test_copies_on_the_host():
  """Asked for from a number of chains on; a refused shape is refused here too, and so is a call without tables."""
  assert _lib.dcontext_copies(_lib.Shape(4, 4, 129, 129, 21, 1), 5) == 8
  assert _lib.dcontext_copies(_lib.Shape(2, 1, 2048, 5, 40, 0), 1) == 8
  assert _lib.dcontext_copies(_lib.Shape(2, 1, 2047, 5, 40, 0), 1) == 0
  with pytest.raises(RuntimeError):
    _lib.dcontext_copies(_lib.Shape(3, 1, 5, 5, 40, 0), 1)
  shape, one = _lib.Shape(2, 1, 2048, 5, 40, 0), 1 << 20  # (an address nobody reads: the call is refused before)
  lib = _lib.load()
  assert lib.mpl_trwp_backward(shape, _lib.F_DCONTEXT_COPIES, 0.5, 1, one, one, one, one, one, one, one, one, one, None,
                               None) != 0
  assert b"DCONTEXT_COPIES" in lib.mpl_last_error()


@pytest.mark.gpu
@pytest.mark.parametrize("mode,L,B,H,W,n_dir,n_iter", [
    ("TRWP", 21, 16, 17, 19, 4, 4), ("ISGMR", 21, 40, 11, 17, 4, 2),    # four wavefronts, packed scans
    ("TRWP", 40, 24, 13, 17, 8, 2), ("ISGMR", 12, 24, 13, 17, 8, 2),    # one wavefront per chain
    ("TRWP", 96, 12, 19, 17, 8, 3), ("ISGMR", 150, 12, 19, 17, 8, 3),   # four wavefronts, one
    ("TRWP", 21, 1, 7, 9, 4, 2), ("ISGMR", 70, 1, 9, 7, 4, 2)])         # too few chains
def test_hard_scans(gpu, oracle, mode, L, B, H, W, n_dir, n_iter):
  from mplayers_amd import ops
  rng = np.random.default_rng(L + B)
  ctx = np.triu(rng.random((L, L)), 1) if L == 21 else np.cumsum(rng.random(L))
  ew = rng.random((n_dir, B, 1, H, W)) - 0.2
  dcost = rng.standard_normal((B, 1, H, W, L))
  imin = rng.integers(0, L, (n_iter, n_dir, B, 1, H, W, L)).astype(np.uint8)
  inorm = rng.integers(0, L, (n_iter, n_dir, B, 1, H, W)).astype(np.uint8)
  rho = 0.5 if mode == "TRWP" else 1.0
  f32 = [np.float32(x) for x in (ctx, ew, dcost)]
  ref = oracle.backward(mode, *[np.float64(x) for x in f32], imin, inorm, rho)
  copies = _lib.dcontext_copies(_lib.Shape(n_dir, B, H, W, L, int(L == 21)), n_iter)
  assert (copies > 0) == (B > 1)
  t = [gpu._t(x) for x in f32] + [gpu._t(x, torch.uint8) for x in (imin, inorm)]
  new = lambda *s: torch.full(s, float("nan"), device=gpu.DEV)
  dunary, dedge = new(*dcost.shape), torch.zeros_like(t[1])
  dctx = new(*ctx.shape) if copies else torch.zeros_like(t[0])  # overwritten, or added to
  tables = torch.zeros((copies,) + ctx.shape, device=gpu.DEV)
  planes = [new(n_dir, *dcost.shape) for _ in range(2)]
  print("case", mode, L, B, H, W, n_dir, n_iter, copies, flush=True)
  if mode == "TRWP":
    ops.TRWP.backward(rho, t[0], t[1], t[2], t[3], t[4], dunary, dctx, dedge, planes[0], tables,
                      flags=_lib.F_DCONTEXT_COPIES)
  else:
    ops.ISGMR.backward(0, rho, t[0], t[1], t[2], t[3], t[4], dunary, dctx, dedge, planes[0], tables, planes[1],
                       flags=_lib.F_DCONTEXT_COPIES)
  for a, b, what in zip((dunary, dctx, dedge), ref, ("dunary", "dcontext", "dedge_weights")):
    # sums of at most some thousands of products: 1e-4 of the largest entry, as everywhere
    assert np.abs(a.cpu().numpy() - b).max() <= 1e-4 * max(1.0, float(np.abs(b).max())), what
  if copies:
    with pytest.raises(RuntimeError):
      ops.TRWP.backward(rho, t[0], t[1], t[2], t[3], t[4], dunary, dctx, dedge, planes[0], tables[1:],
                        flags=_lib.F_DCONTEXT_COPIES)


@pytest.mark.gpu
@pytest.mark.parametrize("L,B,H,W", [(21, 24, 13, 17), (12, 24, 13, 17), (40, 24, 13, 17), (70, 24, 13, 17)])
def test_soft_scans(gpu, L, B, H, W):
  from mplayers_amd import ops
  n_dir, n_iter = 4, 3
  gen = torch.Generator(device=gpu.DEV).manual_seed(L)
  rand = lambda *s: torch.rand(*s, generator=gen, device=gpu.DEV)
  ctx = torch.triu(rand(L, L), 1) if L == 21 else torch.cumsum(rand(L), 0)
  ew, dcost = rand(n_dir, B, 1, H, W), rand(B, 1, H, W, L) - 0.3
  duals = 4 * rand(n_iter, n_dir, B, 1, H, W, L, L)
  inorm = torch.randint(0, L, (n_iter, n_dir, B, 1, H, W), generator=gen, device=gpu.DEV).to(torch.uint8)
  out = {}
  for flags in (0, _lib.F_DCONTEXT_COPIES):
    copies = _lib.dcontext_copies(_lib.Shape(n_dir, B, H, W, L, int(L == 21)), n_iter) if flags else 0
    assert (copies > 0) == (flags != 0)
    dunary, dedge = torch.empty_like(dcost), torch.zeros_like(ew)
    dctx = torch.full_like(ctx, float("nan")) if flags else torch.zeros_like(ctx)
    tables = torch.zeros((copies,) + tuple(ctx.shape), device=gpu.DEV)
    print("case", L, B, H, W, flags, flush=True)
    ops.TRWP_hard_soft.backward_soft(0.5, dcost, ctx, ew, duals, inorm, dunary, dctx, dedge,
                                     rand(n_dir, B, 1, H, W, L), tables, flags=flags)
    out[flags] = dunary, dedge, dctx
  for a, b in zip(out[0][:2], out[_lib.F_DCONTEXT_COPIES][:2]):
    assert torch.equal(a, b)
  # the same parts, one per chain, summed in another order
  a, b = out[0][2], out[_lib.F_DCONTEXT_COPIES][2]
  assert float((a - b).abs().max()) <= 1e-4 * float(a.abs().max())
