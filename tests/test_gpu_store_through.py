"""ISGMR launches large enough to store through the L2 (store_through): a batch that is, against its images one by one,
which are not: the same bits."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("L,side", [(64, 128), (128, 91), (192, 74), (256, 64)])
@pytest.mark.parametrize("n_dir", [4, 8])
@pytest.mark.parametrize("train", [False, True])
def test_batch_equals_its_images(gpu, L, side, n_dir, train):
  from mplayers_amd import ops
  n_iter, B = 2, -(-(132 << 20) // (n_dir * side * side * L * 4))
  assert (B - 1) * n_dir * side * side * L * 4 < 132 << 20 and B > 2
  gen = torch.Generator(device=gpu.DEV).manual_seed(L + n_dir)
  unary = torch.rand(B, 1, side, side, L, generator=gen, device=gpu.DEV)
  ew = torch.rand(n_dir, B, 1, side, side, generator=gen, device=gpu.DEV)
  ctx = 0.1 * torch.arange(L, device=gpu.DEV, dtype=torch.float32).clamp(max=5) ** 2

  def run(first, count):
    u, w = unary[first:first + count].contiguous(), ew[:, first:first + count].contiguous()
    msg = torch.full((n_dir,) + tuple(u.shape), float("nan"), device=gpu.DEV)
    cost, tmp, scratch = torch.empty_like(u), torch.full_like(msg, float("nan")), torch.empty_like(u)
    none = torch.empty(0, dtype=torch.uint8)
    imin = torch.zeros((n_iter,) + tuple(msg.shape), dtype=torch.uint8, device=gpu.DEV) if train else none
    inorm = torch.zeros((n_iter,) + tuple(msg.shape[:-1]), dtype=torch.uint8, device=gpu.DEV) if train else none
    print("case", L, side, n_dir, train, first, count, flush=True)
    ops.ISGMR.forward(0, 1.0, n_iter, 0, u, ctx, w, msg, cost, imin, inorm, scratch, tmp, none, msg_uninit=True)
    return msg, cost, imin, inorm
  whole = run(0, B)
  for b in (0, B - 1):
    for a, c, axis in zip(whole, run(b, 1), (1, 0, 2, 2)):
      assert torch.equal(a.narrow(axis, b, 1) if a.numel() else a, c)


@pytest.mark.parametrize("L,side", [(60, 120), (64, 128), (96, 91), (128, 74)])
@pytest.mark.parametrize("train", [False, True])
def test_trwp_image_equals_its_batch(gpu, L, side, train):
  """TRWP with four wavefronts per chain, the other way round: an image's messages fit the last-level cache, its batch's
  do not (kCachedMessages)."""
  from mplayers_amd import _lib, ops
  n_dir, n_iter = 4, 2
  B = (208 << 20) // (n_dir * side * side * L * 4) + 1
  assert B > 2
  gen = torch.Generator(device=gpu.DEV).manual_seed(L)
  unary = torch.rand(B, 1, side, side, L, generator=gen, device=gpu.DEV)
  ew = torch.rand(n_dir, B, 1, side, side, generator=gen, device=gpu.DEV)
  ctx = 0.3 * torch.arange(L, device=gpu.DEV, dtype=torch.float32).clamp(max=3)

  def run(first, count):
    u, w = unary[first:first + count].contiguous(), ew[:, first:first + count].contiguous()
    msg = torch.full((n_dir,) + tuple(u.shape), float("nan"), device=gpu.DEV)
    cost, scratch = torch.empty_like(u), torch.empty_like(u)
    none = torch.empty(0, dtype=torch.uint8)
    imin = torch.zeros((n_iter,) + tuple(msg.shape), dtype=torch.uint8, device=gpu.DEV) if train else none
    inorm = torch.zeros((n_iter,) + tuple(msg.shape[:-1]), dtype=torch.uint8, device=gpu.DEV) if train else none
    print("case", L, side, train, first, count, flush=True)
    ops.TRWP.forward(0.5, n_iter, 0, u, ctx, w, msg, cost, imin, inorm, scratch, none, msg_uninit=True)
    return msg, cost, imin, inorm
  _lib.set_option(_lib.OPT_TEAM_SCANS, 2)
  try:
    whole = run(0, B)
    for b in (0, B - 1):
      for a, c, axis in zip(whole, run(b, 1), (1, 0, 2, 2)):
        assert torch.equal(a.narrow(axis, b, 1) if a.numel() else a, c)
  finally:
    _lib.set_option(_lib.OPT_TEAM_SCANS, 1)
