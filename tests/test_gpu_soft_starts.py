"""Soft-weighted TRWP with MPL_F_CHAIN_STARTS: buffers nobody cleared, every direction, images thinner than a step."""
import argparse

import pytest
import torch

from mplayers_amd import _lib

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("L,B,H,W,n_dir", [(21, 2, 9, 11, 4), (16, 1, 6, 5, 16), (40, 1, 5, 7, 8), (70, 1, 4, 3, 16),
                                           (21, 3, 1, 1, 16), (21, 1, 1, 13, 8), (3, 2, 7, 2, 16)])
def test_starts_are_zero_and_the_rest_is_written(gpu, L, B, H, W, n_dir):
  from mplayers_amd import ops
  n_iter = 2
  gen = torch.Generator(device=gpu.DEV).manual_seed(H * W + L)
  rand = lambda *s: torch.rand(*s, generator=gen, device=gpu.DEV)
  unary, ew = rand(B, 1, H, W, L), rand(n_dir, B, 1, H, W)
  ctx = torch.triu(rand(L, L), 1) if L == 21 else torch.cumsum(rand(L), 0)
  out = {}
  for flags, fill in ((0, 0.0), (_lib.F_CHAIN_STARTS, float("nan"))):
    msg = torch.zeros(n_dir, B, 1, H, W, L, device=gpu.DEV)
    duals = torch.full((n_iter, n_dir, B, 1, H, W, L, L), fill, device=gpu.DEV)
    norm = torch.full((n_iter, n_dir, B, 1, H, W), 0 if flags == 0 else 255, dtype=torch.uint8, device=gpu.DEV)
    cost = torch.empty_like(unary)
    print("case", L, B, H, W, n_dir, flags, flush=True)
    ops.TRWP_hard_soft.forward_soft(0.5, n_iter, unary, ctx, ew, msg, duals, norm, cost, torch.empty_like(unary),
                                    torch.empty(0, dtype=torch.uint8), flags=flags)
    out[flags] = duals, norm, cost, msg
  for a, b in zip(out[0], out[_lib.F_CHAIN_STARTS]):
    assert torch.equal(a, b)


def test_gradient_of_the_duals_alone(gpu):
  """A loss that does not touch the costs: their gradient is zero, as autograd fills it in, and so are the others."""
  from mplayers_amd.MP_module_hard_soft import TRWPFunction
  args = argparse.Namespace(rho=0.5, mpnet_max_iter=2, mpnet_n_dirs=4, mpnet_enable_soft=True, training=True,
                            enable_saving_label=False, msg_norm_index=None, n_classes=21, enable_seg=True)
  unary = torch.rand(1, 1, 6, 7, 21, device=gpu.DEV, requires_grad=True)
  table = torch.rand(21, 21, device=gpu.DEV, requires_grad=True)
  weights = torch.rand(4, 1, 1, 6, 7, device=gpu.DEV, requires_grad=True)
  _, _, duals, _ = TRWPFunction.apply(unary, table, weights, args)
  duals.sum().backward()
  for t in (unary, table, weights):
    assert float(t.grad.abs().max()) == 0.0
