"""cost_final with the labels first (MPL_F_COST_LABELS_FIRST): the bits of the other layout, turned over."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("L", [1, 3, 16, 21, 32, 33, 64, 96, 128, 129, 192, 255, 256])
@pytest.mark.parametrize("B,H,W,n_dir", [(1, 1, 1, 4), (2, 5, 7, 8), (3, 8, 16, 4), (1, 32, 33, 16), (2, 3, 43, 2), (2, 3, 43, 16), (2, 5, 7, 6), (1, 3, 43, 12)])
def test_costs_turned_over(gpu, L, B, H, W, n_dir):
  from mplayers_amd import _lib, ops
  gen = torch.Generator(device=gpu.DEV).manual_seed(L + H)
  rand = lambda *s: torch.rand(*s, generator=gen, device=gpu.DEV)
  unary, ew = rand(B, 1, H, W, L), rand(n_dir, B, 1, H, W)
  ctx = torch.triu(rand(L, L), 1) if L == 21 else 0.1 * torch.arange(L, device=gpu.DEV).clamp(max=3)
  none = torch.empty(0, dtype=torch.uint8)
  for what in ("TRWP", "min_a_dir", "labels", "ISGMR", "SGM", "soft"):
    out = []
    for flags in (0, _lib.F_COST_LABELS_FIRST):
      msg, tmp = torch.zeros(n_dir, B, 1, H, W, L, device=gpu.DEV), torch.zeros(n_dir, B, 1, H, W, L, device=gpu.DEV)
      cost = torch.full((B, 1, L, H, W) if flags else (B, 1, H, W, L), float("nan"), device=gpu.DEV)
      scratch = torch.empty_like(unary)
      label = torch.zeros(2, B, 1, H, W, dtype=torch.uint8, device=gpu.DEV) if what == "labels" else none
      print("case", L, B, H, W, n_dir, what, flags, flush=True)
      if what == "soft":
        ops.TRWP_hard_soft.forward_soft(0.5, 2, unary, ctx, ew, msg, torch.empty(0), none, cost, scratch, label, flags=flags)
      elif what in ("ISGMR", "SGM"):
        ops.ISGMR.forward(int(what == "SGM"), 1.0, 1 if what == "SGM" else 2, 0, unary, ctx, ew, msg, cost, none, none, scratch,
                          tmp, label, flags=flags)
      else:
        ops.TRWP.forward(0.5, 2, int(what == "min_a_dir"), unary, ctx, ew, msg, cost, none, none, scratch, label, flags=flags)
      out.append((cost, msg, label))
    assert torch.equal(out[0][0].permute(0, 1, 4, 2, 3), out[1][0]), what
    assert torch.equal(out[0][1], out[1][1]) and torch.equal(out[0][2], out[1][2]), what
