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


@pytest.mark.parametrize("L,tile,H,W", [(3, 128, 512, 513), (21, 128, 513, 513), (32, 128, 512, 513), (32, 128, 513, 513),
                                        (33, 64, 384, 342), (96, 64, 384, 342), (96, 64, 363, 363), (128, 64, 363, 363),
                                        (129, 32, 211, 317), (256, 32, 192, 346)])
@pytest.mark.parametrize("n_dir", [2, 4])
def test_every_tile(gpu, L, tile, H, W, n_dir):
  """Images large enough for each tile of pixels, of whole lines and of odd sizes, whose last tile is partial, and for the
  regrouping of workgroups, with the last round of groups incomplete."""
  from mplayers_amd import _lib, ops
  cus = torch.cuda.get_device_properties(0).multi_processor_count
  tiles = -(-H * W // tile)
  assert tiles >= 2 * 4 * cus and tiles % 64 != 0 and tiles > 64
  gen = torch.Generator(device=gpu.DEV).manual_seed(L + H)
  unary = torch.rand(1, 1, H, W, L, generator=gen, device=gpu.DEV)
  ew = torch.rand(n_dir, 1, 1, H, W, generator=gen, device=gpu.DEV)
  ctx = torch.triu(torch.rand(L, L, generator=gen, device=gpu.DEV), 1) if L == 21 else \
      0.1 * torch.arange(L, device=gpu.DEV).clamp(max=3)
  none = torch.empty(0, dtype=torch.uint8)
  out = []
  for flags in (0, _lib.F_COST_LABELS_FIRST):
    msg, scratch = torch.zeros(n_dir, 1, 1, H, W, L, device=gpu.DEV), torch.empty_like(unary)
    cost = torch.full((1, 1, L, H, W) if flags else (1, 1, H, W, L), float("nan"), device=gpu.DEV)
    print("case", L, H, W, n_dir, flags, flush=True)
    ops.TRWP.forward(0.5, 1, 0, unary, ctx, ew, msg, cost, none, none, scratch, none, flags=flags)
    out.append(cost)
  assert torch.equal(out[0].permute(0, 1, 4, 2, 3), out[1])


@pytest.mark.parametrize("L,H,W", [(1, 33, 35), (2, 33, 35), (3, 21, 23), (5, 9, 7), (21, 65, 65), (33, 9, 11), (97, 63, 77),
                                   (191, 46, 65), (255, 23, 29)])
@pytest.mark.parametrize("B,n_dir", [(4, 4), (4, 6), (2, 8), (1, 4)])
def test_fours_across_tiles_and_images(gpu, L, H, W, B, n_dir):
  """Images of a number of elements that four does not divide, in batches that make the planes whole fours, with tiles of
  32, 16 and 8 pixels: fours that begin before the tile, or end after it."""
  from mplayers_amd import _lib, ops
  gen = torch.Generator(device=gpu.DEV).manual_seed(L + B)
  unary = torch.rand(B, 1, H, W, L, generator=gen, device=gpu.DEV)
  ew = torch.rand(n_dir, B, 1, H, W, generator=gen, device=gpu.DEV)
  ctx = torch.triu(torch.rand(L, L, generator=gen, device=gpu.DEV), 1) if L == 21 else \
      0.1 * torch.arange(L, device=gpu.DEV).clamp(max=3)
  none = torch.empty(0, dtype=torch.uint8)
  for min_a_dir in (0, 1):
    out = []
    for flags in (0, _lib.F_COST_LABELS_FIRST):
      msg, scratch = torch.zeros(n_dir, B, 1, H, W, L, device=gpu.DEV), torch.empty_like(unary)
      cost = torch.full((B, 1, L, H, W) if flags else (B, 1, H, W, L), float("nan"), device=gpu.DEV)
      print("case", L, H, W, B, n_dir, min_a_dir, flags, flush=True)
      ops.TRWP.forward(0.5, 1, min_a_dir, unary, ctx, ew, msg, cost, none, none, scratch, none, flags=flags)
      out.append(cost)
    assert torch.equal(out[0].permute(0, 1, 4, 2, 3), out[1])
