"""The reverse scans of 21 labels, soft-weighted and hard, with six helpers (few chains) and with three: the same
operations on a pixel, so the same bits, on chains around a block of either (12 and 6 pixels)."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("W", [1, 2, 5, 6, 7, 11, 12, 13, 14, 24, 25, 37])
@pytest.mark.parametrize("soft", [True, False])
def test_six_and_three_helpers(gpu, W, soft):
  from mplayers_amd import ops
  L, H, n_dir, n_iter = 21, 13, 4, 2
  cus = torch.cuda.get_device_properties(0).multi_processor_count
  n = 3 * cus // max(H, W)  # (more than three chains per unit: one wavefront per chain)
  assert max(H, W) <= cus and 2 * cus < n * max(H, W) and cus < n * H
  gen = torch.Generator(device=gpu.DEV).manual_seed(W)
  rand = lambda *s: torch.rand(*s, generator=gen, device=gpu.DEV)
  ctx, ew, dcost = torch.triu(rand(L, L), 1), rand(n_dir, 1, 1, H, W), rand(1, 1, H, W, L) - 0.4
  duals = 5 * rand(n_iter, n_dir, 1, 1, H, W, L, L)
  imin = torch.randint(0, L, (n_iter, n_dir, 1, 1, H, W, L), generator=gen, device=gpu.DEV).to(torch.uint8)
  inorm = torch.randint(0, L, (n_iter, n_dir, 1, 1, H, W), generator=gen, device=gpu.DEV).to(torch.uint8)
  out = []
  for B in (1, n):
    rep = lambda t, d: t.repeat_interleave(B, d).contiguous()
    dunary, dedge, dctx = torch.empty(B, 1, H, W, L, device=gpu.DEV), torch.zeros(n_dir, B, 1, H, W, device=gpu.DEV), \
        torch.zeros(L, L, device=gpu.DEV)
    print("case", W, B, soft, flush=True)
    if not soft:
      ops.TRWP.backward(0.5, ctx, rep(ew, 1), rep(dcost, 0), rep(imin, 2), rep(inorm, 2), dunary, dctx, dedge,
                        torch.empty(n_dir, B, 1, H, W, L, device=gpu.DEV), torch.empty(0, device=gpu.DEV))
      out.append((dunary, dedge, dctx))
      continue
    ops.TRWP_hard_soft.backward_soft(0.5, rep(dcost, 0), ctx, rep(ew, 1), rep(duals, 2), rep(inorm, 2), dunary, dctx, dedge,
                                     torch.empty(n_dir, B, 1, H, W, L, device=gpu.DEV), torch.empty(0, device=gpu.DEV))
    out.append((dunary, dedge, dctx))
  for b in (0, n // 2, n - 1):
    assert torch.equal(out[0][0][0], out[1][0][b])
    assert torch.equal(out[0][1][:, 0], out[1][1][:, b])
  # n times the same sums in another order
  a, b = out[0][2] * n, out[1][2]
  assert float((a - b).abs().max()) <= 1e-4 * max(1e-30, float(a.abs().max()))
