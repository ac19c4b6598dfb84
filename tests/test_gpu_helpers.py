"""Scans with four wavefronts per chain, with six helpers (few chains) and with three (many): the same operations on a
pixel, so the same bits, on chains around a block of six pixels."""
import numpy as np
import pytest

from tests.test_gpu_forward_team import _problem

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("L,table", [(40, "potts"), (96, "random"), (127, "potts"), (192, "linear"), (256, "potts")])
@pytest.mark.parametrize("W", [1, 2, 5, 6, 7, 12, 13, 26])
def test_six_and_three_helpers(gpu, L, table, W):
  import torch
  from mplayers_amd import _lib
  cus = torch.cuda.get_device_properties(0).multi_processor_count
  n_dir, n_iter, H = 4, 2, 13
  B = 3 * cus // H + 1  # (more rows than three chains per unit)
  unary, ctx, ew = _problem(n_dir, 1, H, W, L, table, W)
  dcost = np.random.default_rng(W).standard_normal(unary.shape).astype(np.float32)
  out = []
  _lib.set_option(_lib.OPT_TEAM_SCANS, 2)
  try:
    for n in (1, B):
      print("case", L, table, W, n, flush=True)
      f = gpu.gpu_forward("TRWP", np.repeat(unary, n, 0), ctx, np.repeat(ew, n, 1), n_dir, n_iter, 0.5)
      b = gpu.gpu_backward("TRWP", ctx, np.repeat(ew, n, 1), np.repeat(dcost, n, 0), f["msg_min_index"],
                           f["msg_norm_index"], 0.5)
      out.append((f, b))
  finally:
    _lib.set_option(_lib.OPT_TEAM_SCANS, 1)
  (f1, b1), (fn, bn) = out
  for k, axis in (("msg", 1), ("cost_final", 0), ("msg_min_index", 2), ("msg_norm_index", 2)):
    for i in (0, B - 1):
      assert np.array_equal(f1[k].take(0, axis), fn[k].take(i, axis)), k
  for i in (0, B - 1):
    assert np.array_equal(b1[0][0], bn[0][i]) and np.array_equal(b1[2][:, 0], bn[2][:, i])
  # B times the same sums in another order
  assert np.abs(b1[1] * B - bn[1]).max() <= 1e-4 * max(1e-30, float(np.abs(bn[1]).max()))
