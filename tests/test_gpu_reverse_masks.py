"""Reverse scans with four wavefronts per chain: launches of few chains multiply with masks, which do not switch off what
is not finite, and walk such blocks by the codes again; launches of many chains have the codes only.  The same bits."""
import numpy as np
import pytest

from tests.test_gpu_forward_team import _problem

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("mode", ["TRWP", "ISGMR"])
@pytest.mark.parametrize("L,table", [(65, "potts"), (96, "random"), (127, "linear"), (192, "potts"), (191, "random")])
@pytest.mark.parametrize("value", [None, np.inf, -np.inf, np.nan, 3e38])
def test_masks_and_codes(gpu, mode, L, table, value):
  import torch
  from mplayers_amd import _lib
  cus = torch.cuda.get_device_properties(0).multi_processor_count
  n_dir, n_iter, H, W, rho = 4, 2, 11, 20, 0.5 if mode == "TRWP" else 1.0
  B = 3 * cus // H + 1  # (more rows than three chains per unit)
  unary, ctx, ew = _problem(n_dir, 1, H, W, L, table, L)
  dcost = np.random.default_rng(L).standard_normal(unary.shape).astype(np.float32)
  if value is not None:  # the label the others point at most, a neighbour of its target, and the last one
    for y, x, l in ((3, 7, 0), (5, 6, L // 2), (8, 13, L - 1)):
      dcost[0, 0, y, x, l] = value
  out = []
  _lib.set_option(_lib.OPT_TEAM_SCANS, 2)
  try:
    for n in (1, B):
      print("case", mode, L, table, value, n, flush=True)
      f = gpu.gpu_forward(mode, np.repeat(unary, n, 0), ctx, np.repeat(ew, n, 1), n_dir, n_iter, rho)
      out.append(gpu.gpu_backward(mode, ctx, np.repeat(ew, n, 1), np.repeat(dcost, n, 0), f["msg_min_index"],
                                  f["msg_norm_index"], rho))
  finally:
    _lib.set_option(_lib.OPT_TEAM_SCANS, 1)
  (few, many) = out
  for i in (0, B - 1):
    assert np.array_equal(few[0][0], many[0][i], equal_nan=True)
    assert np.array_equal(few[2][:, 0], many[2][:, i], equal_nan=True)
