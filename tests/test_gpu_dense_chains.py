"""Dense 1-D tables of more than 128 labels in launches of more chains than the chip has units, where four wavefronts
scan and serve a chain by themselves, against one wavefront per chain: the same bits, on chains around their block of
eight pixels."""
import numpy as np
import pytest

from tests.test_gpu_forward_team import _problem, _run, _same

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("L", [129, 160, 161, 192])
@pytest.mark.parametrize("W", [1, 2, 7, 8, 9, 16, 17])
@pytest.mark.parametrize("training", [True, False])
def test_more_chains_than_units(gpu, L, W, training):
  from mplayers_amd import _lib
  import torch
  B = 3 + torch.cuda.get_device_properties(0).multi_processor_count // 2
  problem = _problem(4, B, 2, W, L, "random", W, W == 9)
  print("case", L, W, training, B, flush=True)
  one = _run(gpu, 0, *problem, 4, 2, training, _lib.F_PACKED_OFF)
  four = _run(gpu, 2, *problem, 4, 2, training, _lib.F_PACKED_OFF | _lib.F_DENSE_TABLE)
  _same(four, one, training)


@pytest.mark.parametrize("L", [17, 33, 64, 96, 128, 160, 192])
@pytest.mark.parametrize("W", [2, 3, 4, 5, 7, 8, 9, 11, 12, 13])
@pytest.mark.parametrize("training", [True, False])
def test_blocks_of_the_served_scan(gpu, L, W, training):
  """Launches of few chains, whose scan has servers: chains around its block of four pixels and its two sets of slots, with
  one launch per pair of directions and with two."""
  from mplayers_amd import _lib
  problem = _problem(4, 1, 3, W, L, "random", W, W == 9)
  for more in (0, _lib.F_FUSED_PAIRS_OFF):
    print("case", L, W, training, more, flush=True)
    one = _run(gpu, 0, *problem, 4, 2, training, _lib.F_PACKED_OFF | more)
    four = _run(gpu, 2, *problem, 4, 2, training, _lib.F_PACKED_OFF | _lib.F_DENSE_TABLE | more)
    _same(four, one, training)
