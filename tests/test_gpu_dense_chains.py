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
