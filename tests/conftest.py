import os
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
if ROOT not in sys.path:
  sys.path.insert(0, ROOT)


def pytest_configure(config):
  config.addinivalue_line("markers", "gpu: needs a real MI355X (run with -m gpu on the GPU box)")


@pytest.fixture(scope="session")
def oracle():
  from oracle import mp_oracle
  mp_oracle.build()
  return mp_oracle


@pytest.fixture(scope="session")
def gpu():
  """Helpers of the GPU parity tests; fails (not skips) without a GPU or without the HIP library."""
  import torch
  assert torch.cuda.is_available(), "these tests need the MI355X"
  from mplayers_amd import _lib
  _lib.load()
  from tests import _gpu_util
  return _gpu_util


@pytest.fixture(params=[1, 0], ids=["by_launch", "one_wavefront"])
def reverse_scans(request, gpu):
  """Runs a test twice: with the reverse scans the launch rule takes (images as small as those of the
  tests put four wavefronts on a chain from 65 labels on) and with one wavefront per chain, which
  larger launches take."""
  from mplayers_amd import _lib
  _lib.set_option(_lib.OPT_TEAM_SCANS, request.param)
  yield request.param
  _lib.set_option(_lib.OPT_TEAM_SCANS, 1)
