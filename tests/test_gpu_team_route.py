"""Which launches of the reverse scans put four wavefronts on a chain.

The two kernels sum in different orders, so the bits of dunary show which one ran: the default must
give those of MPL_OPT_TEAM_SCANS 0 (one wavefront) or 2 (four) on either side of every line of the
launch rule, whichever gradients are wanted.  One pair of directions, so that a TRWP launch has as many
chains as the image has rows and an ISGMR launch twice as many."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

CASES = [
    # mode, labels, chains per compute unit, chains more than that, four wavefronts
    ("TRWP", 33, 1, 0, False), ("TRWP", 64, 1, 0, False), ("ISGMR", 64, 1, 0, False),
    ("TRWP", 65, 3, 0, True), ("TRWP", 128, 3, 1, False), ("ISGMR", 65, 3, 0, True),
    ("ISGMR", 128, 3, 2, False), ("TRWP", 152, 3, 0, True), ("TRWP", 154, 2, 0, True),
    ("TRWP", 154, 2, 1, False), ("ISGMR", 190, 3, 0, True), ("TRWP", 192, 3, 0, True),
    ("TRWP", 192, 3, 1, False), ("ISGMR", 192, 3, 2, False), ("TRWP", 215, 2, 0, True),
    ("TRWP", 215, 2, 1, False), ("TRWP", 217, 1, 0, True), ("TRWP", 217, 1, 1, False),
    ("TRWP", 256, 3, 0, True), ("TRWP", 256, 3, 1, False), ("ISGMR", 256, 2, 0, True),
    ("ISGMR", 256, 2, 2, False), ("ISGMR", 255, 1, 0, True), ("ISGMR", 255, 1, 2, False),
]


@pytest.mark.parametrize("mode,L,per_cu,more,four", CASES)
def test_launches_with_four_wavefronts_per_chain(gpu, mode, L, per_cu, more, four):
  import torch
  from mplayers_amd import _lib
  chains = per_cu * torch.cuda.get_device_properties(0).multi_processor_count + more
  n_dir, H, W, rho = 2, chains if mode == "TRWP" else chains // 2, 8, (0.5 if mode == "TRWP" else 1.0)
  rng = np.random.default_rng(L)
  ctx = rng.random(L).astype(np.float32)
  dcost = rng.standard_normal((1, 1, H, W, L)).astype(np.float32)
  imin = rng.integers(0, L, (1, n_dir, 1, 1, H, W, L)).astype(np.uint8)
  inorm = rng.integers(0, L, (1, n_dir, 1, 1, H, W)).astype(np.uint8)

  def dunary(option, wanted=False):
    _lib.set_option(_lib.OPT_TEAM_SCANS, option)
    try:
      return gpu.gpu_backward(mode, ctx, None, dcost, imin, inorm, rho, flags=_lib.F_PACKED_OFF,
                              want_dctx=wanted, want_dedge=wanted)[0]
    finally:
      _lib.set_option(_lib.OPT_TEAM_SCANS, 1)

  print("case", mode, L, chains, four, flush=True)
  one_wave, four_waves = dunary(0), dunary(2)
  # (up to 64 labels there is the kernel with one wavefront only)
  assert np.array_equal(one_wave, four_waves) == (L <= 64)
  expected = four_waves if four else one_wave
  assert np.array_equal(dunary(1), expected)
  assert np.array_equal(dunary(1, wanted=True), expected)


def test_a_call_reads_the_option_once(gpu):
  """A thread that sets MPL_OPT_TEAM_SCANS while another one is inside a backward call does not change
  the kernels of that call half way: its result has the bits of one of the two kernels."""
  import threading
  from mplayers_amd import _lib
  n_iter, n_dir, H, W, L = 4, 16, 6, 7, 70
  rng = np.random.default_rng(5)
  ctx = rng.random(L).astype(np.float32)
  dcost = rng.standard_normal((1, 1, H, W, L)).astype(np.float32)
  imin = rng.integers(0, L, (n_iter, n_dir, 1, 1, H, W, L)).astype(np.uint8)
  inorm = rng.integers(0, L, (n_iter, n_dir, 1, 1, H, W)).astype(np.uint8)
  run = lambda: gpu.gpu_backward("TRWP", ctx, None, dcost, imin, inorm, 0.5, want_dctx=False,
                                 want_dedge=False)[0]
  done = threading.Event()

  def toggle():
    while not done.is_set():
      _lib.set_option(_lib.OPT_TEAM_SCANS, 0)
      _lib.set_option(_lib.OPT_TEAM_SCANS, 2)

  pure = []
  try:
    for option in (0, 2):
      _lib.set_option(_lib.OPT_TEAM_SCANS, option)
      pure.append(run())
    thread = threading.Thread(target=toggle)
    thread.start()
    try:
      results = [run() for _ in range(200)]
    finally:
      done.set()
      thread.join()
  finally:
    _lib.set_option(_lib.OPT_TEAM_SCANS, 1)
  assert not np.array_equal(*pure)
  assert all(np.array_equal(r, pure[0]) or np.array_equal(r, pure[1]) for r in results)
