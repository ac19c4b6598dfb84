"""Labels of every iteration: the pass that finds them also stores what the next pass over the same
planes would (cost_final, TRWP's re-summed belief plane, ISGMR's U planes of the next iteration).

Without labels those passes run by themselves, so a call with labels must leave the same bits as one
without, and the labels of iteration k are the smallest argmin of the cost of a call that ends there."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


# 3, 29: label counts that keep the passes apart; groups of 1, 2, 16 (15 in use) and 64 lanes
@pytest.mark.parametrize("L", [3, 4, 8, 29, 60, 256])
@pytest.mark.parametrize("mode,rho", [("TRWP", 0.5), ("ISGMR", 1.0), ("ISGMR", 0.5)])
@pytest.mark.parametrize("n_dir", [2, 4, 8, 16])
def test_pass_with_labels_is_the_passes_apart(gpu, mode, rho, n_dir, L):
  from mplayers_amd import _lib
  rng = np.random.default_rng(10 * L + n_dir)
  B, H, W = 2, 7, 11
  unary = rng.random((B, 1, H, W, L)).astype(np.float32)
  ctx = (0.1 * np.minimum(np.arange(L), 2)).astype(np.float32)
  ew = (0.1 + 0.9 * rng.random((n_dir, B, 1, H, W))).astype(np.float32)
  _lib.set_option(_lib.OPT_BELIEF_REBUILD, 2)
  try:
    for min_a_dir in (False, True):
      print("case", mode, rho, n_dir, L, min_a_dir, flush=True)
      run = lambda n_iter, labels: gpu.gpu_forward(mode, unary, ctx, ew, n_dir, n_iter, rho, training=False,
                                                   saving_label=labels, enable_min_a_dir=min_a_dir)
      apart = [run(n + 1, False) for n in range(5)]
      for n_iter in (1, 4, 5):
        got = run(n_iter, True)
        for name in ("msg", "cost_final"):
          assert np.array_equal(got[name], apart[n_iter - 1][name]), (name, n_iter)
        for k in range(n_iter):
          assert np.array_equal(got["label_all"][k], apart[k]["cost_final"].argmin(-1)), (n_iter, k)
  finally:
    _lib.set_option(_lib.OPT_BELIEF_REBUILD, _lib.BELIEF_REBUILD_DEFAULT)


@pytest.mark.parametrize("L", [3, 8, 60, 256])
@pytest.mark.parametrize("n_dir", [2, 4, 6, 8, 16])
def test_sgm_keeps_the_passes_apart(gpu, n_dir, L):
  """The one-iteration operator weights the unary terms by the number of directions; its label pass
  stores nothing else."""
  rng = np.random.default_rng(10 * L + n_dir)
  B, H, W = 2, 7, 11
  unary = rng.random((B, 1, H, W, L)).astype(np.float32)
  ctx = (0.1 * np.minimum(np.arange(L), 2)).astype(np.float32)
  ew = (0.1 + 0.9 * rng.random((n_dir, B, 1, H, W))).astype(np.float32)
  print("case", n_dir, L, flush=True)
  plain, got = (gpu.gpu_forward("ISGMR", unary, ctx, ew, n_dir, 1, 1.0, training=False, enable_sgm=True,
                                saving_label=labels) for labels in (False, True))
  for name in ("msg", "cost_final"):
    assert np.array_equal(got[name], plain[name]), name
  # six directions: the product with the factor rounds, and either pass may fuse it into its first
  # sum, so labels are compared where the two smallest costs are further apart than that (a cost is
  # below 6 + 6 * 0.2, seven roundings of it below 2e-6 in either pass)
  cost = plain["cost_final"].astype(np.float64)
  two = np.partition(cost, 1, axis=-1)[..., :2]
  clear = (two[..., 1] - two[..., 0] > 1e-5) | (n_dir != 6)
  assert np.array_equal(got["label_all"][0][clear], cost.argmin(-1)[clear])
