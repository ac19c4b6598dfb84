"""Dense 1-D tables with four wavefronts per chain: a wavefront whose whole share of the front labels is no number has
no part in the minimum.  Where the table forbids jumps (+inf) and an edge weight is zero the candidate is 0 * inf."""
import numpy as np
import pytest

from tests.test_gpu_forward_team import _run

pytestmark = pytest.mark.gpu

SHARE = {17: 8, 32: 8, 64: 16, 96: 24, 128: 32, 129: 40, 160: 40, 192: 48}  # front labels per wavefront


def _table_with_forbidden_jumps(L, lo, hi, W, iterations, training, B=1):
  rng = np.random.default_rng(L + lo)
  unary = (3 * rng.random((1, 1, 2, W, L))).astype(np.float32)
  ctx = rng.random(L).astype(np.float32)
  ctx[lo:hi] = np.inf
  ctx[0] = 0
  ew = (0.1 + 0.9 * rng.random((4, 1, 1, 2, W))).astype(np.float32)
  ew[:, 0, 0, 1, W // 2] = 0
  return np.repeat(unary, B, 0), ctx, np.repeat(ew, B, 1), 4, iterations, training


def _same(four, one, training):
  for k in ("msg", "cost_final", "label_all") + (("msg_min_index", "msg_norm_index") if training else ()):
    assert np.array_equal(four[k], one[k], equal_nan=True), k


@pytest.mark.parametrize("L", sorted(SHARE))
@pytest.mark.parametrize("share", [0, 1, 2, 3])
@pytest.mark.parametrize("training", [True, False])
def test_share_without_a_number(gpu, L, share, training):
  import torch
  from mplayers_amd import _lib
  lo, hi = share * SHARE[L], min(L, (share + 1) * SHARE[L])
  if lo >= L:
    pytest.skip("no labels")
  many = 3 + torch.cuda.get_device_properties(0).multi_processor_count // 2
  for B in (1,) if L <= 128 else (1, many):  # (more chains than units: the wavefronts serve themselves)
    # (the trip of eight as well: the first and a later one of a share)
    for first, last in ((lo, hi), (lo, min(lo + 8, hi)), (max(hi - 8, lo), hi)):
      problem = _table_with_forbidden_jumps(L, first, last, 9, 2, training, B)
      print("case", L, share, training, B, first, last, flush=True)
      one = _run(gpu, 0, *problem, _lib.F_PACKED_OFF)
      four = _run(gpu, 2, *problem, _lib.F_PACKED_OFF | _lib.F_DENSE_TABLE)
      assert np.isfinite(one["msg"]).all()
      _same(four, one, training)


@pytest.mark.parametrize("L", [32, 96, 128, 160, 192])
@pytest.mark.parametrize("many", [False, True])
def test_argmin_labels_against_the_definition(gpu, L, many):
  """One row, one sweep: the largest front label whose candidate is the minimum of those that are numbers, +inf among
  them; the last label where there is none.  Beliefs and table are small whole numbers: no rounding."""
  import torch
  from mplayers_amd import _lib
  rng = np.random.default_rng(L)
  cus = torch.cuda.get_device_properties(0).multi_processor_count
  B = cus + 3 if many else 1
  unary = rng.integers(0, 50, (1, 1, 1, 2, L)).astype(np.float32)
  dist = np.abs(np.arange(L)[:, None] - np.arange(L))
  n = SHARE[L]
  for kind in range(4):
    ctx = rng.integers(0, 9, L).astype(np.float32)
    u = unary.copy()
    if kind == 0:
      ctx[n:2 * n] = np.nan
    elif kind == 1:  # numbers next to the diagonal only
      ctx[8:] = np.nan
    elif kind == 2:  # the same, and +inf for the labels of the first shares: nothing else is left there
      ctx[8:] = np.nan
      u[..., :2 * n + 3] = np.inf
    else:            # no label has a number near it
      ctx[:L // 2 + 1] = np.nan
    ew = np.ones((2, 1, 1, 1, 2), np.float32)
    with np.errstate(invalid="ignore"):
      cand = 0.5 * u[0, 0, 0, 0] + ctx[dist]  # [label][front label], rho = 0.5, no messages yet
    least = np.where(np.isnan(cand), np.inf, cand).min(1)
    want = np.where((cand == least[:, None]).any(1), L - 1 - np.argmax((cand == least[:, None])[:, ::-1], 1), L - 1)
    print("case", L, B, kind, flush=True)
    # one wavefront per chain, four with the same step, four that share the front labels
    for option, flags in ((0, 0), (2, 0), (2, _lib.F_DENSE_TABLE)):
      got = _run(gpu, option, np.repeat(u, B, 0), ctx, np.repeat(ew, B, 1), 2, 1, True, _lib.F_PACKED_OFF | flags)
      for b in (0, B - 1):
        assert np.array_equal(got["msg_min_index"][0, 0, b, 0, 0, 1], want), (kind, option, flags)
        with np.errstate(invalid="ignore"):
          assert np.array_equal(got["msg"][0, b, 0, 0, 1], (least - least.min()).astype(np.float32), equal_nan=True), kind


@pytest.mark.parametrize("L", [8, 17, 32, 64, 96, 128, 160, 192, 256])
@pytest.mark.parametrize("share", [0, 1, 2, 3])
@pytest.mark.parametrize("training", [True, False])
def test_unary_terms_without_a_number(gpu, L, share, training):
  """Unary terms of a quarter of the labels that are NaN, at a chain's start and inside it: the messages stay numbers, in
  every scan the same ones."""
  import torch
  from mplayers_amd import _lib
  n = SHARE.get(L, -(-L // 4))
  rng = np.random.default_rng(L + share)
  ctx = rng.random(L).astype(np.float32)
  ctx[[0, L - 1]] = 0  # (no band: entries above the last one)
  many = 3 + torch.cuda.get_device_properties(0).multi_processor_count // 2
  for B in (1,) if L <= 128 else (1, many):
    for x in (0, 4, 8):
      unary = (3 * rng.random((1, 1, 2, 9, L))).astype(np.float32)
      unary[0, 0, 1, x, share * n:(share + 1) * n] = np.nan
      ew = (0.1 + 0.9 * rng.random((4, 1, 1, 2, 9))).astype(np.float32)
      problem = np.repeat(unary, B, 0), ctx, np.repeat(ew, B, 1), 4, 2, training
      print("case", L, share, training, B, x, flush=True)
      one = _run(gpu, 0, *problem, _lib.F_PACKED_OFF)
      assert np.isfinite(one["msg"]).all()
      for option, flags in ((2, 0), (2, _lib.F_DENSE_TABLE), (0, _lib.F_DENSE_TABLE)):
        if L < 17 and flags:
          continue
        _same(_run(gpu, option, *problem, _lib.F_PACKED_OFF | flags), one, training)
