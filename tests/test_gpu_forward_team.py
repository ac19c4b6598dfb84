"""TRWP's forward scan with four wavefronts per chain (MPL_OPT_TEAM_SCANS): the bits of the scan with
one wavefront per chain -- messages, costs, labels, both index tensors -- for every kind of table, label
counts on both sides of a lane's share, chains on both sides of a block of pixels, negative weights,
given and undefined initial messages, pairs in one launch and in two."""
import numpy as np
import pytest

from tests.test_gpu_dense_split import _forward_flags

pytestmark = pytest.mark.gpu

TABLES = {
    "potts": lambda k, rng: np.minimum(k, 1),
    "band2": lambda k, rng: np.minimum(k, 2),
    "band4": lambda k, rng: 0.3 * np.minimum(k, 4) ** 2,
    "band7": lambda k, rng: 0.1 * np.minimum(k, 7) ** 2,
    "band14": lambda k, rng: 0.1 * np.minimum(k, 14) ** 2,
    "band20": lambda k, rng: 0.05 * np.minimum(k, 20) ** 2,
    "bent": lambda k, rng: np.where(k == 0, 0.2, np.minimum(k, 3) * 0.15),  # entry 0 is not the smallest
    "linear": lambda k, rng: 0.1 * k,
    "random": lambda k, rng: np.where(k == 0, 0, rng.random(len(k))),
}


def _run(gpu, option, unary, ctx, ew, n_dir, n_iter, training, flags=0, **kw):
  from mplayers_amd import _lib
  _lib.set_option(_lib.OPT_TEAM_SCANS, option)
  try:
    return _forward_flags(gpu, "TRWP", unary, ctx, ew, n_dir, n_iter, 0.5, training, flags, **kw)
  finally:
    _lib.set_option(_lib.OPT_TEAM_SCANS, 1)


def _same(a, b, training):
  for k in ("msg", "cost_final", "label_all") + (("msg_min_index", "msg_norm_index") if training else ()):
    assert np.array_equal(a[k], b[k]), k


def _problem(n_dir, B, H, W, L, table, seed=0, negative=False):
  rng = np.random.default_rng(1000 * L + 10 * H + W + seed)
  unary = (rng.random((B, 1, H, W, L)) * 3).astype(np.float32)
  if table == "2d":
    ctx = np.triu(rng.random((L, L)), 1).astype(np.float32)
  else:
    ctx = TABLES[table](np.arange(L, dtype=np.float64), rng).astype(np.float32)
  ew = (0.1 + 0.9 * rng.random((n_dir, B, 1, H, W))).astype(np.float32)
  if negative:
    ew[rng.random(ew.shape) < 0.1] = -0.5
  return unary, ctx, ew


@pytest.mark.parametrize("training", [True, False])
@pytest.mark.parametrize("L", [2, 16, 21, 33, 64, 65, 96, 127, 130, 192, 193, 256])
def test_same_bits_for_every_table(gpu, L, training):
  from mplayers_amd import _lib
  tables = ["2d"] if L == 21 else [t for t in TABLES if L > 8 or t in ("potts", "random")]
  for i, table in enumerate(tables):
    for negative in (False, True):
      print("case", L, training, table, negative, flush=True)
      problem = _problem(4, 1, 9, 14, L, table, i, negative)
      one = _run(gpu, 0, *problem, 4, 2, training, _lib.F_PACKED_OFF)
      four = _run(gpu, 2, *problem, 4, 2, training, _lib.F_PACKED_OFF)
      _same(four, one, training)


@pytest.mark.parametrize("L,table", [(21, "2d"), (40, "potts"), (96, "band4"), (192, "band4"), (256, "linear")])
@pytest.mark.parametrize("training", [True, False])
def test_chain_lengths_and_launches(gpu, L, table, training):
  """Chains of 1 to 50 pixels, 2 to 16 directions, one and two launches per pair, initial messages that are
  given, zero and undefined."""
  from mplayers_amd import _lib
  for n_dir, B, H, W in ((2, 1, 1, 1), (4, 2, 1, 2), (4, 1, 5, 6), (4, 1, 7, 12), (8, 1, 13, 25), (16, 2, 6, 11),
                         (4, 1, 3, 50)):
    problem = _problem(n_dir, B, H, W, L, table, 3)
    for flags, kw in ((0, {}), (_lib.F_FUSED_PAIRS_OFF, {}), (0, dict(msg_uninit=True))):
      print("case", L, table, n_dir, B, H, W, flags, kw, flush=True)
      flags |= _lib.F_PACKED_OFF
      one = _run(gpu, 0, *problem, n_dir, 3, training, flags, **kw)
      four = _run(gpu, 2, *problem, n_dir, 3, training, flags, **kw)
      _same(four, one, training)
    rng = np.random.default_rng(7)
    init = rng.random((n_dir, B, 1, H, W, L)).astype(np.float32)
    got = []
    for option in (0, 2):
      _lib.set_option(_lib.OPT_TEAM_SCANS, option)
      try:
        got.append(gpu.gpu_forward("TRWP", *problem, n_dir, 2, 0.5, training=training, saving_label=True,
                                   msg_init=init))
      finally:
        _lib.set_option(_lib.OPT_TEAM_SCANS, 1)
    _same(got[1], got[0], training)


@pytest.mark.parametrize("L", [2, 17, 31, 32, 33, 64, 65, 96, 97, 128, 129, 160, 161, 191, 192])
@pytest.mark.parametrize("training", [True, False])
def test_tables_declared_dense(gpu, L, training):
  """Four wavefronts that share the front labels: label counts at the edges of a wavefront's trips, of a lane's
  labels and of the front labels per wavefront; short and long chains (around a block of pixels:
  tests/test_gpu_dense_chains.py)."""
  from mplayers_amd import _lib
  flags = _lib.F_PACKED_OFF | _lib.F_DENSE_TABLE
  for H, W, table, negative in ((3, 1, "random", False), (8, 9, "random", True), (7, 16, "random", False),
                                (17, 25, "linear", False), (2, 40, "potts", True)):
    problem = _problem(4, 1, H, W, L, table, 5, negative)
    for more, kw in ((0, {}), (_lib.F_FUSED_PAIRS_OFF, {}), (0, dict(msg_uninit=True))):
      print("case", L, training, H, W, table, negative, more, kw, flush=True)
      one = _run(gpu, 0, *problem, 4, 3, training, _lib.F_PACKED_OFF | more, **kw)
      four = _run(gpu, 2, *problem, 4, 3, training, flags | more, **kw)
      if table == "linear":  # the label scan and the dense scan differ in the last bits of a tie
        assert np.abs(four["cost_final"] - one["cost_final"]).max() <= 1e-5 * max(1.0, np.abs(one["cost_final"]).max())
      else:
        _same(four, one, training)


@pytest.mark.parametrize("L", [2, 7, 8, 33, 64, 65, 96, 130, 192, 256])
@pytest.mark.parametrize("mode", ["TRWP", "ISGMR"])
def test_argmin_labels_exist_where_no_candidate_is_a_number(gpu, L, mode):
  """An edge weight that is NaN leaves a dense table's scan without a candidate to compare: the last label is kept,
  whichever scan takes the launch, and the reverse scan does not look outside its tables for it."""
  from mplayers_amd import _lib
  unary, ctx, ew = _problem(4, 1, 7, 9, L, "random", 9)
  ew[:, 0, 0, 3, 4] = np.nan
  for option, flags in ((0, 0), (2, 0), (2, _lib.F_DENSE_TABLE)):
    print("case", L, mode, option, flags, flush=True)
    _lib.set_option(_lib.OPT_TEAM_SCANS, option)
    try:
      got = _forward_flags(gpu, mode, unary, ctx, ew, 4, 2, 0.5 if mode == "TRWP" else 1.0, True,
                           flags | _lib.F_PACKED_OFF)
    finally:
      _lib.set_option(_lib.OPT_TEAM_SCANS, 1)
    assert got["msg_min_index"].max() < L and got["msg_norm_index"].max() < L
    assert not np.isfinite(got["msg"][:, 0, 0, 3, 4]).any()
    if L > 2:  # (two entries are a band, whose scan keeps the label itself)
      assert (got["msg_min_index"][:, :, 0, 0, 3, 4] == L - 1).all()


@pytest.mark.parametrize("L,ctx2d", [(2, 1), (20, 1), (22, 1), (33, 1), (64, 1), (21, 0)])
@pytest.mark.parametrize("training", [True, False])
def test_tables_the_operators_do_not_pass(gpu, L, ctx2d, training):
  """2-D tables of other label counts than 21, and 21 labels with a 1-D one, which the library takes."""
  import torch
  from mplayers_amd import _lib
  rng = np.random.default_rng(L)
  n_dir, n_iter, shape = 4, 2, (1, 1, 9, 14, L)
  table = np.triu(rng.random((L, L)), 1) if ctx2d else rng.random(L)
  unary, ctx, ew = gpu._t(3 * rng.random(shape)), gpu._t(table), gpu._t(rng.random((n_dir,) + shape[:4]) - 0.1)
  out = []
  for option in (0, 2):
    msg, cost, scratch = unary.new_zeros((n_dir,) + shape), torch.zeros_like(unary), torch.zeros_like(unary)
    u8 = dict(dtype=torch.uint8, device=unary.device)
    imin = torch.zeros((n_iter, n_dir) + shape, **u8)
    inorm, label = torch.zeros((n_iter, n_dir) + shape[:4], **u8), torch.zeros((n_iter,) + shape[:4], **u8)
    ptr = lambda t: t.data_ptr()
    print("case", L, ctx2d, training, option, flush=True)
    _lib.set_option(_lib.OPT_TEAM_SCANS, option)
    try:
      rc = _lib.load().mpl_trwp_forward(_lib.Shape(n_dir, 1, 9, 14, L, ctx2d), _lib.F_PACKED_OFF, 0.5, n_iter, 0,
                                        ptr(unary), ptr(ctx), ptr(ew), ptr(msg), ptr(cost), ptr(imin) if training else None,
                                        ptr(inorm) if training else None, ptr(scratch), ptr(label), None)
      torch.cuda.synchronize()
    finally:
      _lib.set_option(_lib.OPT_TEAM_SCANS, 1)
    _lib.check(rc, "trwp_forward")
    out.append([t.cpu().numpy() for t in (msg, cost, imin, inorm, label)])
  assert out[0][0].any() and (not training or out[0][2].any())
  for a, b in zip(*out):
    assert np.array_equal(a, b)


@pytest.mark.parametrize("L", [3, 7, 8, 9])
@pytest.mark.parametrize("mode", ["TRWP", "ISGMR"])
@pytest.mark.parametrize("option", [0, 2])
def test_dense_tables_of_few_labels(gpu, oracle, L, mode, option):
  """Both sides of the label count from which a dense 1-D table is scanned with sliding entries, one and four
  wavefronts per chain, against the oracle."""
  from mplayers_amd import _lib
  unary, ctx, ew = _problem(4, 1, 9, 14, L, "random", 2, negative=True)
  rho = 0.5 if mode == "TRWP" else 1.0
  print("case", L, mode, option, flush=True)
  ref = oracle.forward(mode, unary, ctx, ew, 4, 2, rho)
  _lib.set_option(_lib.OPT_TEAM_SCANS, option)
  try:
    got = _forward_flags(gpu, mode, unary, ctx, ew, 4, 2, rho, True, _lib.F_PACKED_OFF)
  finally:
    _lib.set_option(_lib.OPT_TEAM_SCANS, 1)
  scale = float(np.abs(ref["cost_final"]).max())
  for k in ("msg", "cost_final"):
    assert np.abs(got[k] - ref[k]).max() <= 1e-5 * scale, k
  # (labels whose candidates are closer than that aside)
  assert (got["msg_min_index"] != ref["msg_min_index"]).mean() <= 1e-3
