"""The sigmoid re-parameterisation of a learned table under masks: the values and gradients that indexing
with the stored locations gives (MP_module.py:207-220), for every form the locations take, and after they or
the table change."""
import argparse
import copy
import io

import numpy as np
import pytest
import torch

from mplayers_amd import MPModule


def _by_index(table, loc, diag, weight, weight_first, diag_value):
  label_context = table * (weight if weight_first else 1)
  label_context[loc] = (2 if weight_first else 2 * weight) * torch.sigmoid(label_context[loc].flatten())
  label_context[tuple(diag) if isinstance(diag, list) else diag] = diag_value
  return label_context


LOCATIONS = {
    "triangle": (np.triu_indices(5, k=1), [range(5), range(5)], 2),
    "tensor": (tuple(torch.from_numpy(i) for i in np.triu_indices(5, k=1)), [range(5), range(5)], 2),
    "vector": (range(1, 5), range(1), 1),
    "list": ([1, 3], [0], 1),
    "slice": (slice(2, None), 0, 1),
    "negative": (np.array([-1, -2]), range(2), 1),
    "overlap": (range(0, 5), range(2), 1),
    "repeated": ([1, 3, 3], [0], 1),
    "two names of one entry": ([-1, 4], [0], 1),
    "repeated, 2-D": ((np.array([0, 0, 1]), np.array([1, 1, 2])), [range(5), range(5)], 2),
    "pinned twice": ([1, 3], [[0, 0, -5]], 1),
    "no entry": ([], [0], 1),
    "empty range": (range(1, 1), [0], 1),
    "bytes as a mask": (np.array([0, 1, 1, 0, 0], np.uint8), [0], 1),
    "booleans": (np.array([False, True, True, False, False]), [True, False, False, False, False], 1),
    "short integers": (np.array([1, 3], np.int16), [0], 1),
    "floats": (np.array([1., 2.]), [0], 1),
    "rows": (np.triu_indices(5, k=1), np.array([[0, 1], [2, 3]]), 2),
    "all": ([1, 3], Ellipsis, 1),
}


@pytest.mark.parametrize("name", sorted(LOCATIONS))
@pytest.mark.parametrize("weight_first", [False, True])
def test_masks_give_what_indexing_gives(name, weight_first):
  loc, diag, dims = LOCATIONS[name]
  args = argparse.Namespace(mpnet_mrf_mode="TRWP", mpnet_max_iter=1, mpnet_n_dirs=4, n_classes=5,
                            mpnet_term_weight=1.5, mpnet_smoothness_train="sigmoid", mpnet_diag_value=0.25)
  module = MPModule(args)
  gen = torch.Generator().manual_seed(1)
  for round_ in range(3):  # other values, then other locations
    table = torch.nn.Parameter(torch.randn((5,) * dims, generator=gen))
    with torch.no_grad():
      table[(0,) * dims] = float("inf")  # (pinned or not touched in most of the cases)
    if round_ == 2 and name == "vector":
      loc = range(2, 4)
    module.set_label_context(table, loc, diag)
    upstream = torch.randn(table.shape, generator=gen)
    got = module._effective_label_context(weight_first=weight_first)
    (got_grad,) = torch.autograd.grad(got, table, upstream)
    want = _by_index(table, loc, diag, 1.5, weight_first, 0.25)
    (want_grad,) = torch.autograd.grad(want, table, upstream)
    assert torch.equal(got, want) and torch.equal(got_grad, want_grad)


def _module(loc, diag, dims, **more):
  args = argparse.Namespace(**dict(dict(mpnet_mrf_mode="TRWP", mpnet_max_iter=1, mpnet_n_dirs=4, n_classes=5,
                                        mpnet_term_weight=1.5, mpnet_smoothness_train="sigmoid",
                                        mpnet_diag_value=0.25), **more))
  module = MPModule(args)
  table = torch.nn.Parameter(torch.randn((5,) * dims, generator=torch.Generator().manual_seed(2)))
  module.set_label_context(table, loc, diag)
  return module


def _check(module):
  """Value and gradient of the module's table are those of indexing."""
  table = module.label_context
  upstream = torch.arange(1., 1. + table.numel()).reshape(table.shape)
  got = module._effective_label_context()
  want = _by_index(table, module.label_context_loc, module.label_context_diag_loc, 1.5, False,
                   module.args.mpnet_diag_value)
  assert type(got) is torch.Tensor and torch.equal(got, want)
  assert torch.equal(torch.autograd.grad(got, table, upstream)[0], torch.autograd.grad(want, table, upstream)[0])


def test_a_first_call_under_inference_mode():
  """An evaluation before training leaves nothing that autograd cannot save."""
  module = _module(*LOCATIONS["triangle"])
  with torch.inference_mode():
    module._effective_label_context()
  _check(module)


def test_locations_that_are_refused_stay_refused():
  args = argparse.Namespace(mpnet_mrf_mode="TRWP", mpnet_max_iter=1, mpnet_n_dirs=4, n_classes=5,
                            mpnet_term_weight=1.0, mpnet_smoothness_train="sigmoid", mpnet_diag_value=0.0)
  module = MPModule(args)
  module.set_label_context(torch.nn.Parameter(torch.rand(5, 5)), [0, 3], [range(5), range(5)])
  with pytest.raises(RuntimeError):
    module._effective_label_context()
  module.set_label_context(torch.nn.Parameter(torch.rand(5)), [7], [0])
  with pytest.raises(IndexError):
    module._effective_label_context()
  for loc, diag, error in ((slice(None, None, -1), [0], ValueError), ([1, 3], slice(2, None, -1), ValueError),
                           ([1, 3], np.array([1, 0, 0, 0, 1], np.uint8), RuntimeError)):
    module.set_label_context(torch.nn.Parameter(torch.rand(5)), loc, diag)
    with pytest.raises(error):
      module._effective_label_context()


@pytest.mark.parametrize("value", [1, 0.25, True, np.float64(0.5), torch.tensor(0.5), torch.tensor([0.5]),
                                   torch.arange(5.)])
def test_pinned_values(value):
  """One number, or a tensor that indexing spreads over the pinned entries."""
  _check(_module(*LOCATIONS["triangle"], mpnet_diag_value=value))


def test_a_pinned_value_that_is_refused_stays_refused():
  with pytest.raises(TypeError):
    _module(*LOCATIONS["triangle"], mpnet_diag_value=np.float32(0.5))._effective_label_context()


def _fake(f, table):
  from torch._subclasses.fake_tensor import FakeTensorMode
  with FakeTensorMode(allow_non_fake_inputs=True):
    f(table)


def _export(f, table):
  module = type("Module", (torch.nn.Module,), dict(forward=lambda self, x: f(x)))()
  return torch.export.export(module, (table,)).module()(2 * table)


def _make_fx(f, table):
  from torch.fx.experimental.proxy_tensor import make_fx
  return make_fx(f)(table)(2 * table)


TRANSFORMS = {
    "fake tensors": _fake, "export": _export, "make_fx": _make_fx,
    "compile": lambda f, table: torch.compile(f, backend="eager", fullgraph=True)(2 * table),
    "trace": lambda f, table: torch.jit.trace(f, (table,), check_trace=False)(2 * table),
    "vmap": lambda f, table: torch.func.vmap(f)(torch.stack([2 * table, table]))[0],
    "vmap of others": lambda f, table: torch.func.vmap(lambda x: f(2 * table) * x)(torch.ones(3, 1, 1))[1],
    "jvp": lambda f, table: torch.func.jvp(f, (2 * table,), (table,))[0],
    "grad of others": lambda f, table: torch.func.grad(lambda x: (f(2 * table) * x).sum())(torch.ones(5, 5)),
}


@pytest.mark.parametrize("name", sorted(TRANSFORMS))
@pytest.mark.parametrize("warm", [False, True])
def test_traces_and_transforms(name, warm):
  """They see the table's own values, take nothing that another call kept, and leave nothing behind for the next."""
  loc, diag, _ = LOCATIONS["triangle"]
  table = torch.randn(5, 5, generator=torch.Generator().manual_seed(3))
  module = _module(loc, diag, 2)
  if warm:
    module._effective_label_context()
  parameter = module.label_context
  del module.label_context

  def effective(x):
    module.label_context = x
    return module._effective_label_context()

  got = TRANSFORMS[name](effective, table)
  if got is not None:
    assert torch.equal(got, _by_index(2 * table, loc, diag, 1.5, False, 0.25))
  module.label_context = parameter
  _check(module)


@pytest.mark.gpu
def test_masks_on_another_stream(gpu, monkeypatch):
  """A call on another stream than the one the masks were formed on holds their memory until it is through, also
  when other locations have taken their place."""
  loc, diag, _ = LOCATIONS["triangle"]
  table = torch.nn.Parameter(torch.randn(5, 5, generator=torch.Generator().manual_seed(3)).cuda())
  module = _module(loc, diag, 2)
  module.label_context = table
  held = []
  record = torch.Tensor.record_stream
  monkeypatch.setattr(torch.Tensor, "record_stream", lambda self, stream: (held.append(stream), record(self, stream)))
  first = module._effective_label_context()
  assert not held
  side = torch.cuda.Stream()
  side.wait_stream(torch.cuda.current_stream())
  with torch.cuda.stream(side):
    second = module._effective_label_context()
  assert held == [side, side]
  module.set_label_context(table, (np.array([0]), np.array([1])), diag)
  module._effective_label_context()
  torch.cuda.synchronize()
  want = _by_index(table.detach().cpu(), loc, diag, 1.5, False, 0.25)
  assert torch.allclose(first.detach().cpu(), want) and torch.equal(first, second)


@pytest.mark.parametrize("device", ["cpu", pytest.param("cuda", marks=pytest.mark.gpu)])
def test_copies_and_files_of_the_module(device):
  """They hold no masks, nor the stream those were formed on, and work wherever they are loaded."""
  loc, diag, _ = LOCATIONS["triangle"]
  module = _module(loc, diag, 2).to(device)
  want = module._effective_label_context().detach().cpu()
  assert "_kept_masks" in module.__dict__
  file = io.BytesIO()
  torch.save(module, file)
  file.seek(0)
  # (the module of this test, written above)
  loaded = torch.load(file, map_location="cpu", weights_only=False)
  for other in (copy.deepcopy(module), loaded):
    assert "_kept_masks" not in other.__dict__
    assert torch.allclose(other._effective_label_context().detach().cpu(), want)
  assert torch.allclose(loaded.to(device)._effective_label_context().detach().cpu(), want)
