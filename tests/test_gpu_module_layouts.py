"""The modules in training with and without saved labels: without them the operators write the costs in the network's
layout and the gradient is turned over in the backward pass, with them the costs are turned over.  Costs and all gradients
of both against the oracle, and the same bits."""
import argparse

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _close(got, ref, what):
  got = got.detach().cpu().numpy()
  assert got.shape == ref.shape, what
  assert np.abs(got - ref).max() <= 1e-4 * max(1.0, float(np.abs(ref).max())), what  # (as in the other tests of the modules)


@pytest.mark.parametrize("mode,L,cv,n_dir,W", [
    ("TRWP", 21, 1, 4, 9), ("TRWP", 21, 2, 4, 8), ("TRWP", 12, 1, 8, 9), ("TRWP", 40, 2, 4, 9), ("TRWP", 96, 1, 4, 8),
    ("ISGMR", 21, 1, 8, 9), ("ISGMR", 12, 2, 8, 8), ("ISGMR", 70, 1, 4, 9), ("SGM", 33, 1, 8, 9), ("SGM", 64, 2, 4, 8),
    ("soft", 21, 1, 4, 9), ("soft", 21, 2, 4, 8), ("soft", 9, 1, 4, 8), ("soft", 40, 2, 4, 9),
    ("hard_soft", 21, 1, 4, 8), ("hard_soft", 70, 2, 4, 9)])
def test_costs_and_gradients_in_both_layouts(gpu, oracle, mode, L, cv, n_dir, W):
  import torch
  from mplayers_amd import MPModule, MP_module_hard_soft
  rng = np.random.default_rng(L + cv)
  soft = "soft" in mode
  B, H, n_iter = 2, 7, 1 if mode == "SGM" else 2
  rho = 1.0 if mode in ("ISGMR", "SGM") else 0.5
  args = dict(mpnet_mrf_mode="TRWP" if soft else mode, mpnet_max_iter=n_iter, mpnet_n_dirs=n_dir, n_classes=L,
              mpnet_term_weight=1.0, mpnet_smoothness_train="", mpnet_smoothness_mode="",
              mpnet_smoothness_trunct_value=3, mpnet_smoothness_trunct_loc=-1, mpnet_diag_value=0, enable_symmetric=True,
              mpnet_enable_soft=mode == "soft", enable_seg=L == 21)
  if L == 21:
    ctx = np.triu(rng.random((L, L)), 1).astype(np.float32)
    loc, diag = np.triu_indices(L, k=1), [range(L), range(L)]
  else:
    ctx = np.concatenate([[0], rng.random(L - 1)]).astype(np.float32)
    loc, diag = np.arange(1, L), [0]
  unary = rng.standard_normal((B, cv, L, H, W)).astype(np.float32)
  dcost = rng.standard_normal((B, cv, L, H, W)).astype(np.float32)
  # (the modules pass edge weights per batch item, so those of one cost volume only)
  ew = (0.1 + 0.9 * rng.random((B, n_dir, H, W))).astype(np.float32) if cv == 1 else None
  t = lambda a: torch.from_numpy(np.ascontiguousarray(a)).cuda()
  out = {}
  for saving in (True, False):
    cls = MP_module_hard_soft.MPModule if soft else MPModule
    mod = cls(argparse.Namespace(**args), enable_saving_label=saving).cuda().train()
    table = torch.nn.Parameter(t(ctx))
    mod.set_label_context(table, loc, diag)
    # the gradient as autograd may hand it over: contiguous, or the strides of another layout
    for grad in (t(dcost), t(dcost.transpose(0, 1, 3, 4, 2)).permute(0, 1, 4, 2, 3)):
      table.grad = None
      u = t(unary).requires_grad_(True)
      e = t(ew).requires_grad_(True) if ew is not None else None
      print("case", mode, L, cv, n_dir, saving, grad.is_contiguous(), flush=True)
      res = mod(u, e)
      assert res[0].is_contiguous() and (res[2].numel() > 0) == saving
      res[0].backward(grad)
      torch.cuda.synchronize()
      out[saving, grad.is_contiguous()] = res[0].detach(), u.grad, e.grad if e is not None else None, table.grad, res[3:]
  first = out[False, True]
  for key, got in out.items():
    for i in (0, 1, 2):
      assert got[i] is None and first[i] is None or torch.equal(got[i], first[i]), (key, i)
    assert float((got[3] - first[3]).abs().max()) <= 1e-5 * max(1.0, float(first[3].abs().max())), key
  back = lambda a: np.ascontiguousarray(a.transpose(0, 1, 3, 4, 2))
  en = np.ascontiguousarray(ew[:, None].transpose(2, 0, 1, 3, 4)) if ew is not None else None
  f64 = lambda a: None if a is None else a.astype(np.float64)
  cost, du, de, dc, kept = first
  if mode == "soft":
    ref = oracle.forward_soft(back(unary), ctx, en, n_dir, n_iter, rho)
    ones = np.ones((n_dir, B, cv, H, W)) if en is None else f64(en)
    grads = oracle.backward_soft(f64(ctx), ones, f64(back(dcost)), f64(kept[0].detach().cpu().numpy()),
                                 kept[1].cpu().numpy(), rho)
  else:
    base, sgm = ("ISGMR", True) if mode == "SGM" else ("TRWP" if soft else mode, False)
    ref = oracle.forward(base, back(unary), ctx, en, n_dir, n_iter, rho, enable_sgm=sgm)
    grads = oracle.backward(base, f64(ctx), f64(en), f64(back(dcost)), ref["msg_min_index"], ref["msg_norm_index"], rho,
                            enable_sgm=sgm, same_label=soft)
  _close(cost, ref["cost_final"].transpose(0, 1, 4, 2, 3), "cost")
  _close(du, grads[0].transpose(0, 1, 4, 2, 3), "dunary")
  _close(dc, grads[1].reshape(ctx.shape), "dcontext")
  if en is not None:
    _close(de, grads[2].reshape(en.shape)[:, :, 0].transpose(1, 0, 2, 3), "dedge_weights")
