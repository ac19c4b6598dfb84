"""Python surface of the message-passing layers: TRWPFunction, ISGMRFunction, MPModule.

Same names, arguments, return tuples and `args` namespace handling as the reference's
pytorch/MP_module.py:17-234, so a model written against it runs unchanged; the operators
underneath are the HIP library of this package instead of the CUDA extensions.

Tensor layouts (as in the reference):
  Function.apply(unary (B, cv, H, W, L), label_context (L,) or (21, 21),
                 edge_weights (n_dir, B, cv, H, W) or None, args) -> (cost_final, label_all)
  MPModule.forward(unary (B, cv, L, H, W), edge_weights (B, n_dir, H, W) or None)
                 -> (cost_final (B, cv, L, H, W), label_context[None], label_all, None, None)
"""
import numpy as np
import torch
import torch.nn as nn

from . import _lib, lib_seg, lib_stereo
from .label_context import create_label_context
from .layout import gradient_labels_last, labels_first, labels_last


def _ops_for(n_disp):
  # the reference keeps two builds and picks the segmentation one for 21 labels
  # (MP_module.py:24,95); one library backs both names here
  return lib_seg if n_disp == 21 else lib_stereo


_EMPTY_U8 = dict(dtype=torch.uint8)


def _forward_buffers(unary, args, n_dir, n_iter, with_message_tmp, cost_labels_first=False):
  """Allocates what the operators fill in place (MP_module.py:26-45, 97-118).  Nothing is
  zero-filled: the library writes every element that is ever read (index bytes of chain-start
  pixels stay unwritten and are never used), and the operators are told that the messages start
  at zero (msg_uninit) instead of being handed a cleared tensor, so the memsets the reference
  pays for are gone."""
  batch, cv, h, w, n_disp = unary.size()
  buf = dict(
      message=unary.new_empty(n_dir, batch, cv, h, w, n_disp),
      cost_final=unary.new_empty((batch, cv, n_disp, h, w) if cost_labels_first else (batch, cv, h, w, n_disp)),
      unary_update=unary.new_empty(batch, cv, h, w, n_disp))
  if with_message_tmp:
    buf["message_tmp"] = unary.new_empty(n_dir, batch, cv, h, w, n_disp)
  if args.training:
    buf["message_index"] = unary.new_empty(n_iter, n_dir, batch, cv, h, w, n_disp, **_EMPTY_U8)
    buf["cost_index"] = unary.new_empty(n_iter, n_dir, batch, cv, h, w, **_EMPTY_U8)
  else:
    buf["message_index"] = torch.empty(0, **_EMPTY_U8)
    buf["cost_index"] = torch.empty(0, **_EMPTY_U8)
  if args.enable_saving_label:
    buf["label_all"] = unary.new_empty(n_iter, batch, cv, h, w, **_EMPTY_U8)
  else:
    buf["label_all"] = torch.empty(0, **_EMPTY_U8)
  return buf


def _backward_buffers(dcost_final, message_index, with_message_tmp, need_context=True,
                      need_edge_weights=True):
  """Allocates the gradient tensors (MP_module.py:65-74, 139-150).  dedge_weights and
  dlabel_context accumulate and start at zero; dunary is written everywhere and the scratch
  tensors are written before they are read.  A gradient autograd does not ask for (a fixed
  pairwise table, no edge weights or ones that are not learned) is an empty tensor: the operators
  then leave that part of the reverse scan out."""
  n_iter, n_dir, batch, cv, h, w, n_disp = message_index.size()
  buf = dict(
      dunary=dcost_final.new_empty(batch, cv, h, w, n_disp),
      dmessage=dcost_final.new_empty(n_dir, batch, cv, h, w, n_disp),
      dunary_update=dcost_final.new_empty(0))
  if need_edge_weights:
    buf["dedge_weights"] = dcost_final.new_zeros(n_dir, batch, cv, h, w)
  else:
    buf["dedge_weights"] = dcost_final.new_empty(0)
  if with_message_tmp:
    buf["dmessage_tmp"] = dcost_final.new_empty(n_dir, batch, cv, h, w, n_disp)
  buf["flags"] = 0
  if need_context:
    buf["dlabel_context"], buf["dunary_update"], buf["flags"] = _context_gradient(
        dcost_final, n_iter, n_dir, batch * cv, h, w, n_disp,
        (n_disp, n_disp) if n_disp == 21 else (n_disp,))
  else:
    buf["dlabel_context"] = dcost_final.new_empty(0)
  return buf


def _context_gradient(like, n_iter, n_dir, batch, h, w, n_disp, size):
  """dlabel_context, the operators' scratch tensor and their flags: with many chains these take turns on
  tables of their own in the scratch (MPL_F_DCONTEXT_COPIES), whose sum overwrites dlabel_context."""
  ctx2d = n_disp == 21  # (what the operators take the table for)
  copies = 0
  if like.is_cuda and len(size) == (2 if ctx2d else 1):
    copies = _lib.dcontext_copies(_lib.Shape(n_dir, batch, h, w, n_disp, int(ctx2d)), n_iter)
  if copies == 0:
    return like.new_zeros(size), like.new_empty(0), 0
  return like.new_empty(size), like.new_zeros((copies,) + size), _lib.F_DCONTEXT_COPIES


def _sums_labels_first(unary, args):
  """Whether the operators are to write the costs in the network's layout themselves (not in the reference).  Where
  labels are saved, the pass that finds the last ones stores the costs in the kernels' layout."""
  return unary.is_cuda and unary.dtype == torch.float32 and not args.enable_saving_label


def _table_flags(args):
  """MPL_F_DENSE_TABLE when the module says its pairwise table is dense (not in the reference: the
  kind of the table is only known on the device otherwise, see include/mplayers_amd.h)."""
  return _lib.F_DENSE_TABLE if getattr(args, "dense_table", False) else 0


class TRWPFunction(torch.autograd.Function):
  """Tree-reweighted message passing, Gauss-Seidel over directions (MP_module.py:17-86)."""

  @staticmethod
  def forward(ctx, unary, label_context, edge_weights, args, cost_labels_first=False):
    # cost_labels_first: cost_final comes as (batch, cv, labels, H, W), as the module returns it
    n_disp = unary.size(4)
    rho, n_iter, n_dir = args.rho, int(args.mpnet_max_iter), int(args.mpnet_n_dirs)
    buf = _forward_buffers(unary, args, n_dir, n_iter, False, cost_labels_first)
    enable_edge_weights = edge_weights is not None
    if not enable_edge_weights:
      edge_weights = unary.new_ones((n_dir,) + tuple(unary.shape[:4]))
    _ops_for(n_disp).TRWP.forward(rho, n_iter, int(args.enable_min_a_dir), unary, label_context,
                                  edge_weights, buf["message"], buf["cost_final"],
                                  buf["message_index"], buf["cost_index"], buf["unary_update"],
                                  buf["label_all"], msg_uninit=True,
                                  flags=_table_flags(args) | (_lib.F_COST_LABELS_FIRST if cost_labels_first else 0))
    ctx.cost_labels_first = cost_labels_first
    ctx.intermediate_results = (rho, buf["message_index"], buf["cost_index"], label_context,
                                edge_weights, enable_edge_weights)
    return buf["cost_final"], buf["label_all"]

  @staticmethod
  def backward(ctx, dcost_final, dmessage_all):
    rho, message_index, cost_index, label_context, edge_weights, enable_edge_weights = \
        ctx.intermediate_results
    del ctx.intermediate_results
    dcost_final = gradient_labels_last(dcost_final) if ctx.cost_labels_first else dcost_final.contiguous()
    n_disp = message_index.size(6)
    need_context = ctx.needs_input_grad[1]
    need_edge_weights = enable_edge_weights and ctx.needs_input_grad[2]
    buf = _backward_buffers(dcost_final, message_index, False, need_context, need_edge_weights)
    _ops_for(n_disp).TRWP.backward(rho, label_context, edge_weights, dcost_final, message_index,
                                   cost_index, buf["dunary"], buf["dlabel_context"],
                                   buf["dedge_weights"], buf["dmessage"], buf["dunary_update"],
                                   flags=buf["flags"])
    return (buf["dunary"], buf["dlabel_context"] if need_context else None,
            buf["dedge_weights"] if need_edge_weights else None, None, None)


class ISGMRFunction(torch.autograd.Function):
  """Iterative semi-global matching revised, Jacobi over directions (MP_module.py:89-161)."""

  @staticmethod
  def forward(ctx, unary, label_context, edge_weights, args, cost_labels_first=False):
    n_disp = unary.size(4)
    rho, n_iter, n_dir = args.rho, int(args.mpnet_max_iter), int(args.mpnet_n_dirs)
    buf = _forward_buffers(unary, args, n_dir, n_iter, True, cost_labels_first)
    enable_edge_weights = edge_weights is not None
    if not enable_edge_weights:
      edge_weights = unary.new_ones((n_dir,) + tuple(unary.shape[:4]))
    _ops_for(n_disp).ISGMR.forward(int(args.enable_sgm), rho, n_iter, int(args.enable_min_a_dir),
                                   unary, label_context, edge_weights, buf["message"],
                                   buf["cost_final"], buf["message_index"], buf["cost_index"],
                                   buf["unary_update"], buf["message_tmp"], buf["label_all"],
                                   msg_uninit=True,
                                   flags=_table_flags(args) | (_lib.F_COST_LABELS_FIRST if cost_labels_first else 0))
    ctx.cost_labels_first = cost_labels_first
    ctx.intermediate_results = (args.enable_sgm, rho, buf["message_index"], buf["cost_index"],
                                label_context, edge_weights, enable_edge_weights)
    return buf["cost_final"], buf["label_all"]

  @staticmethod
  def backward(ctx, dcost_final, dmessage_all):
    enable_sgm, rho, message_index, cost_index, label_context, edge_weights, \
        enable_edge_weights = ctx.intermediate_results
    del ctx.intermediate_results
    dcost_final = gradient_labels_last(dcost_final) if ctx.cost_labels_first else dcost_final.contiguous()
    n_disp = message_index.size(6)
    need_context = ctx.needs_input_grad[1]
    need_edge_weights = enable_edge_weights and ctx.needs_input_grad[2]
    buf = _backward_buffers(dcost_final, message_index, True, need_context, need_edge_weights)
    _ops_for(n_disp).ISGMR.backward(int(enable_sgm), rho, label_context, edge_weights,
                                    dcost_final, message_index, cost_index, buf["dunary"],
                                    buf["dlabel_context"], buf["dedge_weights"], buf["dmessage"],
                                    buf["dunary_update"], buf["dmessage_tmp"], flags=buf["flags"])
    return (buf["dunary"], buf["dlabel_context"] if need_context else None,
            buf["dedge_weights"] if need_edge_weights else None, None, None)


def _entries(place):
  """`place` as an index that numpy reads as torch does, None for one that it may read otherwise (bytes, which
  torch takes as a mask, floats and short integers, negative steps, lists of lists) and for tensors."""
  if isinstance(place, tuple):
    parts = tuple(None if isinstance(part, tuple) else _entries(part) for part in place)
    return None if any(part is None for part in parts) else parts
  if isinstance(place, range) or (isinstance(place, list) and all(type(i) is int for i in place)):
    return np.array(place, np.int64)
  if isinstance(place, np.ndarray):
    return place if place.dtype in (np.bool_, np.int32, np.int64) else None
  if isinstance(place, slice):
    return place if place.step is None or place.step > 0 else None
  return place if type(place) is int else None


def _runs_now(tensor):
  """Whether operations on `tensor` run as they are called: no trace, transform, dispatch mode or stream capture
  that could hold on to a tensor kept between calls, or leave one of its own in its place."""
  # (compiling first: the compiler refuses the questions after it)
  return (not torch.compiler.is_compiling() and
          type(tensor) is torch.Tensor and torch._C._len_torch_dispatch_stack() == 0 and
          torch._C._functorch.peek_interpreter_stack() is None and not torch.jit.is_tracing() and
          not (tensor.is_cuda and torch.cuda.is_current_stream_capturing()))


class MPModule(torch.nn.Module):
  """nn.Module wrapper (MP_module.py:164-234).

  Reads from `args`: mpnet_mrf_mode ('TRWP' | 'ISGMR' | 'SGM'), mpnet_max_iter, mpnet_n_dirs,
  n_classes, mpnet_term_weight, mpnet_smoothness_train, mpnet_diag_value, enable_symmetric (and the
  fields create_label_context needs); writes rho (0.5 for TRWP, else 1), enable_saving_label,
  enable_min_a_dir, enable_sgm, enable_seg and, per call, training -- as the reference does.
  """

  def __init__(self, args, enable_create_label_context=False, enable_saving_label=False,
               enable_min_a_dir=False):
    super(MPModule, self).__init__()
    self.args = args
    self.args.rho = 0.5 if (args.mpnet_mrf_mode == 'TRWP') else 1
    self.args.enable_saving_label = enable_saving_label
    self.args.enable_min_a_dir = enable_min_a_dir
    self.args.enable_sgm = args.mpnet_mrf_mode == 'SGM'
    self.args.enable_seg = True if (args.n_classes == 21) else False
    if enable_create_label_context:
      self.create_label_context()

  def _fixed_table_is_dense(self, label_context):
    """Whether the forward scans take their O(L^2) step on the 1-D table the kernels read (the
    first n_classes entries of label_context), asked once per table: the answer is kept until the
    stored table is replaced or written to.  It only matters above 64 labels."""
    n_disp = int(self.args.n_classes)
    if n_disp <= 64 or not label_context.is_cuda:
      return False
    key = (self.label_context.data_ptr(), self.label_context._version)
    if getattr(self, "_dense_key", None) != key:
      if torch.cuda.is_current_stream_capturing():
        return False  # no copy to the host inside a capture; the flag is a hint
      self._dense_key = key
      self._dense_answer = _lib.table_is_dense(label_context.reshape(-1)[:n_disp])
    return self._dense_answer

  def get_label_context(self):
    return self.label_context, self.label_context_loc, self.label_context_diag_loc

  def set_label_context(self, label_context, label_context_loc, label_context_diag_loc):
    self.label_context = label_context
    self.label_context_loc = label_context_loc
    self.label_context_diag_loc = label_context_diag_loc

  def create_label_context(self):
    self.label_context, self.label_context_loc, self.label_context_diag_loc = \
        create_label_context(self.args, enable_seg=self.args.enable_seg,
                             enable_symmetric=self.args.enable_symmetric)

  def __getstate__(self):
    """What copies and files hold of the module: not the masks of this process, whose stream cannot be pickled and
    whose device may be another one after loading."""
    state = self.__dict__.copy()
    state.pop("_kept_masks", None)
    return state

  def _location_masks(self, label_context):
    """Masks of label_context_loc and label_context_diag_loc on the table's device, None where a location is
    not a list of different entries that numpy reads as torch does, or more than one value is pinned, and in
    traces, transforms and captures.  They are formed on the host from the locations of the moment and copied
    only when they differ from what was copied last."""
    if not _runs_now(label_context):
      return None
    diag = self.label_context_diag_loc
    places = [_entries(self.label_context_loc), _entries(tuple(diag) if isinstance(diag, list) else diag)]
    if any(place is None for place in places) or not isinstance(self.args.mpnet_diag_value, (int, float)):
      return None
    host = []
    for index in places:
      mask = np.zeros(label_context.shape, bool)
      taken = mask[index]
      if not host and np.ndim(taken) != 1:
        return None  # (what takes the values back entry by entry is one-dimensional)
      mask[index] = True
      if not host and np.count_nonzero(mask) != np.size(taken):
        return None  # (an entry named twice has its gradient twice)
      host.append(mask)
    key = (label_context.device, label_context.shape) + tuple(mask.tobytes() for mask in host)
    stream = torch.cuda.current_stream(label_context.device) if label_context.is_cuda else None
    kept = getattr(self, "_kept_masks", None)
    if kept is None or kept[0] != key:
      # (copies from pageable memory are complete when they return, for every stream; tensors of inference
      # mode could not be saved for a later call's backward pass)
      with torch.inference_mode(False):
        kept = (key, stream, [torch.from_numpy(mask).to(label_context.device) for mask in host])
      self._kept_masks = kept
    if stream != kept[1]:
      # (their memory goes back to the stream they were formed on when other locations take their place)
      for mask in kept[2]:
        mask.record_stream(stream)
    return kept[2]

  def _effective_label_context(self, weight_first=False):
    """Re-parameterisation of the learned context (MP_module.py:207-220).  weight_first: the term
    weight scales the stored parameter before the re-parameterisation instead of the sigmoid's
    output (the hard/soft module, MP_module_hard_soft.py:148-163)."""
    term_weight = self.args.mpnet_term_weight
    label_context = self.label_context * (term_weight if weight_first else 1)
    mode = self.args.mpnet_smoothness_train
    scale = 2 if weight_first else 2 * term_weight
    masks = self._location_masks(label_context) if mode == 'sigmoid' else None
    if masks is not None:
      # entry by entry: indexing with the stored locations copies them to the device in every call, waits for
      # each copy, and sorts them for the gradient
      learned, pinned = masks
      valid = label_context.masked_fill(~learned, 0)
      label_context = torch.where(learned, scale * torch.sigmoid(valid), label_context)
      return label_context.masked_fill(pinned, self.args.mpnet_diag_value)
    if mode == 'sigmoid':
      valid = label_context[self.label_context_loc].flatten()
      label_context[self.label_context_loc] = scale * torch.sigmoid(valid)
    elif mode == 'softmax':
      valid = label_context[self.label_context_loc].flatten()
      norm = nn.Softmax(dim=0)(valid)
      label_context[self.label_context_loc] = norm * valid.max() / norm.max()
    if mode in {'sigmoid', 'softmax'}:
      diag = self.label_context_diag_loc
      label_context[tuple(diag) if isinstance(diag, list) else diag] = self.args.mpnet_diag_value
    return label_context

  def forward(self, unary, edge_weights=None):
    # label axis innermost for the kernels; direction axis outermost for the edge weights
    unary = labels_last(unary)
    if edge_weights is not None:
      edge_weights = edge_weights.unsqueeze(1).permute(2, 0, 1, 3, 4).contiguous()
      assert unary.size()[-3:-1] == edge_weights.size()[-2:]
    if unary.is_cuda and (self.args.mpnet_mrf_mode == 'SGM'):
      assert self.args.mpnet_max_iter == 1
    label_context = self._effective_label_context()
    self.args.training = self.training
    # a table that is being learned is dense in general and a fixed one is looked at once, on the
    # host; args.mpnet_dense_table overrides both
    dense = getattr(self.args, "mpnet_dense_table", None)
    if dense is None:
      dense = self.label_context.requires_grad or self._fixed_table_is_dense(label_context)
    self.args.dense_table = bool(dense)
    turned = _sums_labels_first(unary, self.args)
    if self.args.mpnet_mrf_mode in {'ISGMR', 'SGM'}:
      cost_final, cost_all = ISGMRFunction.apply(unary, label_context, edge_weights, self.args, turned)
    elif self.args.mpnet_mrf_mode == 'TRWP':
      cost_final, cost_all = TRWPFunction.apply(unary, label_context, edge_weights, self.args, turned)
    else:
      assert False
    if not turned:
      cost_final = labels_first(cost_final)
    return cost_final, label_context.unsqueeze(0), cost_all, None, None
