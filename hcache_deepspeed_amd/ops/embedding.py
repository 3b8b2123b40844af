"""Token embedding whose weight gradient is scatter-added in place (csrc/kernels/token_ops.hip embed_bwd_kernel).

The framework's default ``nn.Embedding`` backward sorts the ids, reduces duplicates into a DENSE [V, D]
gradient (fill + compute_grad_weight + sum_and_scatter) and AccumulateGrad then adds that whole tensor into
``.grad`` -- for Llama-3 (V=128256, D=4096) three passes over 1 GB per micro-step. Here the ids are sorted
once (4,096 and fewer are compared with each other instead) and one HIP workgroup per distinct id adds its tokens' rows straight into the parameter's gradient
buffer (the flat ZeRO buffer), touching only the rows that occur. Reference counterpart: the embedding of
every model trained through ``deepspeed.initialize`` (the reference uses the framework kernel).

CPU tensors use ``index_add_`` (the numerics reference of the tests).
"""
import types

import torch
import torch.nn as nn
import torch.nn.functional as F

from . import native
from ..offload import act_plan as _ap


def embedding_grad_add_(grad, ids, dy, padding_idx=None):
    """grad[ids[t]] += dy[t] for every token t (rows equal to ``padding_idx`` skipped); deterministic."""
    V, D = grad.shape
    ids = ids.reshape(-1)
    dy = dy.reshape(-1, D)
    if native.use_native(grad) and D % 8 == 0 and dy.dtype == grad.dtype and \
            grad.dtype in (torch.float32, torch.bfloat16, torch.float16) and grad.is_contiguous():
        dy = dy.contiguous()
        pad = -1 if padding_idx is None else int(padding_idx) % V
        lib = native.kernels()
        if ids.numel() <= lib.hds_embed_bwd_few_max():
            ids = ids.to(torch.int64).contiguous()
            native.check(lib.hds_embed_bwd_few(native.dt(grad), dy.data_ptr(), ids.data_ptr(), grad.data_ptr(), ids.numel(), D,
                                               V, pad, native.stream()), "embed_bwd_few")
            return grad
        srt, perm = torch.sort(ids.to(torch.int64), stable=True)
        native.check(lib.hds_embed_bwd(native.dt(grad), dy.data_ptr(), srt.data_ptr(), perm.data_ptr(), grad.data_ptr(),
                                       ids.numel(), D, V, pad, native.stream()), "embed_bwd")
        return grad
    if padding_idx is not None:
        keep = ids != (int(padding_idx) % V)
        ids, dy = ids[keep], dy[keep]
    grad.index_add_(0, ids.to(torch.int64), dy.to(grad.dtype))
    return grad


def lookup_rows(table, ids):
    """``F.embedding(ids, table)``, on the GPU by a kernel of one launch for tables without a gradient whose rows are whole
    16-byte pieces. Ids outside the table, which a caller with ids on the host refuses, give NaN rows there."""
    row = table.shape[-1] * table.element_size()
    if native.use_native(table) and table.dim() == 2 and ids.dim() == 1 and ids.dtype == torch.int64 and \
            ids.device == table.device and table.is_floating_point() and row % 16 == 0 and \
            16 <= row <= 16 * 256 * 65535 and ids.is_contiguous() and table.is_contiguous() and \
            table.data_ptr() % 16 == 0 and not (torch.is_grad_enabled() and table.requires_grad):
        out = torch.empty(ids.numel(), table.shape[1], dtype=table.dtype, device=table.device)
        native.check(native.kernels().hds_gather_rows(table.data_ptr(), ids.data_ptr(), out.data_ptr(), ids.numel(), row,
                                                      table.shape[0], native.stream()), "gather_rows")
        return out
    return F.embedding(ids, table)


def norm_rows(table, ids, weight, eps):
    """(``lookup_rows(table, ids)``, the RMS norm of those rows) by one kernel, or None where it does not take the call."""
    if not (native.use_native(table) and native.plain(table, ids, weight) and not _ap.tracking()):
        return None
    if not (table.dim() == 2 and ids.dim() == weight.dim() == 1 and ids.dtype == torch.int64
            and table.device == ids.device == weight.device and weight.dtype == table.dtype
            and table.dtype in (torch.float32, torch.bfloat16, torch.float16)
            and 0 < ids.numel() < 1 << 28 and 0 < table.shape[0] < 1 << 31 and table.shape[1] == weight.shape[0] < 1 << 20
            and table.shape[1] % 8 == 0 and table.shape[1] > 0
            and table.is_contiguous() and ids.is_contiguous() and weight.is_contiguous()
            and table.data_ptr() % 16 == 0 and weight.data_ptr() % 16 == 0):
        return None
    h = torch.empty(ids.numel(), table.shape[1], dtype=table.dtype, device=table.device)
    y = torch.empty_like(h)
    native.check(native.kernels().hds_embed_norm(native.dt(table), table.data_ptr(), ids.data_ptr(), weight.data_ptr(),
                                                 h.data_ptr(), y.data_ptr(), ids.numel(), table.shape[1], table.shape[0],
                                                 float(eps), native.stream()), "embed_norm")
    return h, y


class EmbeddingFunction(torch.autograd.Function):

    @staticmethod
    def forward(ctx, ids, weight, padding_idx):
        ctx.save_for_backward(ids)
        ctx.weight = weight  # the Parameter object: under ZeRO-3 its storage is re-gathered for backward
        ctx.shape = tuple(weight.shape)
        ctx.padding_idx = padding_idx
        return F.embedding(ids, weight, padding_idx)

    @staticmethod
    def backward(ctx, dy):
        from ..runtime.zero.linear import grad_accumulator
        (ids, ) = ctx.saved_tensors
        if not ctx.needs_input_grad[1]:
            return None, None, None
        g = grad_accumulator(ctx.weight, dy.dtype)
        if g is not None:
            embedding_grad_add_(g.view(ctx.shape), ids, dy, ctx.padding_idx)
            return None, None, None
        dw = torch.zeros(ctx.shape, dtype=dy.dtype, device=dy.device)
        return None, embedding_grad_add_(dw, ids, dy, ctx.padding_idx), None


def _emb_forward(self, ids):
    return EmbeddingFunction.apply(ids, self.weight, self.padding_idx)


def wrap_embeddings(module, only=None):
    """Route plain dense nn.Embedding modules under ``module`` (or those whose weight id is in ``only``) through
    :class:`EmbeddingFunction` (instance-level forward override)."""
    n = 0
    for m in module.modules():
        if isinstance(m, nn.Embedding) and not getattr(m, "_hds_emb", False) and not m.sparse and \
                m.max_norm is None and not m.scale_grad_by_freq and (only is None or id(m.weight) in only):
            m.forward = types.MethodType(_emb_forward, m)
            m._hds_emb = True
            n += 1
    return n
