"""Serving steps with more than single tokens: portions of prompts on the one-wave-per-SIMD attention kernel over block tables
(csrc/kernels/flash_attn_w64.hip), single tokens on the split-key kernel (csrc/kernels/paged_attn.hip)."""
import torch

from . import native
from .paged import DECODE_MAX

# new tokens of a workgroup of the prefill kernel
PREFILL_ROWS = 256


def make_portions(seq_meta_host):
    """How a step with more than single tokens is divided: (rows of the tokens that run one by one, flat list of (sequence,
    first new token) of the prefill kernel's workgroups, those that see the most keys first)."""
    toks, blocks = [], []
    for s, (q0, n, seen) in enumerate(seq_meta_host):
        if n <= DECODE_MAX:
            toks += range(q0, q0 + n)
        else:
            blocks += [(seen + min(r + PREFILL_ROWS, n), s, r) for r in range(0, n, PREFILL_ROWS)]
    blocks.sort(reverse=True)
    return toks, [v for b in blocks for v in b[1:]]


def portions_ok(q, cache, n_q, n_kv):
    """Does the prefill kernel take these heads and this cache?"""
    return (native.use_native(q) and q.dtype == torch.bfloat16 and cache.dtype == q.dtype and cache.dim() == 5
            and q.shape[2] == 128 and cache.is_contiguous() and cache.shape[1] % 64 == 0 and n_q % n_kv == 0
            and cache.shape[0] * cache.shape[1] < 2**31 and cache.stride(0) // cache.shape[1] <= 2**23
            and q.stride(0) % 8 == 0 and q.stride(1) == 128 and q.data_ptr() % 16 == 0)


def paged_attention_portions(q, cache, toks, blocks, batch, n_q, n_kv, scale, window=0):
    """``paged_attention`` of a step that mixes single tokens and portions of prompts: ``toks`` (int32 rows of q) on the
    split-key kernel, which spreads a token's context over the chip, ``blocks`` ([n, 2] int32) on the prefill kernel. In
    row blocks of the matrix-core kernel a single token walks its whole context in one workgroup (9 such tokens, up to 3,000
    keys, 8 key heads, beside 512 new ones: 171 us; apart 29 + 38 us)."""
    T, _, D = q.shape
    o = torch.empty(T, n_q, D, device=q.device, dtype=q.dtype)
    lib, st, tab = native.kernels(), native.stream(), batch.block_tables
    mb, bs = tab.shape[1], cache.shape[1]
    n = 0 if toks is None else toks.numel()
    if n:
        keys = mb * bs
        splits = lib.hds_paged_decode_splits(n, n_kv, min(keys, window) if window else keys)
        part_o = part_ml = None
        if splits > 1:
            part_o = torch.empty(n * n_q * splits * D, device=q.device, dtype=torch.float32)
            part_ml = torch.empty(n * n_q * splits * 2, device=q.device, dtype=torch.float32)
        native.check(
            lib.hds_paged_decode(native.dt(q), 0, q.data_ptr(), q.stride(0), cache.data_ptr(), o.data_ptr(), n_q * D,
                                 native.ptr(part_o), native.ptr(part_ml), None, toks.data_ptr(),
                                 batch.tok_seq.data_ptr(), batch.tok_pos.data_ptr(), tab.data_ptr(), mb, bs, n, n_q,
                                 n_kv, D, D, splits, float(scale), int(window), 0, 0, 0.0, None, None, 0, 1, None, st),
            "paged_decode")
    if blocks is not None and blocks.shape[0]:
        native.check(
            lib.hds_paged_prefill(q.data_ptr(), q.stride(0), cache.data_ptr(), o.data_ptr(), n_q * D,
                                  blocks.data_ptr(), blocks.shape[0], batch.seq_meta.data_ptr(), tab.data_ptr(), mb, bs,
                                  n_q, n_kv, float(scale), int(window), st), "paged_prefill")
    return o
