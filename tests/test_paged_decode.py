"""Decode attention over the paged cache: the matrix-core kernel (heads of 128), with and without the rotation and the
append in front of it, and the merge of key splits, against 64 bits."""
import pytest
import torch

from hcache_deepspeed_amd.ops.paged import decode_qkv_ok, kv_rope_scatter, paged_attention, paged_decode_qkv
from hcache_deepspeed_amd.ops.rope import rope_tables

pytestmark = pytest.mark.gpu
EDGES = [1, 2, 31, 32, 33, 64, 65, 128, 129, 257, 1000]  # keys a token sees


def _setup(lens, nq, nkv, D, bs, mb, seed=0):
    g = torch.Generator(device="cuda").manual_seed(seed)
    S = len(lens)
    cache = torch.full((S * mb + 1, bs, 2, nkv, D), float("nan"), device="cuda", dtype=torch.bfloat16)
    tables = (torch.randperm(S * mb, device="cuda", generator=g) + 1).to(torch.int32).view(S, mb)
    for i, n in enumerate(lens):  # the tokens before the step; every other place holds NaN
        rows = torch.randn(n - 1, 2, nkv, D, device="cuda", generator=g).to(torch.bfloat16)
        for j in range(0, n - 1, bs):
            cache[tables[i, j // bs].item(), :min(bs, n - 1 - j)] = rows[j:j + bs]
    meta = torch.tensor([[i, 1, n - 1] for i, n in enumerate(lens)], dtype=torch.int32, device="cuda")
    qkv = torch.randn(S, nq + 2 * nkv, D, device="cuda", generator=g).to(torch.bfloat16)
    return cache, tables, meta, qkv


def _exact(q, cache, tables, lens, nq, nkv, scale, window):
    out, G = [], nq // nkv
    for i, n in enumerate(lens):
        kv = cache[tables[i].long()].flatten(0, 1)[:n][max(0, n - window) if window else 0:].double()
        k, v = (kv[:, j].repeat_interleave(G, 1).transpose(0, 1) for j in (0, 1))
        p = torch.softmax((k @ q[i].double()[:, :, None])[:, :, 0] * scale, -1)
        out.append((p[:, None] @ v)[:, 0])
    return torch.stack(out)


@pytest.mark.parametrize("nq,nkv", [(1, 1), (8, 2), (24, 3), (16, 1)])
@pytest.mark.parametrize("bs,mb", [(32, 33), (64, 64), (96, 11)])
@pytest.mark.parametrize("window", [0, 33, 200])
@pytest.mark.parametrize("rot", [128, 64, None])
def test_decode_from_the_projection(nq, nkv, bs, mb, window, rot):
    """Lengths around a tile of 32, a workgroup's turn and a block; places outside a sequence hold NaN."""
    D, scale = 128, 0.11
    cache, tables, meta, qkv = _setup(EDGES, nq, nkv, D, bs, mb)
    cos, sin = rope_tables(2048, rot or D, 10000.0, device="cuda")
    if rot is None:
        cos = sin = None
    seq = torch.arange(len(EDGES), dtype=torch.int32, device="cuda")
    pos = meta[:, 2].contiguous()
    want_cache, want_qkv = cache.clone(), qkv.clone()
    kv_rope_scatter(want_qkv, want_cache, seq, pos, tables, cos, sin, nq, nkv, do_rope=rot is not None, rotary_dim=rot or 0)
    assert decode_qkv_ok(qkv, cache, nq, nkv, cos, sin, rot or 0)
    got = paged_decode_qkv(qkv, cache, meta, tables, nq, nkv, scale, window, cos, sin, rot or 0)
    same = (cache == want_cache) | (cache.isnan() & want_cache.isnan())
    # the same products and sums: at most the fused multiply-add falls elsewhere
    assert same.all() or (cache - want_cache).abs()[~same].le(2**-7 * want_cache.abs()[~same]).all()
    ref = _exact(want_qkv[:, :nq], want_cache, tables, EDGES, nq, nkv, scale, window)
    # one rounding of the result; 32-bit sums and exponentials in front of it (|v| <= 6)
    assert ((got.double() - ref).abs() <= 2**-8 * ref.abs() + 2e-4).all()
    plain = paged_attention(want_qkv[:, :nq], want_cache, None, 0, meta, tables, nq, nkv, scale, window, decode=True)
    assert ((plain.double() - ref).abs() <= 2**-8 * ref.abs() + 2e-4).all()


@pytest.mark.parametrize("D,nq,nkv", [(64, 8, 2), (80, 6, 6), (128, 34, 2), (256, 4, 1), (128, 4, 4)])
@pytest.mark.parametrize("lens,mb", [([1, 63, 64, 65, 300], 8), ([4000], 64), ([700] * 40, 16)])
def test_decode_splits_and_merge(D, nq, nkv, lens, mb):
    """Splits that get no keys, one split, 64 of them; the vector kernel's sizes too (more than 16 query heads a key head)."""
    scale = D**-0.5
    cache, tables, meta, qkv = _setup(lens, nq, nkv, D, 64, mb, seed=1)
    seq = torch.arange(len(lens), dtype=torch.int32, device="cuda")
    kv_rope_scatter(qkv, cache, seq, meta[:, 2].contiguous(), tables, None, None, nq, nkv, do_rope=False)
    got = paged_attention(qkv[:, :nq], cache, None, 0, meta, tables, nq, nkv, scale, decode=True)
    ref = _exact(qkv[:, :nq], cache, tables, lens, nq, nkv, scale, 0)
    assert ((got.double() - ref).abs() <= 2**-8 * ref.abs() + 2e-4).all()
