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


@pytest.mark.parametrize("D,nq,nkv,turn", [(256, 16, 1, 16), (256, 8, 8, 32), (64, 34, 2, 64), (64, 2, 2, 128), (80, 2, 2, 64)])
def test_decode_splits_of_one_turn(D, nq, nkv, turn):
    """Lengths around one and two turns of a workgroup of the vector kernel, where the number of splits with keys changes."""
    lens = [1, turn - 1, turn, turn + 1, 2 * turn - 1, 2 * turn, 2 * turn + 1, 9 * turn + 3]
    scale = D**-0.5
    cache, tables, meta, qkv = _setup(lens, nq, nkv, D, 64, 20, seed=4)
    seq = torch.arange(len(lens), dtype=torch.int32, device="cuda")
    kv_rope_scatter(qkv, cache, seq, meta[:, 2].contiguous(), tables, None, None, nq, nkv, do_rope=False)
    got = paged_attention(qkv[:, :nq], cache, None, 0, meta, tables, nq, nkv, scale, decode=True)
    ref = _exact(qkv[:, :nq], cache, tables, lens, nq, nkv, scale, 0)
    # one rounding of the result; 32-bit sums and exponentials in front of it (|v| <= 6)
    assert ((got.double() - ref).abs() <= 2**-8 * ref.abs() + 2e-4).all()


@pytest.mark.parametrize("nq,nkv,line", [(8, 8, 32), (32, 16, 64)])
@pytest.mark.parametrize("over", [0, 1])
@pytest.mark.parametrize("window", [0, 33])
def test_few_query_heads_a_key_head_on_both_kernels(nq, nkv, line, over, window):
    """One token below the number from which the vector kernel is the faster one, and at it: the same step by both ways.
    Without rotation: the two rotations may round an element differently, and both kernels are to see the same numbers."""
    T, D, scale = line - 1 + over, 128, 0.11
    lens = [1 + 7 * (i % 23) for i in range(T)]
    cache, tables, meta, qkv = _setup(lens, nq, nkv, D, 32, 5, seed=5)
    seq = torch.arange(T, dtype=torch.int32, device="cuda")
    want_cache, want_qkv = cache.clone(), qkv.clone()
    kv_rope_scatter(want_qkv, want_cache, seq, meta[:, 2].contiguous(), tables, None, None, nq, nkv, do_rope=False)
    ref = _exact(want_qkv[:, :nq], want_cache, tables, lens, nq, nkv, scale, window)
    plain = paged_attention(want_qkv[:, :nq], want_cache, None, 0, meta, tables, nq, nkv, scale, window, decode=True)
    fused = paged_decode_qkv(qkv, cache, meta, tables, nq, nkv, scale, window, None, None)
    assert decode_qkv_ok(qkv, cache, nq, nkv, None, None) == (over == 0)
    for got in (plain, fused):  # one rounding of the result; 32-bit sums and exponentials in front of it (|v| <= 6)
        assert ((got.double() - ref).abs() <= 2**-8 * ref.abs() + 2e-4).all()


@pytest.mark.parametrize("sink", [False, True])
@pytest.mark.parametrize("gate_width", [0, 1, 128])
@pytest.mark.parametrize("window", [0, 50])
@pytest.mark.parametrize("rows", [False, True])
@pytest.mark.parametrize("splits", [1, 7])
def test_matrix_core_kernel_against_the_plain_one(sink, gate_width, window, rows, splits):
    """Every option that the rule for the matrix-core kernel lets through, on both kernels of the same entry point: a sink, a
    gate a head or an element, a window, one token of each sequence or chosen rows of a step, strided rows."""
    from hcache_deepspeed_amd.ops import native
    lib, nq, nkv, D, bs, mb = native.kernels(), 12, 3, 128, 64, 8
    lens = [1, 40, 64, 333, 500]
    cache, tables, meta, qkv = _setup(lens, nq, nkv, D, bs, mb, seed=2)
    g = torch.Generator(device="cuda").manual_seed(3)
    seq = torch.arange(len(lens), dtype=torch.int32, device="cuda")
    pos = meta[:, 2].contiguous()
    kv_rope_scatter(qkv, cache, seq, pos, tables, None, None, nq, nkv, do_rope=False)
    toks = torch.tensor([4, 0, 3], dtype=torch.int32, device="cuda") if rows else None
    n = 3 if rows else len(lens)
    sinks = torch.randn(nq, device="cuda", generator=g) if sink else None
    gate = torch.randn(len(lens), max(1, nq * gate_width) + 8, device="cuda", generator=g).to(torch.bfloat16) if gate_width else None
    out = []
    for plain in (0, 1):
        o = torch.zeros(len(lens), nq * D + 8, device="cuda", dtype=torch.bfloat16)
        po = torch.empty(n * nq * splits * D, device="cuda")
        pm = torch.empty(n * nq * splits * 2, device="cuda")
        native.check(
            lib.hds_paged_decode(native.dt(qkv), plain, qkv.data_ptr(), qkv.stride(0), cache.data_ptr(), o.data_ptr(),
                                 o.stride(0), po.data_ptr(), pm.data_ptr(), None if rows else meta.data_ptr(),
                                 native.ptr(toks), seq.data_ptr(), pos.data_ptr(), tables.data_ptr(), mb, bs, n, nq, nkv, D,
                                 D, splits, 0.09, window, 0, 0, 0.0, native.ptr(sinks), native.ptr(gate),
                                 0 if gate is None else gate.stride(0), max(1, gate_width), None, native.stream()), "decode")
        out.append(o.float())
    a, b = out
    # both sum in 32 bits and round once
    assert ((a - b).abs() <= 2**-7 * b.abs() + 2e-4).all() and a.abs().sum() > 0


@pytest.mark.parametrize("bs,mb", [(32, 520), (96, 174)])
@pytest.mark.parametrize("window", [0, 8200])
def test_splits_of_more_tiles_than_a_wave_looks_up_at_once(bs, mb, window):
    """One split for the whole sequence: around 64 and 128 tiles a wave, whose places it looks up 64 at a time."""
    from hcache_deepspeed_amd.ops import native
    lens, nq, nkv, D = [8161, 8192, 8193, 8320, 16400, 16600], 4, 1, 128
    cache, tables, meta, qkv = _setup(lens, nq, nkv, D, bs, mb, seed=4)
    seq = torch.arange(len(lens), dtype=torch.int32, device="cuda")
    kv_rope_scatter(qkv, cache, seq, meta[:, 2].contiguous(), tables, None, None, nq, nkv, do_rope=False)
    o = torch.zeros(len(lens), nq * D, device="cuda", dtype=torch.bfloat16)
    native.check(
        native.kernels().hds_paged_decode(native.dt(qkv), 0, qkv.data_ptr(), qkv.stride(0), cache.data_ptr(), o.data_ptr(), o.stride(0),
                                          None, None, meta.data_ptr(), None, None, None, tables.data_ptr(), mb, bs, len(lens), nq,
                                          nkv, D, D, 1, 0.09, window, 0, 0, 0.0, None, None, 0, 1, None, native.stream()), "decode")
    ref = _exact(qkv[:, :nq], cache, tables, lens, nq, nkv, 0.09, window)
    assert ((o.view(-1, nq, D).double() - ref).abs() <= 2**-8 * ref.abs() + 2e-4).all()


@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("splits", [8, 16, 24, 63, 64])
def test_rounds_of_splits(D, splits):
    """Splits in whole rounds of 8 and others, most of them without keys, on both kernels against 64 bits."""
    from hcache_deepspeed_amd.ops import native
    lens, nq, nkv, bs, mb = [1, 130, 3000, 257, 2049], 12, 3, 64, 48
    cache, tables, meta, qkv = _setup(lens, nq, nkv, D, bs, mb, seed=5)
    seq = torch.arange(len(lens), dtype=torch.int32, device="cuda")
    kv_rope_scatter(qkv, cache, seq, meta[:, 2].contiguous(), tables, None, None, nq, nkv, do_rope=False)
    o = torch.zeros(len(lens), nq * D, device="cuda", dtype=torch.bfloat16)
    po, pm = (torch.empty(len(lens) * nq * splits * w, device="cuda") for w in (D, 2))
    native.check(
        native.kernels().hds_paged_decode(native.dt(qkv), 0, qkv.data_ptr(), qkv.stride(0), cache.data_ptr(), o.data_ptr(), o.stride(0),
                                          po.data_ptr(), pm.data_ptr(), meta.data_ptr(), None, None, None, tables.data_ptr(), mb, bs,
                                          len(lens), nq, nkv, D, D, splits, 0.09, 0, 0, 0, 0.0, None, None, 0, 1, None, native.stream()),
        "decode")
    ref = _exact(qkv[:, :nq], cache, tables, lens, nq, nkv, 0.09, 0)
    assert ((o.view(-1, nq, D).double() - ref).abs() <= 2**-8 * ref.abs() + 2e-4).all()
