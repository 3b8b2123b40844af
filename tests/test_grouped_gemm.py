"""Grouped (MoE) GEMM (csrc/kernels/grouped_gemm.hip) and the dropless MoE FFN against fp32 torch references.

Reference test model: tests/unit/inference/v2/kernels/cutlass_ops/test_moe_gemm.py (grouped GEMM with ragged
per-expert token counts, including empty experts, vs per-expert torch matmuls).
"""
import pathlib
import re

import pytest
import torch

from hcache_deepspeed_amd.ops.activations import glu
from hcache_deepspeed_amd.ops.grouped_gemm import expert_offsets, grouped_gemm, moe_ffn_dropless
from hcache_deepspeed_amd.ops.moe import moe_combine, moe_dispatch, topk_assign, topk_route


def _ref(x, w, counts):
    out, o = [], 0
    for e, c in enumerate(counts):
        out.append(x[o:o + c].float() @ w[e].float().t())
        o += c
    return torch.cat(out)


def _bmm_moe(x, logits, k, w13, w2):
    E, H = w13.shape[0], x.shape[1]
    ex, pos, w, C, _, _ = topk_route(logits, k, 1.0, 1, drop_tokens=False, use_rts=False, training=False)
    d = moe_dispatch(x, ex, pos, E, C).view(E, C, H)
    h = torch.bmm(d, w13.transpose(1, 2))
    y = torch.bmm(glu(h.reshape(E * C, -1), "silu").view(E, C, -1), w2.transpose(1, 2))
    return moe_combine(y.reshape(E * C, H), ex, pos, w, C)


def test_dropless_moe_matches_capacity_formulation_cpu():
    torch.manual_seed(0)
    T, H, I, E, k = 37, 16, 24, 4, 2
    x, logits = torch.randn(T, H), torch.randn(T, E)
    w13, w2 = torch.randn(E, 2 * I, H) * 0.1, torch.randn(E, H, I) * 0.1
    ex, pos, w, counts = topk_assign(logits, k)
    out = moe_ffn_dropless(x, ex, pos, w, counts, w13, w2, lambda h: glu(h, "silu"))
    torch.testing.assert_close(out, _bmm_moe(x, logits, k, w13, w2), atol=1e-5, rtol=1e-5)


def test_grouped_gemm_autograd_cpu():
    torch.manual_seed(1)
    counts = [5, 0, 9, 3]
    x = torch.randn(sum(counts), 8, requires_grad=True)
    w = torch.randn(4, 6, 8, requires_grad=True)
    y = grouped_gemm(x, w, expert_offsets(torch.tensor(counts)))
    g = torch.randn_like(y)
    (y * g).sum().backward()
    xr, wr = x.detach().clone().requires_grad_(True), w.detach().clone().requires_grad_(True)
    (_ref(xr, wr, counts) * g).sum().backward()
    torch.testing.assert_close(x.grad, xr.grad)
    torch.testing.assert_close(w.grad, wr.grad)


@pytest.mark.gpu
@pytest.mark.parametrize("variant", [1, 2])
@pytest.mark.parametrize("counts,N,K", [([300, 0, 1, 129, 128, 77], 256, 384), ([4096, 2048], 512, 1024),
                                        ([0, 0, 3], 256, 128), ([513, 255, 256, 1000], 768, 256)])
def test_grouped_gemm_hip(cuda, counts, N, K, variant):
    torch.manual_seed(2)
    E, T = len(counts), sum(counts)
    x = torch.randn(T, K, device=cuda, dtype=torch.bfloat16)
    w = torch.randn(E, N, K, device=cuda, dtype=torch.bfloat16) / K**0.5
    y = grouped_gemm(x, w, expert_offsets(torch.tensor(counts, device=cuda)), variant=variant)
    ref = _ref(x, w, counts)
    assert y.dtype == torch.bfloat16
    torch.testing.assert_close(y.float(), ref, atol=2e-2, rtol=2e-2)


@pytest.mark.gpu
def test_grouped_gemm_backward_hip(cuda):
    torch.manual_seed(3)
    counts = [200, 57, 0, 311]
    x = torch.randn(sum(counts), 256, device=cuda, dtype=torch.bfloat16, requires_grad=True)
    w = (torch.randn(4, 384, 256, device=cuda, dtype=torch.bfloat16) / 16).requires_grad_(True)
    y = grouped_gemm(x, w, expert_offsets(torch.tensor(counts, device=cuda)))
    g = torch.randn_like(y)
    (y.float() * g.float()).sum().backward()
    xr, wr = x.detach().float().requires_grad_(True), w.detach().float().requires_grad_(True)
    (_ref(xr, wr, counts) * g.float()).sum().backward()
    torch.testing.assert_close(x.grad.float(), xr.grad, atol=5e-2, rtol=3e-2)
    torch.testing.assert_close(w.grad.float(), wr.grad, atol=5e-2, rtol=3e-2)


@pytest.mark.gpu
def test_dropless_moe_hip(cuda):
    torch.manual_seed(4)
    T, H, I, E, k = 333, 256, 384, 8, 2
    x = torch.randn(T, H, device=cuda, dtype=torch.bfloat16)
    logits = torch.randn(T, E, device=cuda)
    w13 = torch.randn(E, 2 * I, H, device=cuda, dtype=torch.bfloat16) / 16
    w2 = torch.randn(E, H, I, device=cuda, dtype=torch.bfloat16) / 20
    ex, pos, w, counts = topk_assign(logits, k)
    out = moe_ffn_dropless(x, ex, pos, w, counts, w13, w2, lambda h: glu(h, "silu"))
    ref = _bmm_moe(x.float().cpu(), logits.cpu(), k, w13.float().cpu(), w2.float().cpu())
    torch.testing.assert_close(out.float().cpu(), ref, atol=3e-2, rtol=3e-2)


@pytest.mark.gpu
@pytest.mark.parametrize("counts", [[1], [0, 64, 65, 0, 1, 128], [129, 192, 193, 3], [255, 256, 257, 0], [700, 20, 513],
                                    [1100, 1030]])
@pytest.mark.parametrize("N,K", [(128, 128), (384, 256), (256, 1152)])
@pytest.mark.parametrize("gather,glu", [(False, False), (True, True), (True, False), (False, True)])
def test_experts_gemm_hip(cuda, counts, N, K, gather, glu):
    """The serving products over a ready tile list: one to four blocks of 64 rows a tile, several tiles an expert, empty
    experts, more tile slots than tiles, 256 x 256 tiles from 512 rows an expert on (the last counts; N % 256 == 0)."""
    from hcache_deepspeed_amd.ops import native
    lib = native.kernels()
    E, T, tm = len(counts), sum(counts), lib.hds_experts_gemm_tile()
    g = torch.Generator(device="cuda").manual_seed(T + N + K)
    n_src = T + 5 if gather else T
    x = torch.randn(n_src, K + 8, device="cuda", generator=g).to(torch.bfloat16)[:, :K]
    w = (torch.randn(E, (2 if glu else 1) * N, K, device="cuda", generator=g) * K**-0.5).to(torch.bfloat16)
    src = torch.randint(0, n_src, (T, ), device="cuda", generator=g).to(torch.int32) if gather else None
    weight = torch.rand(T, device="cuda", generator=g) if glu else None
    offs = [0]
    tiles = []
    for e, c in enumerate(counts):
        offs.append(offs[-1] + c)
        tiles += [(e, m) for m in range(0, c, tm)]
    slots = T // tm + min(E, T) + 1
    i32 = lambda v: torch.tensor(v, dtype=torch.int32, device="cuda")  # noqa: E731
    pad = [(0, 0)] * (slots - len(tiles))
    te, tmm = (i32([t[j] for t in tiles + pad]) for j in (0, 1))
    nt, of = i32([len(tiles)]), i32(offs)
    y = torch.full((T, N + 8), float("nan"), device="cuda", dtype=torch.bfloat16)
    native.check(
        lib.hds_experts_gemm(x.data_ptr(), x.stride(0), native.ptr(src), n_src, w.data_ptr(), y.data_ptr(), N + 8,
                             of.data_ptr(), te.data_ptr(), tmm.data_ptr(), nt.data_ptr(), slots, T, N, K, E, int(glu), 0,
                             0.0, native.ptr(weight), native.stream()), "experts_gemm")
    rows = (x if src is None else x[src.long()]).double()
    z = torch.cat([rows[offs[e]:offs[e + 1]] @ w[e].double().t() for e in range(E)])
    mag = torch.cat([rows[offs[e]:offs[e + 1]].abs() @ w[e].double().abs().t() for e in range(E)]) * (2**-24 * 8 * K**0.5)
    if glu:
        f = weight.double()[:, None]
        gate, up = z[:, :N] * f, z[:, N:] * f
        ref = torch.nn.functional.silu(gate) * up
        bound = 2**-8 * ref.abs() + 1.13 * f * (mag[:, :N] * up.abs() + mag[:, N:] * gate.abs()) + 1e-5 * ref.abs() + 1e-6
    else:
        ref, bound = z, 2**-8 * z.abs() + mag
    assert ((y[:, :N].double() - ref).abs() <= bound).all() and y[:, N:].isnan().all()


@pytest.mark.gpu
@pytest.mark.parametrize("counts", [[129, 192, 193, 3], [64, 1, 256, 65]])
@pytest.mark.parametrize("N,K,gather,glu", [(4096, 128, True, True), (8192, 384, False, True), (16384, 128, True, False),
                                            (8192, 256, False, False), (4096, 2048, True, True), (8192, 2048, False, False),
                                            (1024, 4096, False, False), (512, 4096, True, True)])
def test_experts_gemm_tiles_of_weight_rows(cuda, counts, N, K, gather, glu):
    """128 and 256 weight rows a tile, which many rounds choose, with one to four blocks of 64 rows; fewer steps than the ring
    holds; walks along K that begin apart."""
    test_experts_gemm_hip(cuda, counts, N, K, gather, glu)


@pytest.mark.gpu
@pytest.mark.parametrize("N,K,gather,glu", [(8192, 384, False, True), (16384, 128, True, False), (4096, 2048, True, True),
                                            (8192, 2048, False, False), (1024, 4096, False, False)])
def test_experts_gemm_weights_of_several_row_tiles(cuda, N, K, gather, glu):
    """More rows an expert than a tile holds: weights through the caches, whatever the tile of weight rows."""
    test_experts_gemm_hip(cuda, [300, 420], N, K, gather, glu)


@pytest.mark.gpu
@pytest.mark.parametrize("E,k,T,N,K,glu,rows,apart", [
    (8, 2, 66, 14336, 4096, 1, 128, 1), (8, 2, 300, 14336, 4096, 1, 256, 0), (16, 4, 66, 6400, 4096, 1, 128, 1),
    (4, 1, 66, 8192, 4096, 1, 256, 1), (64, 6, 66, 1024, 2048, 1, 256, 1), (64, 6, 3000, 1024, 2048, 1, 256, 0),
    (8, 2, 66, 2048, 5632, 0, 64, 0), (8, 2, 900, 2048, 5632, 0, 128, 0), (8, 2, 1000, 3072, 8192, 0, 128, 0),
    (16, 4, 1000, 4096, 6400, 0, 128, 0), (16, 2, 66, 4096, 4096, 0, 256, 1), (16, 2, 1000, 4096, 8192, 0, 256, 0),
    (64, 4, 200, 4096, 2048, 0, 256, 1), (64, 4, 1500, 4096, 2048, 0, 256, 0), (2, 1, 10, 96, 128, 0, 64, 0)])
def test_experts_gemm_choice_of_tiles(E, k, T, N, K, glu, rows, apart):
    """Tiles by rounds over the chip, with room for an expert that has a second one; walks apart in single rounds."""
    from hcache_deepspeed_amd.ops import native
    assert native.kernels().hds_experts_gemm_rows(T * k, N, K, E, glu) == rows + apart


def test_counted_waits_retire_lds_reads():
    """A statement that waits for loads and joins a barrier, behind which others overwrite what the wave has read from LDS,
    waits for those reads too: nothing else keeps their use in front of it."""
    import hcache_deepspeed_amd
    kernels = pathlib.Path(hcache_deepspeed_amd.__file__).parent / "csrc" / "kernels"
    found = []
    for f in sorted(kernels.glob("*.hip")):
        found += [(f.name, a) for a in re.findall(r'asm volatile\("([^"]*)"', f.read_text())
                  if "s_waitcnt" in a and "s_barrier" in a]
    assert [f for f, _ in found].count("grouped_gemm.hip") == 2
    for f, a in found:
        assert "lgkmcnt(0)" in a.split("s_barrier")[0], (f, a)
