"""Evoformer attention HIP forward (csrc/kernels/evoformer.hip) vs an fp32 torch softmax reference; the backward
(chunked recompute from the kernel's LSE) vs autograd of the reference (reference
tests/unit/ops/deepspeed4science/test_DS4Sci_EvoformerAttention.py)."""
import math

import pytest
import torch

from hcache_deepspeed_amd.ops.deepspeed4science import DS4Sci_EvoformerAttention


def _ref(q, k, v, b1, b2):
    qh, kh, vh = (x.float().transpose(-2, -3) for x in (q, k, v))
    s = torch.matmul(qh, kh.transpose(-1, -2)) / math.sqrt(q.shape[-1])
    if b1 is not None:
        s = s + b1.float()
    if b2 is not None:
        s = s + b2.float()
    return torch.matmul(torch.softmax(s, -1), vh).transpose(-2, -3)


@pytest.mark.gpu
@pytest.mark.parametrize("D", [32, 64, 128])
@pytest.mark.parametrize("L", [70, 256])
@pytest.mark.parametrize("bias_dtype", [torch.bfloat16, torch.float32])
def test_evoformer_fwd_bwd_hip(cuda, D, L, bias_dtype):
    torch.manual_seed(0)
    B, N, H = 1, 5, 4
    q, k, v = (torch.randn(B, N, L, H, D, device=cuda, dtype=torch.bfloat16, requires_grad=True) for _ in range(3))
    b1 = torch.randn(B, N, 1, 1, L, device=cuda, dtype=bias_dtype) * 0.5
    b1[..., -7:] = -1e9
    b1.requires_grad_(True)
    b2 = torch.randn(B, 1, H, L, L, device=cuda, dtype=bias_dtype).requires_grad_(True)
    out = DS4Sci_EvoformerAttention(q, k, v, [b1, b2])
    ref = _ref(q, k, v, b1, b2)
    assert out.dtype == torch.bfloat16
    torch.testing.assert_close(out.float(), ref, atol=2e-2, rtol=2e-2)
    g = torch.randn_like(out)
    assert out.grad_fn is not None
    ga = torch.autograd.grad(out, (q, k, v, b1, b2), g)
    gb = torch.autograd.grad(ref, (q, k, v, b1, b2), g.float())
    for x, y in zip(ga, gb):
        err = (x.float() - y).abs().max().item()
        assert err <= 5e-2 * max(1.0, y.abs().max().item()), err


@pytest.mark.gpu
def test_evoformer_no_bias_hip(cuda):
    torch.manual_seed(1)
    q, k, v = (torch.randn(2, 3, 96, 2, 32, device=cuda, dtype=torch.bfloat16) for _ in range(3))
    out = DS4Sci_EvoformerAttention(q, k, v, [])
    torch.testing.assert_close(out.float(), _ref(q, k, v, None, None), atol=2e-2, rtol=2e-2)


@pytest.mark.gpu
def test_evoformer_backward_runs_hip_kernels(cuda, monkeypatch):
    """The GPU backward is the HIP one (no chunked torch recompute)."""
    from hcache_deepspeed_amd.ops.deepspeed4science import evoformer_attn as ev
    called = []
    orig = ev._hip_backward
    monkeypatch.setattr(ev, "_hip_backward", lambda *a, **k: called.append(1) or orig(*a, **k))
    q, k, v = (torch.randn(1, 2, 64, 2, 32, device=cuda, dtype=torch.bfloat16, requires_grad=True) for _ in range(3))
    DS4Sci_EvoformerAttention(q, k, v, []).sum().backward()
    assert called and q.grad is not None and torch.isfinite(q.grad.float()).all()


@pytest.mark.gpu
@pytest.mark.parametrize("B,N,L,H,D,which,bias_dtype", [
    (1, 1, 1, 1, 32, "both", torch.bfloat16), (1, 3, 31, 2, 64, "both", torch.bfloat16),
    (2, 5, 33, 3, 32, "both", torch.float32), (1, 2, 64, 2, 128, "mask", torch.bfloat16),
    (1, 9, 193, 4, 32, "pair", torch.bfloat16), (1, 2, 257, 1, 64, "both", torch.bfloat16),
    (1, 33, 300, 2, 32, "both", torch.bfloat16), (1, 70, 40, 4, 64, "pair", torch.float32),
    (1, 2, 545, 2, 128, "both", torch.bfloat16), (2, 130, 17, 4, 32, "both", torch.bfloat16)])
def test_evoformer_edges_hip(cuda, B, N, L, H, D, which, bias_dtype):
    """Tails of the 32-position tiles, odd rows of the pair bias, one and several LDS chunks, one and several chunks of
    the rows in the pair gradient; masked keys at -1e9 and at minus infinity. Against float64; p, ds and the results are
    rounded to bf16 (2^-9 each), the sums to 32 bits."""
    g = torch.Generator(device="cuda").manual_seed(L)
    rnd = lambda *s: torch.randn(*s, device="cuda", generator=g)  # noqa: E731
    q, k, v, do = (rnd(B, N, L, H, D).bfloat16() for _ in range(4))
    b1 = b2 = None
    if which != "pair":
        gone = torch.rand(B, N, 1, 1, L, device="cuda", generator=g) < 0.2
        gone[..., 0] = False
        low = torch.full_like(gone, -1e9, dtype=bias_dtype)
        low[:, ::2] = float("-inf")
        b1 = torch.where(gone, low, torch.zeros((), dtype=bias_dtype, device="cuda"))
    if which != "mask":
        b2 = rnd(B, 1, H, L, L).to(bias_dtype)
    leaves = [t.requires_grad_() for t in (q, k, v, b2) if t is not None]
    out = DS4Sci_EvoformerAttention(q, k, v, [b1, b2])
    got = [out] + list(torch.autograd.grad(out, leaves, do))
    exact = [t.detach().double().requires_grad_() for t in leaves]
    qh, kh, vh = (t.transpose(-2, -3) for t in exact[:3])
    s = torch.matmul(qh, kh.transpose(-1, -2)) / math.sqrt(D)
    if b1 is not None:
        s = s + b1.double()
    if b2 is not None:
        s = s + exact[3]
    ref = torch.matmul(torch.softmax(s, -1), vh).transpose(-2, -3)
    want = [ref] + list(torch.autograd.grad(ref, exact, do.double()))
    for x, y in zip(got, want):
        assert torch.isfinite(x).all()
        assert (x.double() - y).norm() <= 4 * 2**-8 * y.norm() + 1e-6
    if b2 is not None:  # no atomics in these gradients
        again = torch.autograd.grad(DS4Sci_EvoformerAttention(q, k, v, [b1, b2]), leaves, do)
        assert all(torch.equal(x, y) for x, y in zip(got[1:], again))


@pytest.mark.gpu
@pytest.mark.parametrize("B,N,L,H,which", [(1, 70, 250, 8, "both"), (2, 75, 100, 4, "both"), (1, 1100, 40, 2, "mask"),
                                           (1, 3, 256, 2, "pair"), (1, 5, 160, 1, "both"), (1, 2100, 32, 1, "both"),
                                           (1, 515, 20, 8, "both"), (1, 520, 64, 8, "mask")])
def test_evoformer_rows_of_one_head(cuda, B, N, L, H, which):
    """The gradient kernel that takes a whole row in a workgroup: one and several rows after each other, the last chunk of
    them shorter, full and partial tiles of 32, odd counts of tiles, each of its four sizes."""
    test_evoformer_edges_hip(cuda, B, N, L, H, 32, which, torch.bfloat16)


@pytest.mark.gpu
@pytest.mark.parametrize("bias_dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("B,N,L,D,which", [(1, 9, 2, 32, "both"), (1, 33, 65, 32, "both"), (2, 21, 129, 64, "both"),
                                           (1, 17, 161, 32, "pair"), (1, 13, 256, 64, "both"), (1, 7, 290, 64, "pair")])
def test_evoformer_pair_gradient_of_shared_rows(cuda, B, N, L, D, which, bias_dtype):
    """The pair bias' gradient, of few rows: one or two blocks of keys, the second past the end, queries past the end, several
    workgroups of either, one and several chunks of rows of which the last is shorter. (Two keys at least: with one, dS is exactly zero and
    a relative bound has nothing to hold against the 2^-24 sum |dO V| that dP and delta may differ by, 1.06e-6 in dQ's
    norm here.)"""
    test_evoformer_edges_hip(cuda, B, N, L, 3, D, which, bias_dtype)


@pytest.mark.gpu
@pytest.mark.parametrize("bias_dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("where", ["mask", "pair"])
@pytest.mark.parametrize("low", ["inf", "lowest"])
@pytest.mark.parametrize("L,D,first", [(70, 32, 32), (257, 64, 64), (96, 128, 32), (300, 32, 256)])
def test_evoformer_leading_keys_masked(cuda, L, D, first, low, where, bias_dtype):
    """Queries whose first one or several tiles of 32 keys (or of 256, a whole chunk) are masked by minus infinity or the
    lowest value while later ones are visible, and queries without any visible key, whose result and gradients are zero.
    Against float64, with the bound of the edge tests."""
    B, N, H = 1, 3, 2
    g = torch.Generator(device="cuda").manual_seed(L + D)
    rnd = lambda *s: torch.randn(*s, device="cuda", generator=g)  # noqa: E731
    q, k, v, do = (rnd(B, N, L, H, D).bfloat16() for _ in range(4))
    low = -math.inf if low == "inf" else torch.finfo(bias_dtype).min
    b1, b2 = torch.zeros(B, N, 1, 1, L, dtype=bias_dtype, device="cuda"), rnd(B, 1, H, L, L).to(bias_dtype)
    if where == "mask":
        b1[:, 1, ..., :first] = low
        b1[:, 2] = -math.inf
    else:
        b2[:, :, 0, L // 2:, :first] = low
        b2[:, :, 1, 3:40] = -math.inf
    leaves = [t.requires_grad_() for t in (q, k, v, b2)]
    out = DS4Sci_EvoformerAttention(q, k, v, [b1, b2])
    got = [out] + list(torch.autograd.grad(out, leaves, do))
    qh, kh, vh, pair = exact = [t.detach().double().requires_grad_() for t in leaves]
    s = torch.matmul(qh.transpose(-2, -3), kh.transpose(-2, -3).transpose(-1, -2)) / math.sqrt(D) + b1.double() + pair
    top = s.detach().amax(-1, keepdim=True)
    p = torch.exp(s - torch.where(top.isinf(), 0., top))
    ref = torch.matmul(p / p.sum(-1, keepdim=True).clamp_min(1e-300), vh.transpose(-2, -3)).transpose(-2, -3)
    want = [ref] + list(torch.autograd.grad(ref, exact, do.double()))
    if where == "mask":
        assert not out[:, 2].any() and not got[1][:, 2].any()
    for x, y in zip(got, want):
        assert torch.isfinite(x).all()
        assert (x.double() - y).norm() <= 4 * 2**-8 * y.norm() + 1e-6


@pytest.mark.gpu
@pytest.mark.parametrize("bias_dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("D", [32, 64, 128])
def test_evoformer_large_finite_mask(cuda, D, bias_dtype):
    """A finite mask stays finite: a query whose keys are all masked by -1e38, beside which the scores do not count in 32
    bits, has the mean of the values."""
    torch.manual_seed(D)
    q, k, v = (torch.randn(1, 2, 90, 2, D, device=cuda, dtype=torch.bfloat16) for _ in range(3))
    b1 = torch.zeros(1, 2, 1, 1, 90, dtype=bias_dtype, device=cuda)
    b1[:, 1] = -1e38
    out = DS4Sci_EvoformerAttention(q, k, v, [b1, None])
    torch.testing.assert_close(out[:, :1].float(), _ref(q, k, v, None, None)[:, :1], atol=2e-2, rtol=2e-2)
    mean = v[:, 1:].double().mean(2, keepdim=True).expand(-1, -1, 90, -1, -1)
    assert (out[:, 1:].double() - mean).norm() <= 2 * 2**-8 * mean.norm()


@pytest.mark.gpu
@pytest.mark.parametrize("bias_dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("D,scale", [(32, 0.125), (32, 0.249), (128, 0.3), (64, 0.1), (64, 0.3), (64, 0.0), (32, -0.1)])
def test_evoformer_kernel_takes_a_scale_or_refuses_it(cuda, D, scale, bias_dtype):
    """The kernels' entry with other scales than D^-0.5: 1 / scale of one bf16 piece, of three, just above one; a mask of
    minus infinity; scales that it cannot take are refused (64 columns with bf16 biases hold one piece)."""
    from hcache_deepspeed_amd.ops import native
    torch.manual_seed(D)
    N, L, H = 3, 70, 2
    q, k, v = (torch.randn(1, N, L, H, D, device=cuda, dtype=torch.bfloat16) for _ in range(3))
    b1 = torch.zeros(1, N, 1, 1, L, device=cuda, dtype=bias_dtype)
    b1[:, 1, ..., :40] = -math.inf
    b2 = torch.randn(1, 1, H, L, L, device=cuda).mul_(100).to(bias_dtype)
    o, lse = torch.empty_like(q), torch.empty(1, N, H, L, device=cuda)
    rc = native.kernels().hds_evoformer_fwd(q.data_ptr(), k.data_ptr(), v.data_ptr(), b1.data_ptr(), b2.data_ptr(),
                                            native.dt(b1), o.data_ptr(), lse.data_ptr(), 1, N, L, H, D, scale,
                                            native.stream())
    if scale <= 0 or (scale == 0.3 and D == 64 and bias_dtype == torch.bfloat16):
        assert rc != 0
        return
    assert rc == 0
    scale = torch.tensor(scale, dtype=torch.float32).double().item()
    s = (q.double().transpose(-2, -3) @ k.double().transpose(-2, -3).transpose(-1, -2)) * scale + b1.double() + b2.double()
    ref = (torch.softmax(s, -1) @ v.double().transpose(-2, -3)).transpose(-2, -3)
    assert (o.double() - ref).norm() <= 2 * 2**-8 * ref.norm()
    # 32-bit scores of a few hundred, in units of 1 / scale
    assert (lse.double() - torch.logsumexp(s, -1)).abs().max() <= 2e-6 * s.abs().nan_to_num(0, 0, 0).max() + 1e-4


@pytest.mark.gpu
def test_evoformer_saved_tensors_in_another_order(cuda):
    """Saved tensors that come back from pinned host memory are contiguous as they were saved, [B, N, H, L, D]."""
    g = torch.Generator(cuda).manual_seed(2)
    q, k, v, do = (torch.randn(1, 3, 70, 4, 32, device=cuda, generator=g).bfloat16().requires_grad_(i < 3) for i in range(4))
    want = torch.autograd.grad(DS4Sci_EvoformerAttention(q, k, v, []), (q, k, v), do)
    with torch.autograd.graph.save_on_cpu(pin_memory=True):
        out = DS4Sci_EvoformerAttention(q, k, v, [])
    torch.cuda.synchronize()
    for a, b in zip(torch.autograd.grad(out, (q, k, v), do), want):
        assert torch.equal(a, b)


@pytest.mark.gpu
@pytest.mark.parametrize("bias_dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("N,L,H,D,bf16,fp32", [
    (512, 32, 8, 64, 0, 0), (512, 64, 8, 64, 0, 0), (20, 100, 4, 64, 0, 0), (128, 32, 8, 32, 0, 0), (64, 128, 4, 32, 0, 0),
    (512, 160, 8, 32, 0, 0), (4, 512, 8, 32, 0, 0), (128, 192, 8, 32, 1, 0), (128, 256, 8, 32, 1, 1), (128, 256, 8, 128, 0, 0),
    (114, 65, 3, 64, 1, 0), (38, 161, 3, 64, 1, 0), (14, 290, 3, 64, 1, 0), (43, 256, 3, 64, 1, 1), (170, 120, 3, 32, 1, 0),
    (43, 250, 3, 32, 1, 0), (18, 384, 3, 32, 1, 1), (170, 128, 3, 32, 1, 1)])
def test_evoformer_pair_gradient_kernels(cuda, N, L, H, D, bf16, fp32, bias_dtype):
    """Which kernel sums the pair bias' gradient: staged rows want a filled chip and full workgroups. The smaller sizes run: one
    and two waves of keys, the second past the end, queries past the end, a last chunk of one row."""
    from hcache_deepspeed_amd.ops import native
    want = bf16 if bias_dtype == torch.bfloat16 else fp32
    dt = native.dt(torch.empty(0, dtype=bias_dtype))
    assert native.kernels().hds_evoformer_pair_staged(1, N, L, H, D, dt) == want
    if H == 3:
        test_evoformer_edges_hip(cuda, 1, N, L, H, D, "both", bias_dtype)


def test_launch_attributes_are_set_for_the_current_device():
    """A kernel's largest LDS size belongs to a device: set once a process, the others would refuse the launch."""
    import pathlib
    import re
    import hcache_deepspeed_amd
    src = (pathlib.Path(hcache_deepspeed_amd.__file__).parent / "csrc" / "kernels" / "evoformer.hip").read_text()
    assert "hipFuncSetAttribute" in src and re.search(r"\bstatic\b[^;{]*hipFuncSetAttribute", src) is None


@pytest.mark.gpu
@pytest.mark.parametrize("B,N,L,H", [(1, 520, 17, 8), (1, 4100, 31, 1), (1, 260, 64, 8), (2, 140, 57, 8), (1, 140, 97, 8),
                                     (1, 66, 200, 8), (2, 70, 256, 4)])
def test_evoformer_walked_rows(cuda, B, N, L, H):
    """Forward workgroups that walk over rows (three and more of a head), and both gradients from their normalisers, against
    the general kernels, which 32-bit biases of the same values take. Among the rows: all keys masked by -1e9, by -1e38 and by
    minus infinity, half of them by -1e38, and queries whose scores are large, far from zero or minus infinity. Both sides
    round p and ds to bf16 (2^-9 each), the results too."""
    g = torch.Generator(device="cuda").manual_seed(L)
    rnd = lambda *s: torch.randn(*s, device="cuda", generator=g)  # noqa: E731
    q, k, v, do = (rnd(B, N, L, H, 32).bfloat16() for _ in range(4))
    b1 = torch.where(rnd(B, N, 1, 1, L) < -1, -1e9, 0.).bfloat16()
    b1[..., 0] = 0
    b1[:, 1], b1[:, 2], b1[:, 3], b1[:, 5, ..., ::2] = -1e9, -1e38, -math.inf, -1e38
    b2 = rnd(B, 1, H, L, L).bfloat16()
    b2[:, :, 0, 5] += 300
    b2[:, :, 0, 6] -= 300
    b2[:, :, 0, 7, 3:9] = -math.inf
    b2[:, :, H - 1, 8] = -1e9
    do[:, 1:3] = 0  # (keys that are all masked: their weights add up to one only to the rounding of 1e9)
    sides = []
    for dtype in (torch.bfloat16, torch.float32):
        leaves = [t.detach().clone().requires_grad_() for t in (q, k, v, b2.to(dtype))]
        out = DS4Sci_EvoformerAttention(*leaves[:3], [b1.to(dtype), leaves[3]])
        with torch.no_grad():
            assert torch.equal(out, DS4Sci_EvoformerAttention(*leaves[:3], [b1.to(dtype), leaves[3]]))
        sides.append([out] + list(torch.autograd.grad(out, leaves, do)))
    for x, y in zip(*sides):
        assert torch.isfinite(x).all() and torch.isfinite(y).all()
        assert (x.double() - y.double()).norm() <= 4 * 2**-8 * y.double().norm()
    x, y = (side[0].double() for side in sides)  # the rows out of the ordinary by themselves
    for part in [(slice(None), n) for n in (1, 2, 5)] + [
            (slice(None), slice(None), i, h) for i, h in ((5, 0), (6, 0), (7, 0), (8, H - 1))]:
        assert (x[part] - y[part]).norm() <= 4 * 2**-8 * y[part].norm()
    assert not x[:, 3].any() and not y[:, 3].any()


@pytest.mark.gpu
@pytest.mark.parametrize("N,L,H", [(520, 17, 8), (190, 97, 8), (66, 200, 8), (130, 240, 4), (66, 161, 8)])
def test_evoformer_positions_past_the_end_are_not_read(cuda, N, L, H):
    """Rows whose last tile of 32 is partial, with NaN in the rows behind: nothing of a neighbour comes into a row, and nothing
    of what lies behind the last one into the pair bias' gradient."""
    g = torch.Generator(device="cuda").manual_seed(L)
    rnd = lambda *s: torch.randn(*s, device="cuda", generator=g)  # noqa: E731
    q, k, v, do = whole = [rnd(1, N + 1, L, H, 32).bfloat16() for _ in range(4)]
    b1, b2 = torch.zeros(1, N, 1, 1, L, dtype=torch.bfloat16, device="cuda"), rnd(1, 1, H, L, L).bfloat16()

    def call(rows):
        q, k, v, do = (t[:, :N].detach() for t in rows)
        assert q.is_contiguous()
        leaves = [t.requires_grad_() for t in (q, k, v, b2.detach())]
        out = DS4Sci_EvoformerAttention(*leaves[:3], [b1, leaves[3]])
        return [out.detach()] + list(torch.autograd.grad(out, leaves, do))
    clean = call(whole)
    for t in whole:
        t[:, N:] = math.nan
    assert all(torch.equal(a, b) for a, b in zip(call(whole), clean))
    for t in whole:
        t[:, 1::2] = math.nan
    for a, b in zip(call(whole)[:4], clean):
        assert torch.equal(a[:, ::2], b[:, ::2])


@pytest.mark.parametrize("L,H,D,want", [(65, 174000, 64, 1), (65, 175000, 64, 0), (128, 263000, 32, 1), (128, 264000, 32, 0),
                                        (300, 78000, 64, 1), (300, 79000, 64, 0), (100, 1 << 25, 64, 0)])
def test_evoformer_staged_rows_have_offsets_in_32_bits(L, H, D, want):
    """The pair bias' gradient by staged rows, whose distances are 32 bits, only where (L + 127) rows of H heads fit."""
    from hcache_deepspeed_amd.ops import native
    assert native.kernels().hds_evoformer_pair_staged(1, 4, L, H, D, 1) == want
    assert want == (2 * (L + 127) * H * D < 1 << 32)


def _walked(cuda, N, L, H, b1, b2, g):
    """Inputs, result, normalisers and gradients of a call, against float64 in blocks of rows."""
    rnd = lambda *s: torch.randn(*s, device="cuda", generator=g)  # noqa: E731
    q, k, v, do = (rnd(1, N, L, H, 32).bfloat16() for _ in range(4))
    leaves = [t.requires_grad_() for t in (q, k, v, b2)]
    out = DS4Sci_EvoformerAttention(q, k, v, [b1, b2])
    got = [out] + list(torch.autograd.grad(out, leaves, do))
    want = [torch.empty(t.shape, dtype=torch.float64, device=cuda) for t in got]
    want[4].zero_()
    for n in range(N):
        qh, kh, vh = one = [t[:, n:n + 1].detach().double().requires_grad_() for t in (q, k, v)]
        pair = b2.detach().double().requires_grad_()
        s = qh.transpose(-2, -3) @ kh.transpose(-2, -3).transpose(-1, -2) / math.sqrt(32) + b1[:, n:n + 1].double() + pair
        top = s.detach().amax(-1, keepdim=True)
        p = torch.exp(s - torch.where(top.isinf(), 0., top))
        ref = (p / p.sum(-1, keepdim=True).clamp_min(1e-300) @ vh.transpose(-2, -3)).transpose(-2, -3)
        grads = torch.autograd.grad(ref, one + [pair], do[:, n:n + 1].double())
        for w, x in zip(want, (ref, ) + grads[:3]):
            w[:, n:n + 1] = x.detach()
        want[4] += grads[3]
    return got, want


_LOWS = (-1e9, -2e10, -1e12, -1e15, -1e30, -1e35, -1e37, -3e37, -math.inf, torch.finfo(torch.bfloat16).min)


@pytest.mark.gpu
@pytest.mark.parametrize("N,L,H,where", [(66, 200, 8, "mask"), (66, 256, 8, "pair"), (190, 97, 8, "mask"), (190, 128, 8, "pair"),
                                         (130, 161, 4, "mask"), (260, 64, 8, "mask"), (260, 40, 8, "pair")])
def test_evoformer_walked_rows_leading_keys(cuda, N, L, H, where):
    """Rows whose first one, two or four tiles of keys have a large negative bias of any size, in walking workgroups: later keys
    have the weight. Against float64, with the bound of the edge tests, and each such row by itself."""
    g = torch.Generator(device="cuda").manual_seed(L)
    b1 = torch.zeros(1, N, 1, 1, L, dtype=torch.bfloat16, device="cuda")
    b2 = torch.randn(1, 1, H, L, L, device="cuda", generator=g).bfloat16()
    firsts = [f for f in (32, 64, 128) if f < L]
    if where == "mask":
        for i, low in enumerate(_LOWS):
            for j, first in enumerate(firsts):
                b1[:, 3 * i + j, ..., :first] = low
    else:
        for i, low in enumerate(_LOWS):
            for j, first in enumerate(firsts):
                b2[:, :, i % H, 3 * i + j, :first] = low
    got, want = _walked(cuda, N, L, H, b1, b2, g)
    for x, y in zip(got, want):
        assert torch.isfinite(x).all()
        assert (x.double() - y).norm() <= 4 * 2**-8 * y.norm() + 1e-6
    x, y = got[0].double(), want[0]
    rows = (range(3 * len(_LOWS)) if where == "mask" else [])
    for part in [(slice(None), n) for n in rows] + [(slice(None), slice(None), n) for n in range(min(L, 3 * len(_LOWS)))]:
        assert (x[part] - y[part]).norm() <= 4 * 2**-8 * y[part].norm()


@pytest.mark.gpu
@pytest.mark.parametrize("scale", [0.125, 0.249, 1.0, 3.0])
@pytest.mark.parametrize("N,L,H", [(66, 200, 8), (190, 97, 8), (260, 64, 8)])
def test_evoformer_walked_rows_of_a_scale(cuda, N, L, H, scale):
    """The same of other scales than D^-0.5 through the kernels' entry: with scales of one and more the lowest value stays finite
    over them. 32-bit scores of up to 20 (lse), the result rounded to bf16."""
    from hcache_deepspeed_amd.ops import native
    g = torch.Generator(device="cuda").manual_seed(L)
    q, k, v = (torch.randn(1, N, L, H, 32, device="cuda", generator=g).bfloat16() for _ in range(3))
    q /= 32**0.5 * scale
    b1 = torch.zeros(1, N, 1, 1, L, device=cuda, dtype=torch.bfloat16)
    for i, low in enumerate(_LOWS):
        b1[:, 2 * i, ..., :32], b1[:, 2 * i + 1, ..., :L // 2] = low, low
    b2 = torch.randn(1, 1, H, L, L, device=cuda, generator=g).bfloat16()
    o, lse = torch.empty_like(q), torch.empty(1, N, H, L, device=cuda)
    native.check(native.kernels().hds_evoformer_fwd(q.data_ptr(), k.data_ptr(), v.data_ptr(), b1.data_ptr(), b2.data_ptr(), 1,
                                                    o.data_ptr(), lse.data_ptr(), 1, N, L, H, 32, scale, native.stream()), "fwd")
    scale = torch.tensor(scale, dtype=torch.float32).double().item()
    for n in range(N):
        a, b, e = (t[0, n].double().transpose(0, 1) for t in (q, k, v))
        s = a @ b.transpose(1, 2) * scale + b1[0, n].double() + b2[0, 0].double()
        ref = (torch.softmax(s, -1) @ e).transpose(0, 1)
        assert (o[0, n].double() - ref).norm() <= 2 * 2**-8 * ref.norm()
        assert (lse[0, n].double() - torch.logsumexp(s, -1)).abs().max() <= 1e-4


@pytest.mark.gpu
@pytest.mark.parametrize("N,L,H", [(128, 256, 8), (66, 200, 8), (190, 97, 8), (260, 64, 8), (520, 17, 8)])
def test_evoformer_walked_rows_round_as_single_ones(cuda, N, L, H):
    """The walking workgroups raise a row's maximum with every tile of 32 keys, as the general kernel does, so that the weights
    are rounded alike: of its values (as those rows give them in calls of one row each) but for the rounding of 32-bit sums,
    which turns few of the results' last bits."""
    g = torch.Generator(device="cuda").manual_seed(L)
    q, k, v = (torch.randn(1, N, L, H, 32, device="cuda", generator=g).bfloat16() for _ in range(3))
    b1 = torch.where(torch.rand(1, N, 1, 1, L, device="cuda", generator=g) < 0.1, -1e9, 0.).bfloat16()
    b2 = torch.randn(1, 1, H, L, L, device="cuda", generator=g).bfloat16()
    with torch.no_grad():
        out = DS4Sci_EvoformerAttention(q, k, v, [b1, b2])
        for n in range(0, N, 7):
            one = DS4Sci_EvoformerAttention(*(t[:, n:n + 1].contiguous() for t in (q, k, v, )), [b1[:, n:n + 1].contiguous(), b2])
            a, b = out[:, n].double(), one[:, 0].double()
            # a weight near the middle of two bf16 values may fall either way: 2^-8 of it. One in a hundred does (2^-24 of a
            # sum's rounding against 2^-8 would be one in thousands); with a maximum raised less often all of them may
            assert (a - b).norm() <= 0.1 * 2**-8 * b.norm()


@pytest.mark.gpu
@pytest.mark.parametrize("N,L,H", [(66, 200, 8), (190, 97, 8), (130, 256, 8), (260, 64, 8)])
def test_evoformer_biases_of_opposite_signs(cuda, N, L, H):
    """Large biases that take each other back to the scores' range. What the scores are then depends on the order of the sums, but
    it is one order: a query's weights add up to one in the result, in dV and (dS to zero) in the pair bias' gradient."""
    g = torch.Generator(device="cuda").manual_seed(L)
    rnd = lambda *s: torch.randn(*s, device="cuda", generator=g)  # noqa: E731
    q, k, v, do = (rnd(1, N, L, H, 32).bfloat16() for _ in range(4))
    b1, b2 = torch.zeros(1, N, 1, 1, L, dtype=torch.bfloat16, device="cuda"), rnd(1, 1, H, L, L).bfloat16()
    sides = ((-1e9, 1e9), (-1e38, 1e38), (-2e37, 2e37), (1e9, -1e9), (1e38, -1e38), (5e4, -5e4), (-300, 300), (1e38, -math.inf))
    for i, (mask, pair) in enumerate(sides):  # 32 queries of a head each, so that nothing else decides about them
        b1[:, i, ..., 4:14] = mask
        b2[:, :, i, :32, 4:14] = pair
    keep = [do[0, i, :32, i].clone() for i in range(8)]
    do.zero_()
    for i in range(8):
        do[0, i, :32, i] = keep[i]
    leaves = [t.requires_grad_() for t in (q, k, v, b2)]
    with torch.no_grad():
        total = DS4Sci_EvoformerAttention(q, k, torch.ones_like(v), [b1, b2])
    assert (total.double() - 1).abs().max() <= 2**-6  # (p and the result are rounded to bf16)
    out = DS4Sci_EvoformerAttention(q, k, v, [b1, b2])
    grads = torch.autograd.grad(out, leaves, do)
    assert all(torch.isfinite(t).all() for t in (out, ) + grads)
    for i, (mask, pair) in enumerate(sides):
        # p and dV are rounded to bf16; from 1e37 on, in units of 1e30, the order of a product's own sums counts
        dv, want = grads[2][0, i, :, i].double().sum(0), keep[i].double().sum(0)
        assert pair > 1e10 or (dv - want).norm() <= 2 * 2**-8 * keep[i].double().norm(), (i, (dv - want).norm() / want.norm())
        ds = grads[3][0, 0, i, :32].double()
        assert (ds.sum(-1).abs() <= 2**-6 * ds.abs().sum(-1)).all()


@pytest.mark.parametrize("B,N,L,H,want", [
    (1, 64, 256, 8, 0), (1, 65, 256, 8, 3), (1, 128, 256, 8, 4), (1, 2048, 256, 8, 64), (1, 2049, 256, 8, 0), (1, 128, 257, 8, 0),
    (192, 1, 256, 8, 0), (96, 2, 200, 8, 0), (48, 4, 256, 8, 0), (24, 8, 256, 8, 0), (32, 6, 256, 8, 6), (16, 12, 250, 8, 6),
    (1, 257, 256, 3, 4), (1, 512, 256, 3, 7), (384, 1, 128, 8, 0), (192, 2, 128, 8, 0), (96, 4, 128, 8, 4), (24, 16, 100, 8, 6),
    (1, 131, 128, 8, 0), (1, 192, 128, 8, 3), (768, 1, 64, 8, 1), (1, 256, 64, 8, 0), (1, 257, 64, 8, 3), (1536, 1, 17, 8, 1)])
def test_evoformer_rows_of_a_walk(B, N, L, H, want):
    """Rows of a forward workgroup: as many as let the launch run in one round, and a workgroup a row where walks would be short
    or a second round mostly empty."""
    from hcache_deepspeed_amd.ops import native
    assert native.kernels().hds_evoformer_walk(B, N, L, H) == want


def test_evoformer_sizes_above_walk():
    """The sizes of the tests of walking workgroups are theirs."""
    from hcache_deepspeed_amd.ops import native
    for N, L, H in [(66, 200, 8), (66, 256, 8), (66, 161, 8), (128, 256, 8), (130, 256, 8), (130, 240, 4), (130, 161, 4), (190, 97, 8),
                    (190, 128, 8), (260, 64, 8), (260, 40, 8), (520, 17, 8)]:
        assert native.kernels().hds_evoformer_walk(1, N, L, H) >= 3


@pytest.mark.gpu
@pytest.mark.parametrize("B,N,L,H", [(40, 8, 250, 3), (32, 6, 200, 8), (700, 3, 40, 2), (96, 4, 100, 8), (2100, 1, 20, 2)])
def test_evoformer_walks_in_many_batches(cuda, B, N, L, H):
    """Walks that end with a batch, against the rows of some batches in calls of their own."""
    g = torch.Generator(device="cuda").manual_seed(L)
    rnd = lambda *s: torch.randn(*s, device="cuda", generator=g).bfloat16()  # noqa: E731
    q, k, v = (rnd(B, N, L, H, 32) for _ in range(3))
    b1 = torch.where(torch.rand(B, N, 1, 1, L, device="cuda", generator=g) < 0.1, -1e9, 0.).bfloat16()
    b2 = rnd(B, 1, H, L, L)
    with torch.no_grad():
        out = DS4Sci_EvoformerAttention(q, k, v, [b1, b2])
        for b in sorted({0, 1, B // 2, B - 1}):
            one = DS4Sci_EvoformerAttention(*(t[b:b + 1] for t in (q, k, v)), [b1[b:b + 1], b2[b:b + 1]])
            x, y = out[b].double(), one[0].double()
            assert (x - y).norm() <= 0.1 * 2**-8 * y.norm()  # (as rows by themselves above)


@pytest.mark.gpu
@pytest.mark.parametrize("which", ["none", "mask", "pair"])
@pytest.mark.parametrize("N,L,H", [(66, 200, 8), (190, 97, 8), (520, 17, 8)])
def test_evoformer_walks_with_fewer_biases(cuda, N, L, H, which):
    """Walking workgroups without the mask, the pair bias or both, with the bound of the edge tests."""
    if which != "none":
        test_evoformer_edges_hip(cuda, 1, N, L, H, 32, which, torch.bfloat16)
        return
    g = torch.Generator(device="cuda").manual_seed(L)
    q, k, v, do = (torch.randn(1, N, L, H, 32, device="cuda", generator=g).bfloat16() for _ in range(4))
    leaves = [t.requires_grad_() for t in (q, k, v)]
    out = DS4Sci_EvoformerAttention(*leaves, [])
    got = [out] + list(torch.autograd.grad(out, leaves, do))
    exact = [t.detach().double().requires_grad_() for t in leaves]
    qh, kh, vh = (t.transpose(-2, -3) for t in exact)
    ref = (torch.softmax(qh @ kh.transpose(-1, -2) / math.sqrt(32), -1) @ vh).transpose(-2, -3)
    for x, y in zip(got, [ref] + list(torch.autograd.grad(ref, exact, do.double()))):
        assert (x.double() - y).norm() <= 4 * 2**-8 * y.norm()
