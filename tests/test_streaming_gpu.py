"""The flat optimizer kernels at the edges of their workgroups: 2,048 elements (Adam), rounds of four vectors a lane (sum of
squares), four elements a lane (scaled gradient). Against the same arithmetic in float64."""
import pytest
import torch

pytestmark = pytest.mark.gpu

from hcache_deepspeed_amd.ops import native  # noqa: E402

BF16 = torch.bfloat16


@pytest.mark.parametrize("n", [1, 2047, 2048, 2049, 6 * 2048 + 5])
@pytest.mark.parametrize("pt,gt", [(torch.float32, BF16), (torch.float32, torch.float32), (torch.float32, torch.float16), (BF16, BF16),
                                   (BF16, torch.float32)])
def test_adam_flat_sizes(n, pt, gt):
    from hcache_deepspeed_amd.ops.optimizers import adam_flat
    gen = torch.Generator(device="cuda").manual_seed(n)
    p, g, m = (torch.randn(n, device="cuda", generator=gen) for _ in range(3))
    v = torch.rand(n, device="cuda", generator=gen)
    p, g, lp = p.to(pt), g.to(gt), torch.full((n + 8, ), 7.0, device="cuda", dtype=BF16)
    pd, gd, md, vd = (t.double() for t in (p, g, m, v))
    md = 0.9 * md + 0.1 * gd * 0.5
    vd = 0.95 * vd + 0.05 * (gd * 0.5)**2
    pd = pd - 1e-2 * ((md / (1 - 0.9**3)) / ((vd / (1 - 0.95**3)).sqrt() + 1e-8) + 0.1 * pd)
    adam_flat(p, g, m, v, 3, 1e-2, (0.9, 0.95), 1e-8, 0.1, adamw=True, lp_out=lp[:n], grad_scale=0.5)
    # a dozen roundings of 32-bit arithmetic; the master's own rounding in bf16
    torch.testing.assert_close(m.double(), md, rtol=1e-6, atol=1e-7)
    torch.testing.assert_close(v.double(), vd, rtol=1e-6, atol=1e-7)
    torch.testing.assert_close(p.double(), pd, rtol=2e-6 if pt == torch.float32 else 2**-8, atol=1e-6)
    torch.testing.assert_close(lp[:n].double(), pd, rtol=2**-8, atol=1e-6)
    assert (lp[n:] == 7.0).all()


@pytest.mark.parametrize("n", [1, 7, 8, 8 * 1024 * 4 - 8, 8 * 1024 * 4 + 3, 8 * 1024 * 4 * 256 * 2 + 8 * 1024 + 13])
@pytest.mark.parametrize("dtype", [BF16, torch.float16, torch.float32])
def test_sum_of_squares(n, dtype):
    x = torch.randn(n, device="cuda", generator=torch.Generator(device="cuda").manual_seed(n)).to(dtype)
    lib = native.kernels()

    def run(t):
        out, bad = torch.zeros(1, device="cuda"), torch.zeros(1, device="cuda", dtype=torch.int32)
        native.check(lib.hds_sumsq(native.dt(t), t.data_ptr(), n, out.data_ptr(), bad.data_ptr(), native.stream()), "sumsq")
        return out.item(), bad.item()

    want = x.double().square().sum().item()
    got, bad = run(x)
    assert bad == 0 and abs(got - want) <= 1e-4 * want  # chains of at most a few hundred 32-bit sums
    top = torch.finfo(dtype).max
    for at, value, flag in [(0, top, 0), (n - 1, -top, 0), (0, float("inf"), 1), (n - 1, float("-inf"), 1),
                            (n // 2, float("nan"), 1), (n - 1, float("nan"), 1)]:
        y = x.clone()
        y[at] = value
        assert run(y)[1] == flag, (at, value)


@pytest.mark.parametrize("n", [1, 3, 1024, 1027, 5000])
@pytest.mark.parametrize("dtype", [BF16, torch.float16, torch.float32])
@pytest.mark.parametrize("accumulate", [False, True])
def test_scaled_grad(n, dtype, accumulate):
    from hcache_deepspeed_amd.ops.cross_entropy import _scaled_grad_
    x = torch.randn(n, device="cuda")
    scale = torch.tensor([0.3], device="cuda")
    out = torch.randn(n, device="cuda").to(dtype)
    want = x.double() * scale.double() + (out.double() if accumulate else 0)
    _scaled_grad_(out, x, scale, accumulate)
    eps = {BF16: 2**-8, torch.float16: 2**-11, torch.float32: 2**-22}[dtype]
    torch.testing.assert_close(out.double(), want, rtol=eps, atol=1e-6)


def test_scaled_grad_of_more_threads_than_a_launch_has():
    """A launch has fewer than 2^32 threads: with four elements a thread, gradients of 2^34 and more go round again."""
    from hcache_deepspeed_amd.ops.cross_entropy import _scaled_grad_
    n = 2**34 + 1027
    torch.cuda.empty_cache()
    if torch.cuda.mem_get_info()[0] < 7 * n:
        pytest.skip("needs 120 GB")
    x, out = torch.ones(n, device="cuda"), torch.zeros(n, device="cuda", dtype=BF16)
    x[-1], x[0], x[2**33] = 5.0, 3.0, 2.0
    _scaled_grad_(out, x, torch.tensor([0.5], device="cuda"), False)
    assert [out[i].item() for i in (0, 1, 2**33, 2**33 + 1, n - 2, n - 1)] == [1.5, 0.5, 1.0, 0.5, 0.5, 2.5]
    whole = all((c == 0.5).sum().item() >= c.numel() - 2 for c in out.split(2**31))
    del x, out
    torch.cuda.empty_cache()
    assert whole
