"""Weight gradients of short reductions with their scale in the product (ops/gemm.py): products against 64 bits, and the fused LM
head's gradients against the general way of making them."""
import pytest
import torch

from hcache_deepspeed_amd.ops.cross_entropy import fused_linear_cross_entropy
from hcache_deepspeed_amd.ops.gemm import SCALED_WGRAD_ROWS, scaled_wgrad, scaled_wgrad_operands

pytestmark = pytest.mark.gpu


def _near(got, want, size, what=""):
    """One rounding to bf16, and sums of 32 bits over parts whose magnitudes add up to ``size``."""
    bound = 2.0**-8 * want.abs() + 1e-5 * size + 1e-30
    assert ((got.double() - want).abs() <= bound).all(), what


# around the tiles of 128 and both kernels
@pytest.mark.parametrize("T,N,K", [(T, 8192, 2048) for T in (1, 63, 64, 65, 127, 128, 129, 509, 1018, 2046, 3000)] +
                         [(T, 65536, 256) for T in (1, 1100)])
def test_products(T, N, K):
    g = torch.Generator(device="cuda").manual_seed(T)
    wide = torch.randn(T, N + 8, device="cuda", generator=g).bfloat16()
    dy, x = wide[:, :N], torch.randn(T, K, device="cuda", generator=g).bfloat16()  # rows further apart than they are long
    a, b = scaled_wgrad_operands(dy, x)
    scale = torch.tensor(0.37, device="cuda")
    out = torch.randn(N, K, device="cuda", generator=g).bfloat16()
    old = out.clone()
    assert scaled_wgrad(a, b, scale, out, True)
    fresh = torch.empty_like(out)
    assert scaled_wgrad(a, b, scale, fresh)
    for r in range(0, N, 8192):
        p = slice(r, r + 8192)
        want = (dy[:, p].double().t() @ x.double()) * scale.double()
        size = (dy[:, p].double().abs().t() @ x.double().abs()) * scale.double()
        _near(fresh[p], want, size, "fresh")
        _near(out[p], want + old[p].double(), size + old[p].double().abs(), "added")


def test_other_calls_are_left():
    m = lambda *s: torch.randn(*s, device="cuda").bfloat16()  # noqa: E731
    for dy, x in ((m(SCALED_WGRAD_ROWS + 1, 8192), m(SCALED_WGRAD_ROWS + 1, 2048)), (m(64, 8200), m(64, 2048)),
                  (m(1101, 65536), m(1101, 256)), (m(64, 8192), m(64, 2040)), (m(64, 2048), m(64, 2048)), (m(64, 8192).float(), m(64, 2048)),
                  (m(64, 8196)[:, 4:], m(64, 2048)), (m(8192, 64).t(), m(64, 2048))):
        assert scaled_wgrad_operands(dy, x) is None
    a, b = scaled_wgrad_operands(m(64, 8192), m(64, 2048))
    for out in (torch.empty(8192, 2048, device="cuda"), m(8192, 4096)[:, :2048], m(2048, 8192)):
        assert not scaled_wgrad(a, b, torch.ones((), device="cuda"), out)
    assert not scaled_wgrad(a, b, torch.ones((), device="cuda").double(), m(8192, 2048))


@pytest.mark.parametrize("T", [5, 300])
def test_loss_and_gradients(T):
    H, V = 512, 32768
    g = torch.Generator(device="cuda").manual_seed(T)
    h0 = torch.randn(T, H, device="cuda", generator=g).bfloat16()
    w0 = (torch.randn(V, H, device="cuda", generator=g) * H**-0.5).bfloat16()
    t = torch.randint(0, V, (T, ), device="cuda", generator=g)
    t[1] = -100
    got = {}
    for rows in (4096, (T + 1) // 2):  # one chunk, two of them
        h, w = h0.clone().requires_grad_(), w0.clone().requires_grad_()
        loss = fused_linear_cross_entropy(h, w, t, chunk_rows=rows)
        got[rows] = [loss.detach()] + list(torch.autograd.grad(loss * 3, (h, w)))
    one, two = got.values()
    z = h0.double() @ w0.double().t()
    p = torch.softmax(z, -1)
    p[torch.arange(T, device="cuda"), t.clamp_min(0)] -= 1
    p[t < 0] = 0
    want = (p.t() @ h0.double()) * 3 / (T - 1)
    e = [(x[2].double() - want).norm() / want.norm() for x in (one, two)]
    # both from the same rounded logits and their gradients (2^-9 each), once rounded
    assert e[0] < 0.01 and e[0] < 1.05 * e[1], e
    assert torch.allclose(one[0], two[0], rtol=1e-5) and (one[1].float() - two[1].float()).norm() < 0.01 * two[1].float().norm()


@pytest.mark.parametrize("T,V,H,want", [(200, 65536, 256, True), (257, 65536, 256, False), (640, 32768, 512, True), (641, 32768, 512, False),
                                        (1100, 16384, 1024, True), (1101, 16384, 1024, False), (1101, 8192, 2048, True)])
def test_short_heads_are_left_where_their_transposes_cost_more(cuda, monkeypatch, T, V, H, want):
    """Which way the LM head's gradient is made, by its columns; the same gradient either way."""
    from hcache_deepspeed_amd.ops import gemm
    g = torch.Generator(device="cuda").manual_seed(T)
    h = torch.randn(T, H, device="cuda", generator=g).bfloat16()
    w = (torch.randn(V, H, device="cuda", generator=g) * H**-0.5).bfloat16().requires_grad_()
    ids = torch.randint(0, V, (T, ), device="cuda", generator=g)
    calls, plain, grads = [], gemm.scaled_wgrad, []
    monkeypatch.setattr(gemm, "scaled_wgrad", lambda *a: calls.append(1) or plain(*a))
    for off in (False, True):
        if off:
            monkeypatch.setattr(gemm, "scaled_wgrad_operands", lambda *a: None)
        loss = fused_linear_cross_entropy(h, w, ids)
        grads.append(torch.autograd.grad(loss, w)[0].double())
        assert bool(calls) == (want and not off)
        calls.clear()
    assert (grads[0] - grads[1]).norm() <= 2**-8 * grads[1].norm()
