"""Stacked-expert GEMMs on MI355X at Mixtral-8x7B width: the per-expert 2-D GEMM path (parallel/moe.py
``expert_linear``) against an fp32 reference, forward and both gradients. The batched hipBLASLt form of the
down projection failed on this shape (HIPBLAS_STATUS_INTERNAL_ERROR, then an illegal access in the fallback)."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.fixture(autouse=True)
def _gpu():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")


@pytest.mark.parametrize("E,C,N,K", [(8, 1280, 4096, 14336), (8, 1280, 28672, 4096), (4, 96, 256, 512)])
def test_expert_linear_matches_fp32(E, C, N, K):
    from hcache_deepspeed_amd.parallel.moe import expert_linear
    g = torch.Generator(device="cuda").manual_seed(0)
    x = (torch.randn(E, C, K, device="cuda", generator=g) * 0.5).to(torch.bfloat16).requires_grad_(True)
    w = (torch.randn(E, N, K, device="cuda", generator=g) * K**-0.5).to(torch.bfloat16).requires_grad_(True)
    y = expert_linear(x, w)
    dy = torch.randn(E, C, N, device="cuda", generator=g).to(torch.bfloat16)
    y.backward(dy)
    torch.cuda.synchronize()
    for e in (0, E - 1):
        xf, wf, dyf = x[e].detach().float(), w[e].detach().float(), dy[e].float()
        ref = xf @ wf.t()
        rel = lambda a, b: ((a.float() - b).norm() / b.norm()).item()  # noqa: E731
        assert rel(y[e], ref) < 1e-2
        assert rel(x.grad[e], dyf @ wf) < 1e-2
        assert rel(w.grad[e], dyf.t() @ xf) < 1e-2


def test_mixtral_layer_full_width_step():
    """One full-width Mixtral decoder layer (8 experts x 14336, top-2) forward + backward at S=4096."""
    from hcache_deepspeed_amd.models.mixtral import MixtralForCausalLM, mixtral_8x7b
    torch.manual_seed(0)
    m = MixtralForCausalLM(mixtral_8x7b(num_hidden_layers=1)).cuda().to(torch.bfloat16)
    x = torch.randint(0, 32000, (1, 4096), device="cuda")
    loss = m(x, labels=x)
    loss.backward()
    torch.cuda.synchronize()
    assert torch.isfinite(loss).item()
    g = m.layers[0].block_sparse_moe.deepspeed_moe.experts.w2.grad
    assert g is not None and torch.isfinite(g.float()).all().item() and g.abs().sum().item() > 0


def test_mixtral_engine_direct_expert_wgrad_matches():
    """Stacked expert weight gradients written in place into the ZeRO gradient buffer (per-expert GEMMs with
    out=slice) train the same trajectory as the dense AccumulateGrad path (``mi355x.direct_wgrad: false``),
    with gradient accumulation over 2 micro-steps."""
    import os
    import hcache_deepspeed_amd as ds
    from hcache_deepspeed_amd.models.mixtral import MixtralForCausalLM, tiny_moe
    os.environ.setdefault("MASTER_PORT", "29571")
    res = {}
    for direct in (True, False):
        torch.manual_seed(0)
        m = MixtralForCausalLM(tiny_moe(hidden_size=256, intermediate_size=512, num_hidden_layers=2))
        cfg = {"train_micro_batch_size_per_gpu": 2, "gradient_accumulation_steps": 2, "bf16": {"enabled": True},
               "optimizer": {"type": "AdamW", "params": {"lr": 1e-3}}, "zero_optimization": {"stage": 3},
               "data_types": {"grad_accum_dtype": "bf16"}, "mi355x": {"direct_wgrad": direct}}
        eng, _, _, _ = ds.initialize(model=m, config=cfg)
        if direct:
            assert id(m.layers[0].block_sparse_moe.deepspeed_moe.experts.w13) in eng.optimizer._wgrad_ok
        g = torch.Generator(device="cuda").manual_seed(1)
        losses = []
        for _ in range(6):
            x = torch.randint(0, 512, (2, 256), device="cuda", generator=g)
            loss = eng(x, labels=x)
            eng.backward(loss)
            eng.step()
            losses.append(float(loss))
        res[direct] = losses
    assert res[True] == pytest.approx(res[False], rel=2e-2, abs=2e-2), res


# tiles of 16 weight rows (8 + 8 with the gate) and of 128 columns; more waves from K = 2048 on; rotated walks at multiples of 2048
@pytest.mark.parametrize("N,K", [(8, 128), (24, 384), (17, 1920), (40, 2048), (33, 2176), (16, 4096)])
@pytest.mark.parametrize("T,E,k", [(1, 8, 2), (5, 3, 2), (40, 4, 2)])  # fewer choices than experts; more; over 16 rows an expert
@pytest.mark.parametrize("glu", [0, 1])
def test_experts_of_few_rows(N, K, T, E, k, glu):
    from hcache_deepspeed_amd.ops import native
    gen = torch.Generator(device="cuda").manual_seed(N * K + T)

    def rand(*shape):
        return torch.randn(*shape, device="cuda", generator=gen).mul_(K**-0.25).to(torch.bfloat16)

    expert = torch.stack([torch.randperm(E, device="cuda", generator=gen)[:k] for _ in range(T)]).int()
    n, Ns, Ks = T * k, N + 8, 256
    x, w, xs, ws = rand(T, K), rand(E, (1 + glu) * N, K), rand(T, Ks), rand((1 + glu) * Ns, Ks)
    out, outs = torch.full((n + 1, N), 7.0, device="cuda", dtype=torch.bfloat16), rand(T, Ns)
    weight = torch.rand(n, device="cuda", generator=gen)
    native.check(
        native.kernels().hds_experts_skinny(glu, x.data_ptr(), K, w.data_ptr(), out.data_ptr(), N, expert.data_ptr(), n, k, E, N, K,
                                            xs.data_ptr(), Ks, ws.data_ptr(), outs.data_ptr(), Ns, T, Ns, Ks, 0, 0.0,
                                            weight.data_ptr(), native.stream()), "experts_skinny")

    def product(rows, m, scale):
        z = rows.double() @ m.double().T
        if not glu:
            return z
        g, u = (z * scale).chunk(2, -1)
        return torch.nn.functional.silu(g) * u

    for a in range(n):
        want = product(x[a // k], w[int(expert[a // k, a % k])], weight[a].double())
        # a result of bf16, and sums of K products in 32 bits
        torch.testing.assert_close(out[a].double(), want, rtol=2**-7, atol=1e-3)
    torch.testing.assert_close(outs.double(), product(xs, ws, 1.0), rtol=2**-7, atol=1e-3)
    assert (out[n:] == 7.0).all()


@pytest.mark.parametrize("T,R,K", [(1, 8, 128), (700, 65, 384), (1100, 65, 2048), (1623, 65, 2048), (1623, 33, 256),
                                   (2500, 65, 1024), (513, 257, 128)])
def test_router_logits_tiles(T, R, K):
    """16, 32, 48 and 80 routers a workgroup, by how many workgroups there are, with both sides' last tiles part-filled.
    The products are exact and summed in 32 bits: within K 2^-24 of their magnitudes' sum."""
    from hcache_deepspeed_amd.ops import native
    g = torch.Generator(device="cuda").manual_seed(T + R)
    x = torch.randn(T, K + 8, device="cuda", generator=g).bfloat16()[:, :K]
    w = torch.randn(R, K, device="cuda", generator=g).bfloat16()
    z = torch.full((T, R + 3), 7.0, device="cuda")
    native.check(native.kernels().hds_router_logits(x.data_ptr(), x.stride(0), w.data_ptr(), z.data_ptr(), R + 3, T, R, K,
                                                    native.stream()), "router_logits")
    bound = K * 2.0**-24 * (x.double().abs() @ w.double().abs().t())
    assert ((z[:, :R].double() - x.double() @ w.double().t()).abs() <= bound).all()
    assert (z[:, R:] == 7.0).all()


@pytest.mark.parametrize("T,R,K", [(1, 65, 4096), (64, 65, 4096), (64, 8, 4096)])
def test_router_logits_of_few_tokens_are_summed_in_short_chains(T, R, K):
    """Sixteen waves share a sum of few tokens. Its error grows with the root of a wave's chain of K / (32 waves) additions:
    1.15e-7 of the logits' norm at K = 4096, 1.36e-7 with eight waves. The bound lies between the two."""
    from hcache_deepspeed_amd.ops import native
    err = []
    for seed in range(20):
        g = torch.Generator(device="cuda").manual_seed(seed)
        w = torch.randn(R, K, device="cuda", generator=g).bfloat16() * 0.02
        x = torch.randn(T, K, device="cuda", generator=g).bfloat16()
        z = torch.empty(T, R, device="cuda")
        native.check(native.kernels().hds_router_logits(x.data_ptr(), K, w.data_ptr(), z.data_ptr(), R, T, R, K, native.stream()),
                     "router_logits")
        want = x.double() @ w.double().t()
        err.append(((z.double() - want).norm() / want.norm()).item())
    assert sum(err) / len(err) <= 1.25e-7
