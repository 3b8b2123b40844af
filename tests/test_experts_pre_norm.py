"""The pre-norm that sums a routed layer's output on the way in (csrc/kernels/output_norm.hip ``experts_pre_norm_kernel``)."""
import pytest
import torch

from hcache_deepspeed_amd.ops.experts import ExpertSum
from hcache_deepspeed_amd.ops.norm import rms_norm
from hcache_deepspeed_amd.ops.output_norm import experts_pre_norm, sum_experts


def _parts(T, W, k, shared, sorted_rows, device, pad=0):
    g = torch.Generator().manual_seed(T + W)
    bf = lambda *s: torch.randn(*s, generator=g).to(torch.bfloat16).to(device)  # noqa: E731
    row = torch.randperm(T * k, generator=g).view(T, k).to(torch.int32).to(device) if sorted_rows else None
    p = ExpertSum(bf(T * k, W + pad), torch.randint(0, 8, (T, k), generator=g).to(torch.int32).to(device),
                  torch.rand(T, k, generator=g).to(device), row, 8)
    if shared:
        p.shared, p.gate = bf(T, W + pad), torch.randn(T, 9, generator=g).to(device)[:, 8]
    return p, bf(T, W), bf(W)


def _check(p, x, w):
    y, r = experts_pre_norm(p, x, w, 1e-5)
    yw, rw = rms_norm(sum_experts(x, p, torch.bfloat16), w, 1e-5, x)
    assert torch.equal(r, rw)
    # the row's sum of squares in another order: at most a rounding of the result
    assert ((y.double() - yw.double()).abs() <= 2**-7 * yw.double().abs()).all()


@pytest.mark.gpu
@pytest.mark.parametrize("W", [8, 128, 2040, 2048, 2056, 4096, 8192, 8200])
@pytest.mark.parametrize("T,k,shared,sorted_rows", [(1, 1, False, False), (4, 6, True, False), (65, 2, True, True), (3, 9, False, True)])
def test_norm_of_an_expert_sum(W, T, k, shared, sorted_rows):
    """Rows of one to four turns of a workgroup and their remainders; widths that two kernels take."""
    _check(*_parts(T, W, k, shared, sorted_rows, "cuda", pad=8))


def test_norm_of_an_expert_sum_elsewhere():
    _check(*_parts(3, 24, 2, True, True, "cpu"))


def test_parts_of_stock_modules_only():
    """A module that derives from the stock one and computes something else is called, not passed by."""
    from types import SimpleNamespace

    from hcache_deepspeed_amd.inference.v2.model import RaggedTransformer, _Layer
    from hcache_deepspeed_amd.inference.v2.modules import DSMoEConfig
    from hcache_deepspeed_amd.inference.v2.modules.implementations import DSPreRMSNorm, GroupedGemmMoE, RaggedUnembed

    class Own(GroupedGemmMoE):

        def forward(self, x, *a):
            return 2 * x

        def parts(self, *a):
            raise AssertionError("passed by")

    L = _Layer()
    L.w.update({"w13": torch.zeros(2, 8, 8), "w2": torch.zeros(2, 8, 4), "router.w": None})
    L.routed = {}
    m = SimpleNamespace(tp=1, layers=[L], moe_mod=Own(DSMoEConfig(8, 4, 2, 1, "silu_glu", True)),
                        norm_mod=DSPreRMSNorm(None), unembed_mod=RaggedUnembed(None))
    x = torch.ones(3, 8)
    assert RaggedTransformer._expert_parts(m, L, x) is None
    m._moe = lambda L, x: RaggedTransformer._moe(m, L, x)
    assert torch.equal(RaggedTransformer._mlp(m, L, x), 2 * x)
