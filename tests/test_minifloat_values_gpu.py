"""Minifloat dequantization by whole vectors (csrc/kernels/fpq.hip)."""
import pytest
import torch

from hcache_deepspeed_amd.ops import quantizer as Q

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("q_bits,mantissa", [(6, 1), (6, 2), (6, 3), (8, 1), (8, 3), (12, 4), (12, 7), (12, 9)])
@pytest.mark.parametrize("groups,G", [(1, 16), (3, 48), (514, 64), (5, 12), (33, 512)])
def test_minifloat_values_are_those_of_the_reference(dtype, q_bits, mantissa, groups, G):
    """Every code, subnormal and negative zero included, bit for bit; groups of whole 16s and others."""
    g = torch.Generator().manual_seed(G + q_bits)
    q = torch.randint(0, 256, (groups * G * q_bits // 8, ), generator=g, dtype=torch.uint8)
    s = torch.rand(groups, generator=g) + 0.5
    want = Q.dequantize_minifloat(q, s, G, q_bits, mantissa, dtype)
    got = Q.dequantize_minifloat(q.cuda(), s.cuda(), G, q_bits, mantissa, dtype).cpu()
    view = torch.int32 if dtype == torch.float32 else torch.int16
    assert torch.equal(got.view(view), want.view(view))
