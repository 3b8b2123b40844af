"""Embedding gradients of few ids, which are compared instead of sorted (csrc/kernels/token_ops.hip embed_bwd_few_kernel): the same
bits as from sorted ones, whose sums are in the same order."""
import pytest
import torch

from hcache_deepspeed_amd.ops import native
from hcache_deepspeed_amd.ops.embedding import embedding_grad_add_


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("n,V", [(1, 9), (63, 2000), (64, 3), (65, 2000), (1018, 32000), (4095, 40), (4096, 32000)])
@pytest.mark.parametrize("pad", [None, 1])
def test_few_ids(cuda, dtype, n, V, pad):
    lib = native.kernels()
    assert lib.hds_embed_bwd_few_max() == 4096
    g = torch.Generator(device="cuda").manual_seed(n)
    D = 520
    ids = torch.randint(0, V, (n, ), device="cuda", generator=g)
    if n > 2:
        ids[n // 2], ids[-1] = -1, V  # (ignored, as by the kernel of sorted ids)
    dy = torch.randn(n, D, device="cuda", generator=g).to(dtype)
    old = torch.randn(V, D, device="cuda", generator=g).to(dtype)
    got = embedding_grad_add_(old.clone(), ids, dy, pad)
    srt, perm = torch.sort(ids, stable=True)
    want = old.clone()
    native.check(lib.hds_embed_bwd(native.dt(want), dy.data_ptr(), srt.data_ptr(), perm.data_ptr(), want.data_ptr(), n, D, V,
                                   -1 if pad is None else pad, native.stream()), "embed_bwd")
    assert torch.equal(got, want)
    apart = torch.stack([ids, ids + 1], 1)[:, 0].to(torch.int32)  # strided, 32 bits
    assert torch.equal(embedding_grad_add_(old.clone(), apart, dy, pad), want)
