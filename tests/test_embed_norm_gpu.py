"""A step's embedding rows and their first norm by one kernel (csrc/kernels/norm.hip): the same bits as lookup and norm."""
import pytest
import torch

from hcache_deepspeed_amd.ops.embedding import lookup_rows, norm_rows
from hcache_deepspeed_amd.ops.norm import rms_norm


def test_other_calls_are_left():
    table, w, ids = torch.randn(9, 16), torch.ones(16), torch.tensor([1, 2])
    with torch.no_grad():
        assert norm_rows(table, ids, w, 1e-5) is None


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("W", [8, 512, 520, 2048, 4096, 8192])  # any width, one wave a row, several
@pytest.mark.parametrize("n", [1, 3, 64, 65, 700])  # several waves a row up to 64 rows
def test_rows_and_norm(dtype, W, n):
    g = torch.Generator(device="cuda").manual_seed(W + n)
    table = torch.randn(301, W, device="cuda", generator=g).to(dtype)
    w = torch.randn(W, device="cuda", generator=g).to(dtype)
    ids = torch.randint(0, 301, (n, ), device="cuda", generator=g)
    ids[0], ids[-1] = 0, 300
    with torch.no_grad():
        h, y = norm_rows(table, ids, w, 1e-5)
        assert torch.equal(h, lookup_rows(table, ids)) and torch.equal(y, rms_norm(h, w, 1e-5))
        ids[0] = -1
        ids[-1] = 301
        h, y = norm_rows(table, ids, w, 1e-5)
        assert all(t[i].isnan().all() for t in (h, y) for i in (0, -1))
        assert torch.equal(h[1:-1], table[ids[1:-1]])
    assert norm_rows(table, ids, w.clone().requires_grad_(), 1e-5) is None
    with torch.no_grad():
        assert norm_rows(table, ids.int(), w, 1e-5) is None and norm_rows(table[:, :W - 1], ids, w[:W - 1], 1e-5) is None
        if W > 8:
            assert norm_rows(table[:, 8:], ids, w[8:], 1e-5) is None
