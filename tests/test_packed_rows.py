"""What the products of more rows on packed weights refuse (ops/quantizer.py ``_packed_rows``), without a GPU."""
import types

import pytest
import torch

from hcache_deepspeed_amd.ops import quantizer as Q

M, N, K, G = 128, 512, 1024, 128


@pytest.fixture
def launched(monkeypatch):
    """The kernel's arguments; tensors pass for such of the GPU."""
    calls = []
    lib = types.SimpleNamespace(hds_packed_rows=lambda *a: calls.append(a) or 0)
    monkeypatch.setattr(Q.native, "kernels", lambda: lib)
    monkeypatch.setattr(Q.native, "stream", lambda: 0)
    monkeypatch.setattr(Q, "_packed_plan", lambda *a: 16)
    return calls


def _rows(n=N, k=K, scales=N * K // G, bias=None, glu=0, dev=("cpu", "cpu")):
    return Q._packed_rows(torch.zeros(M, k, dtype=torch.bfloat16), torch.zeros(N * K, dtype=torch.int8, device=dev[0]),
                          torch.zeros(scales, device=dev[1]), n, k, G, "int8", 3, bias, glu)


def test_sizes_are_those_of_the_weight(launched):
    """The dequantized weight has as many values as the scales say: another size than the call's is refused, not read."""
    assert _rows().shape == (M, N) and len(launched) == 1
    assert _rows(n=2 * N) is None and _rows(n=N // 2) is None and _rows(k=2 * K) is None and _rows(scales=N) is None
    assert _rows(n=N // 2, glu=1).shape == (M, N // 2) and _rows(n=N, glu=1) is None
    assert _rows(dev=("meta", "cpu")) is None and _rows(dev=("cpu", "meta")) is None  # another device than the rows'
    assert len(launched) == 2


def test_bias_is_a_row_of_the_result(launched):
    for bias in (torch.zeros(N - 8, dtype=torch.bfloat16), torch.zeros(1, dtype=torch.bfloat16), torch.zeros(N), torch.zeros(1, N).bfloat16(),
                 torch.zeros(N, dtype=torch.bfloat16, device="meta")):
        assert _rows(bias=bias) is None
    assert not launched and _rows(bias=torch.zeros(N).bfloat16()).shape == (M, N)


def test_row_limit_of_the_environment(launched, monkeypatch):
    """HDS_WMIX_MAX_M bounds these tiles too, but not the few rows that would run as a stream otherwise."""
    monkeypatch.setattr(Q, "_PACKED_MAX_M", M - 1)
    assert _rows() is None and not launched
    monkeypatch.setattr(Q, "_PACKED_MAX_M", M)
    assert _rows() is not None
    monkeypatch.setattr(Q, "_PACKED_MAX_M", 0)
    monkeypatch.setitem(globals(), "M", 16)
    assert _rows() is not None
