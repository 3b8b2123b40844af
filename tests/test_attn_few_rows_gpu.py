"""FlashAttention forward by 128 rows a workgroup (csrc/kernels/flash_attn_pair.hip) and where the 256-row kernel takes over."""
import math

import pytest
import torch

from hcache_deepspeed_amd.ops.attention import flash_attn
from hcache_deepspeed_amd.ops.paged_prefill import make_portions, paged_attention_portions
from .test_paged_prefill import _setup

pytestmark = pytest.mark.gpu
D = 128


def _attend(q, k, v, first, causal, window):
    """64-bit output and logsumexp of [n, hq, D] queries at positions first .. over [m, hkv, D]."""
    k, v = (t.double().repeat_interleave(q.shape[1] // k.shape[1], 1).transpose(0, 1) for t in (k, v))
    s = q.double().transpose(0, 1) @ k.transpose(1, 2) / math.sqrt(D)
    at, mine = torch.arange(k.shape[1], device=q.device)[None], first + torch.arange(q.shape[0], device=q.device)[:, None]
    hide = at > mine if causal else torch.zeros_like(at > mine)
    if window:
        hide = hide | (at <= mine - window)
    s = s.masked_fill(hide, float("-inf"))
    return (torch.softmax(s, -1) @ v).transpose(0, 1), torch.logsumexp(s, -1)


def _close(got, want):
    """p is rounded to bf16 against a 32-bit sum and the result to bf16: 2^-8 of the norm twice, with room for two more."""
    assert (got.double() - want).norm() <= 4 * 2**-8 * want.norm()
    assert ((got.double() - want).norm(dim=-1) / want.norm(dim=-1)).max() < 0.03  # no single row off either


@pytest.mark.parametrize("causal,window", [(True, 0), (False, 0), (True, 1), (True, 70), (True, 200)])
@pytest.mark.parametrize("lens,hq,hkv", [([1], 2, 2), ([31, 33, 64], 4, 2), ([63, 65, 1, 96], 4, 1), ([127, 128, 129], 8, 2),
                                         ([191, 193, 255, 257], 2, 1), ([640, 1100], 16, 4), ([2050], 8, 8)])
def test_forward_of_few_rows(lens, hq, hkv, causal, window):
    """Edges of the 32 rows of a wave, of the 128 of a workgroup and of the tiles of 64 keys, one group without a tile, waves
    that end before others, windows that hide whole tiles of either group."""
    g = torch.Generator(device="cuda").manual_seed(sum(lens) + window)
    rnd = lambda h: torch.randn(sum(lens), h, D, device="cuda", generator=g).bfloat16()  # noqa: E731
    q, k, v = rnd(hq), rnd(hkv), rnd(hkv)
    cu = torch.tensor([0] + lens).cumsum(0).int()
    with torch.no_grad():
        o, lse = flash_attn(q, k, v, causal=causal, cu_seqlens=cu.cuda(), window=window, return_lse=True)
    for a, b in zip(cu[:-1].tolist(), cu[1:].tolist()):
        want, sums = _attend(q[a:b], k[a:b], v[a:b], 0, causal, window)
        _close(o[a:b], want)
        # a score of 128 products of bf16 values in 32 bits, and exp2 and log2 of a few units of the last place
        assert (lse.view(hq, -1)[:, a:b] - sums).abs().max() < 1e-4


def test_padded_batch_of_few_rows():
    g = torch.Generator(device="cuda").manual_seed(3)
    rnd = lambda h: torch.randn(3, 200, h, D, device="cuda", generator=g).bfloat16()  # noqa: E731
    q, k, v, lens = rnd(4), rnd(2), rnd(2), [200, 37, 129]
    k[1, 37:], v[1, 37:] = 300.0, 300.0
    with torch.no_grad():
        o = flash_attn(q, k, v, causal=False, seq_lens=torch.tensor(lens, dtype=torch.int32, device="cuda"))
    for i, n in enumerate(lens):
        _close(o[i, :n], _attend(q[i, :n], k[i, :n], v[i, :n], 0, False, 0)[0])


def test_many_blocks_take_the_larger_workgroups():
    """More 256-row workgroups than two a CU: sequences, and portions behind earlier tokens."""
    g = torch.Generator(device="cuda").manual_seed(4)
    rnd = lambda h: torch.randn(16, 1000, h, D, device="cuda", generator=g).bfloat16()  # noqa: E731
    q, k, v = rnd(16), rnd(4), rnd(4)
    with torch.no_grad():
        o = flash_attn(q, k, v, causal=True)
    for i in (0, 7, 15):
        _close(o[i], _attend(q[i], k[i], v[i], 0, True, 0)[0])
    lens, seen, hq, hkv = [257, 300, 10] * 5, [0, 130, 900] * 5, 32, 8
    cache, tab, metas, T, batch = _setup(lens, seen, hkv, 64, "cuda", torch.Generator().manual_seed(5))
    q = torch.randn(T, hq, D, device="cuda", generator=g).bfloat16()
    toks, blocks = make_portions(metas)
    assert not toks and len(blocks) // 2 * hq > 512
    o = paged_attention_portions(q, cache, None, torch.tensor(blocks, dtype=torch.int32, device="cuda").view(-1, 2), batch, hq, hkv,
                                 D**-0.5)
    for i, (q0, n, s) in enumerate(metas):
        at = torch.arange(s + n)
        kv = cache[tab[i, at // 64].long().cuda(), (at % 64).cuda()]
        _close(o[q0:q0 + n], _attend(q[q0:q0 + n], kv[:, 0], kv[:, 1], s, True, 0)[0])
