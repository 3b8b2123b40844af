"""Prefill attention by 128 rows a workgroup (csrc/kernels/flash_attn_pair.hip) and where the 256-row kernel takes over."""
import math

import pytest
import torch

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


@pytest.mark.parametrize("window", [0, 1, 70, 200])
@pytest.mark.parametrize("lens,seen,hq,hkv", [([1], [0], 2, 2), ([31, 33, 64], [0, 1, 63], 4, 2), ([63, 65, 1, 96], [65, 0, 300, 33], 4, 1),
                                              ([127, 128, 129], [0, 64, 127], 8, 2), ([191, 193, 255, 257], [1, 0, 130, 5000], 2, 1),
                                              ([640, 1100], [0, 333], 16, 4), ([2050], [0], 8, 8)])
def test_portions_of_few_rows(lens, seen, hq, hkv, window):
    """Edges of the 32 rows of a wave, of the 128 of a workgroup and of the tiles of 64 keys, one group without a tile, waves
    that end before others, windows that hide whole tiles of either group, more than 64 tiles."""
    g = torch.Generator(device="cuda").manual_seed(sum(lens) + window)
    cache, tab, metas, T, batch = _setup(lens, seen, hkv, 64, "cuda", torch.Generator().manual_seed(6))
    q = torch.randn(T, hq, D, device="cuda", generator=g).bfloat16()
    blocks = [(i, r) for i, n in enumerate(lens) for r in range(0, n, 256)]
    assert len(blocks) * hq <= 512
    o = paged_attention_portions(q, cache, None, torch.tensor(blocks, dtype=torch.int32, device="cuda"), batch, hq, hkv, D**-0.5,
                                 window)
    for i, (q0, n, s) in enumerate(metas):
        at = torch.arange(s + n)
        kv = cache[tab[i, at // 64].long().cuda(), (at % 64).cuda()]
        _close(o[q0:q0 + n], _attend(q[q0:q0 + n], kv[:, 0], kv[:, 1], s, True, window)[0])


def test_many_blocks_take_the_larger_workgroups():
    """More 256-row workgroups than two a CU."""
    g = torch.Generator(device="cuda").manual_seed(4)
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


@pytest.mark.parametrize("few", [True, False])
@pytest.mark.parametrize("what,window", [("query", 0), ("query", 100), ("inf", 0), ("inf", 100), ("nan", 0), ("nan", 100), ("tile", 0),
                                         ("all", 0)])
def test_values_that_are_not_finite(what, window, few):
    """On either side of the 512 workgroups: rows of a NaN query (with and without masked keys in their last tile), rows that
    see a score of plus infinity, a NaN key, or minus infinity alone come out NaN, as softmax gives them; scores of minus
    infinity, a whole tile of them too, count nothing. Finite rows as above."""
    g = torch.Generator(device="cuda").manual_seed(7)
    lens, seen, hq, hkv = ([130, 300, 40], [64, 200, 0], 8, 2) if few else ([130, 300] * 6, [64, 200] * 6, 32, 8)
    cache, tab, metas, T, batch = _setup(lens, seen, hkv, 64, "cuda", torch.Generator().manual_seed(8))
    q = torch.randn(T, hq, D, device="cuda", generator=g).bfloat16()
    blocks = [(i, r) for i, n in enumerate(lens) for r in range(0, n, 256)]
    assert (len(blocks) * hq <= 512) == few
    for i, (q0, n, s) in enumerate(metas):
        at = torch.arange(s + n)
        blk, slot = tab[i, at // 64].long().cuda(), (at % 64).cuda()
        if what == "query":
            for row in {63 - s % 64, 0, 17, n // 2, n - 1} & set(range(n)):
                q[q0 + row] = math.nan
        elif what in ("inf", "nan"):  # half of the queries see plus, half minus infinity
            first = s + n // 3
            cache[blk[first], slot[first], 0, :, 0] = math.inf if what == "inf" else math.nan
        else:
            gone = slice(64, 128) if what == "tile" else slice(None)
            q[q0:q0 + n, :, 0] = 1
            cache[blk[gone], slot[gone], 0, :, 0] = -math.inf
    o = paged_attention_portions(q, cache, None, torch.tensor(blocks, dtype=torch.int32, device="cuda"), batch, hq, hkv, D**-0.5,
                                 window)
    for i, (q0, n, s) in enumerate(metas):
        at = torch.arange(s + n)
        kv = cache[tab[i, at // 64].long().cuda(), (at % 64).cuda()]
        want, got = _attend(q[q0:q0 + n], kv[:, 0], kv[:, 1], s, True, window)[0].transpose(0, 1), o[q0:q0 + n].transpose(0, 1)
        gone = want.isnan().any(-1)
        assert what == "tile" or gone.any()
        assert got[gone].isnan().all() and not got[~gone].isnan().any(), i
        if not gone.all():
            _close(got[~gone], want[~gone])


@pytest.mark.parametrize("hq,hkv", [(1, 1), (3, 1), (6, 2), (12, 4), (24, 8), (40, 8), (64, 8)])
def test_every_row_of_every_head(hq, hkv):
    """Short entries between long ones, heads and entries that do not fill a group of the launch's order."""
    g = torch.Generator(device="cuda").manual_seed(hq)
    lens, seen = [256, 9, 129, 1, 128, 300, 20], [0, 70, 3, 64, 0, 5, 130]
    cache, tab, metas, T, batch = _setup(lens, seen, hkv, 64, "cuda", torch.Generator().manual_seed(9))
    q = torch.randn(T, hq, D, device="cuda", generator=g).bfloat16()
    blocks = [(i, r) for i, n in enumerate(lens) for r in range(0, n, 256)]
    assert len(blocks) * hq <= 512
    o = paged_attention_portions(q, cache, None, torch.tensor(blocks, dtype=torch.int32, device="cuda"), batch, hq, hkv, D**-0.5)
    for i, (q0, n, s) in enumerate(metas):
        at = torch.arange(s + n)
        kv = cache[tab[i, at // 64].long().cuda(), (at % 64).cuda()]
        _close(o[q0:q0 + n], _attend(q[q0:q0 + n], kv[:, 0], kv[:, 1], s, True, 0)[0])


@pytest.mark.parametrize("rows", [128, 256])
def test_either_kernel_on_request(rows):
    """The caller's choice, on both sides of where the length of the list would make it."""
    g = torch.Generator(device="cuda").manual_seed(3)
    for lens, seen, hq, hkv in (([200, 300], [60, 5], 8, 2), ([200, 70, 140] * 6, [60, 0, 500] * 6, 32, 8)):
        cache, tab, metas, T, batch = _setup(lens, seen, hkv, 64, "cuda", torch.Generator().manual_seed(2))
        q = torch.randn(T, hq, D, device="cuda", generator=g).bfloat16()
        blocks = torch.tensor([(i, r) for i, n in enumerate(lens) for r in range(0, n, 256)], dtype=torch.int32, device="cuda")
        o = paged_attention_portions(q, cache, None, blocks, batch, hq, hkv, D**-0.5, rows=rows)
        for i, (q0, n, s) in enumerate(metas):
            at = torch.arange(s + n)
            kv = cache[tab[i, at // 64].long().cuda(), (at % 64).cuda()]
            _close(o[q0:q0 + n], _attend(q[q0:q0 + n], kv[:, 0], kv[:, 1], s, True, 0)[0])
        with pytest.raises(RuntimeError):
            paged_attention_portions(q, cache, None, blocks, batch, hq, hkv, D**-0.5, rows=64)
