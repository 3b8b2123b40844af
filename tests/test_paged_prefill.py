"""Attention of steps that mix single tokens and portions of prompts over the paged cache: the prefill kernel
(csrc/kernels/flash_attn_w64.hip over block tables) and the division of a step, against float64 over the same tables."""
import math
import types

import pytest
import torch

from hcache_deepspeed_amd.inference.v2.modules.configs import DSSelfAttentionConfig
from hcache_deepspeed_amd.inference.v2.modules.implementations import DSDenseBlockedAttention
from hcache_deepspeed_amd.ops.paged import DECODE_MAX, build_atoms
from hcache_deepspeed_amd.ops.paged_prefill import divide_step, make_portions, paged_attention_portions, portions_ok

D = 128


def test_portions_cover_every_token_once():
    metas, q0 = [], 0
    for n, seen in [(1, 50), (700, 0), (DECODE_MAX, 9), (DECODE_MAX + 1, 1000), (0, 3), (256, 7), (257, 0)]:
        metas.append((q0, n, seen))
        q0 += n
    toks, flat = make_portions(metas)
    blocks = list(zip(flat[::2], flat[1::2]))
    rows = set(toks)
    for s, r in blocks:
        own = range(metas[s][0] + r, metas[s][0] + min(r + 256, metas[s][1]))
        assert len(own) and not rows & set(own)
        rows |= set(own)
    assert rows == set(range(q0)) and len(toks) == 1 + DECODE_MAX
    last = [metas[s][2] + min(r + 256, metas[s][1]) for s, r in blocks]
    assert last == sorted(last, reverse=True)


@pytest.mark.parametrize("lens,seen,heads,one_by_one,kernel", [
    ([512, 1, 1], [700, 3000, 9], (32, 8), [1, 1], "prefill"),        # a piece of a prompt beside single tokens
    ([2048], [0], (32, 8), [], "prefill"), ([9], [0], (8, 1), [], "prefill"),
    ([8] * 8 + [1], [3000] * 9, (32, 8), [8] * 8 + [1], None),        # few sequences of a few tokens each
    ([8] * 32 + [1], [2400] * 33, (32, 8), [], "rows"),               # many of them
    ([1] * 100 + [8] * 32, [4000] * 100 + [200, 1000] * 16, (32, 8), [1] * 100, "rows"),
    ([4] * 32, [200, 1000] * 16, (32, 8), [4] * 32, None), ([8] * 32, [200, 1000] * 16, (16, 4), [8] * 32, None),
    ([16] * 32 + [1, 0], [2400] * 34, (32, 8), [], "rows"),           # many short portions
    ([60] * 30, [0] * 30, (32, 32), [], "rows"), ([20] * 32, [2400] * 32, (32, 32), [], "prefill"),
    ([16] * 8, [2400] * 8, (32, 8), [], "prefill"), ([256] * 32, [2400] * 32, (32, 8), [], "prefill"),
    ([8] * 32 + [512] * 4, [2400] * 36, (32, 32), [], "prefill")])
def test_division_of_a_step(lens, seen, heads, one_by_one, kernel):
    """Which kernel runs which sequences, and that every row of every head runs once."""
    metas, q0 = [], 0
    for n, s in zip(lens, seen):
        metas.append((q0, n, s))
        q0 += n
    toks, blocks, atoms = divide_step(metas, *heads)
    assert len(toks) == sum(one_by_one) and bool(blocks) == (kernel == "prefill") and bool(atoms) == (kernel == "rows")
    G = heads[0] // heads[1]
    seen_rows = [(t, h) for t in toks for h in range(heads[0])]
    for s, r in zip(blocks[::2], blocks[1::2]):
        q0, n, _ = metas[s]
        seen_rows += [(q0 + i, h) for i in range(r, min(r + 256, n)) for h in range(heads[0])]
    for s, hk, r in zip(atoms[::3], atoms[1::3], atoms[2::3]):
        q0, n, _ = metas[s]
        seen_rows += [(q0 + i // G, hk * G + i % G) for i in range(r, min(r + 128, n * G))]
    assert len(seen_rows) == len(set(seen_rows)) == sum(lens) * heads[0]


def _setup(lens, seen, hkv, bs, device, g):
    need = [-(-(n + s) // bs) for n, s in zip(lens, seen)]
    width = max(need) + 1
    perm = torch.randperm(sum(need) + 3, generator=g)
    tab = torch.zeros(len(lens), width, dtype=torch.int32)
    k = 0
    for i, m in enumerate(need):
        tab[i, :m] = perm[k:k + m].int()
        k += m
    cache = torch.randn(sum(need) + 3, bs, 2, hkv, D, generator=g).bfloat16().to(device)
    metas, q0 = [], 0
    for n, s in zip(lens, seen):
        metas.append((q0, n, s))
        q0 += n
    seq = torch.tensor([i for i, n in enumerate(lens) for _ in range(n)], dtype=torch.int32)
    pos = torch.tensor([s + j for n, s in zip(lens, seen) for j in range(n)], dtype=torch.int32)
    batch = types.SimpleNamespace(seq_meta=torch.tensor(metas, dtype=torch.int32).to(device), tok_seq=seq.to(device),
                                  tok_pos=pos.to(device), block_tables=tab.to(device))
    return cache, tab, metas, q0, batch


@pytest.mark.gpu
@pytest.mark.parametrize("lens,seen,hq,hkv,bs,window", [
    ([9], [0], 8, 2, 64, 0), ([64, 1, 65], [0, 700, 63], 16, 4, 64, 0), ([256, 8, 257], [1, 130, 64], 4, 4, 128, 0),
    ([300, 1, 1], [5000, 4500, 3], 8, 1, 64, 0), ([1100], [0], 6, 2, 192, 0), ([513, 20], [100, 900], 32, 8, 64, 200),
    ([40], [4090], 8, 8, 64, 64), ([2, 3], [500, 17], 8, 2, 64, 0), ([4400], [0], 2, 1, 64, 0)])
def test_portions_match_float64(lens, seen, hq, hkv, bs, window):
    """Tails of the 64-key tiles and of the 256-token workgroups, a portion behind a long context (more than 64 tiles, the
    run of cache slots that a wave holds at a time), windows, blocks of several tiles, head counts that are no multiple of
    8. p is rounded to bf16 against a 32-bit sum and the result to bf16: 2^-8 of the norm twice, with room for two more."""
    g = torch.Generator().manual_seed(sum(lens) + hq)
    dev = torch.device("cuda")
    cache, tab, metas, T, batch = _setup(lens, seen, hkv, bs, dev, g)
    qkv = torch.randn(T, hq + 2 * hkv, D, generator=g).bfloat16().to(dev)
    q = qkv[:, :hq]
    assert portions_ok(q, cache, hq, hkv)
    toks, blocks = make_portions(metas)
    toks = torch.tensor(toks, dtype=torch.int32, device=dev) if toks else None
    blocks = torch.tensor(blocks, dtype=torch.int32, device=dev).view(-1, 2) if blocks else None
    scale = 1 / math.sqrt(D)
    o = paged_attention_portions(q, cache, toks, blocks, batch, hq, hkv, scale, window)
    for i, (q0, n, s) in enumerate(metas):
        at = torch.arange(s + n)
        rows = cache[tab[i, at // bs].long().to(dev), (at % bs).to(dev)].double()
        k, v = (rows[:, j].repeat_interleave(hq // hkv, 1).transpose(0, 1) for j in (0, 1))
        sc = q[q0:q0 + n].double().transpose(0, 1) @ k.transpose(1, 2) * scale
        mine = (s + torch.arange(n))[:, None]
        hide = at[None] > mine
        if window:
            hide |= at[None] <= mine - window
        want = (torch.softmax(sc.masked_fill(hide.to(dev), float("-inf")), -1) @ v).transpose(0, 1)
        got = o[q0:q0 + n].double()
        assert (got - want).norm() <= 4 * 2**-8 * want.norm(), i
        worst = (got - want).norm(dim=-1) / want.norm(dim=-1)  # no single row off either
        assert worst.max() < 0.03, (i, worst.max())


@pytest.mark.gpu
@pytest.mark.parametrize("lens,window", [([20] * 40 + [1, 1], 0), ([8] * 40 + [1] * 3, 0), ([33, 2] * 20, 90)])
def test_many_short_portions_match_float64(lens, window):
    """Steps that run in row blocks beside single tokens; the bounds of the test above."""
    seen = [(37 * i) % 290 for i in range(len(lens))]
    hq, hkv = 32, 8
    g = torch.Generator().manual_seed(len(lens))
    dev = torch.device("cuda")
    cache, tab, metas, T, batch = _setup(lens, seen, hkv, 64, dev, g)
    q = torch.randn(T, hq, D, generator=g).bfloat16().to(dev)
    i32 = lambda v, shape: torch.tensor(v, dtype=torch.int32, device=dev).view(shape) if v else None  # noqa: E731
    toks, blocks, atoms = divide_step(metas, hq, hkv)
    assert atoms and not blocks
    o = paged_attention_portions(q, cache, i32(toks, (-1, )), None, batch, hq, hkv, D**-0.5, window, i32(atoms, (-1, 3)))
    for i, (q0, n, s) in enumerate(metas):
        at = torch.arange(s + n)
        rows = cache[tab[i, at // 64].long().to(dev), (at % 64).to(dev)].double()
        k, v = (rows[:, j].repeat_interleave(hq // hkv, 1).transpose(0, 1) for j in (0, 1))
        sc = q[q0:q0 + n].double().transpose(0, 1) @ k.transpose(1, 2) * D**-0.5
        mine = (s + torch.arange(n))[:, None]
        hide = at[None] > mine
        if window:
            hide |= at[None] <= mine - window
        want = (torch.softmax(sc.masked_fill(hide.to(dev), float("-inf")), -1) @ v).transpose(0, 1)
        worst = (o[q0:q0 + n].double() - want).norm(dim=-1) / want.norm(dim=-1)
        assert worst.max() < 0.03, (i, worst.max())


@pytest.mark.gpu
@pytest.mark.parametrize("scale", [0.0, -0.09, 1e-30, -1e-30, 0.09, 2.0])
def test_any_scale_in_a_portion(scale):
    """The attention module takes any scale: zero and tiny ones give every visible key the same weight, negative ones turn the
    order round. The prefill kernel takes positive ones, the others run in row blocks. Bounds as above."""
    lens, seen, hq, hkv = [70, 1, 300], [100, 50, 7], 8, 2
    g = torch.Generator().manual_seed(5)
    dev = torch.device("cuda")
    cache, tab, metas, T, batch = _setup(lens, seen, hkv, 64, dev, g)
    qkv = torch.randn(T, hq + 2 * hkv, D, generator=g).bfloat16().to(dev)
    i32 = lambda v, shape: torch.tensor(v, dtype=torch.int32, device=dev).view(shape) if v else None  # noqa: E731
    toks, blocks, rows = divide_step(metas, hq, hkv)
    assert blocks and portions_ok(qkv[:, :hq], cache, hq, hkv, scale) == (scale > 1e-20)
    batch.portions = i32(toks, (-1, )), i32(blocks, (-1, 2)), i32(rows, (-1, 3))
    atoms, batch.n_atoms = build_atoms(metas, hq, hkv)
    batch.atoms = atoms.to(dev)
    batch.current_sequences, batch.max_new, batch.seq_meta_host, batch.tables_host = len(lens), max(lens), metas, tab
    o = DSDenseBlockedAttention(DSSelfAttentionConfig(hq, hkv, D, scale_factor=scale, positional_embedding_type="none"))(
        qkv, cache, batch, None, None).view(T, hq, D)
    for i, (q0, n, s) in enumerate(metas):
        at = torch.arange(s + n)
        kv = cache[tab[i, at // 64].long().to(dev), (at % 64).to(dev)].double()
        k, v = (kv[:, j].repeat_interleave(hq // hkv, 1).transpose(0, 1) for j in (0, 1))
        sc = qkv[q0:q0 + n, :hq].double().transpose(0, 1) @ k.transpose(1, 2) * scale
        hide = at[None] > (s + torch.arange(n))[:, None]
        want = (torch.softmax(sc.masked_fill(hide.to(dev), float("-inf")), -1) @ v).transpose(0, 1)
        worst = (o[q0:q0 + n].double() - want).norm(dim=-1) / want.norm(dim=-1)
        assert worst.max() < 0.03, (i, worst.max())


@pytest.mark.gpu
@pytest.mark.parametrize("window", [0, 100])
@pytest.mark.parametrize("later", ["rising", math.inf, -math.inf, math.nan])
def test_later_keys_do_not_reach_earlier_rows(later, window):
    """Scores that rise by 131,072 a position, so that every masked one is far above the visible ones, and keys that are
    infinite or NaN from the middle of a portion on: rows in front of them are what they are without them."""
    lens, seen, hq, hkv = [300, 130], [37, 0], 8, 2
    g = torch.Generator().manual_seed(1)
    dev = torch.device("cuda")
    cache, tab, metas, T, batch = _setup(lens, seen, hkv, 64, dev, g)
    qkv = torch.randn(T, hq + 2 * hkv, D, generator=g).bfloat16().to(dev)
    u = torch.where(torch.rand(D, generator=g) < 0.5, -1.0, 1.0).bfloat16().to(dev)
    good = []
    for i, (q0, n, s) in enumerate(metas):
        at = torch.arange(s + n)
        blk, slot = tab[i, at // 64].long().to(dev), (at % 64).to(dev)
        if later == "rising":
            qkv[q0:q0 + n, :hq] = 16 * u
            cache[blk, slot, 0] = ((at // 4) * 256).bfloat16().to(dev)[:, None, None] * u
        else:
            cache[blk[s + n // 2:], slot[s + n // 2:], 0] = later
        good.append(n if later == "rising" else n // 2)
    q = qkv[:, :hq]
    toks, blocks = make_portions(metas)
    assert not toks
    blocks = torch.tensor(blocks, dtype=torch.int32, device=dev).view(-1, 2)
    o = paged_attention_portions(q, cache, None, blocks, batch, hq, hkv, 1 / math.sqrt(D), window)
    for i, (q0, _, s) in enumerate(metas):
        n = good[i]
        at = torch.arange(s + n)
        rows = cache[tab[i, at // 64].long().to(dev), (at % 64).to(dev)].double()
        k, v = (rows[:, j].repeat_interleave(hq // hkv, 1).transpose(0, 1) for j in (0, 1))
        sc = q[q0:q0 + n].double().transpose(0, 1) @ k.transpose(1, 2) / math.sqrt(D)
        mine = (s + torch.arange(n))[:, None]
        hide = at[None] > mine
        if window:
            hide |= at[None] <= mine - window
        want = (torch.softmax(sc.masked_fill(hide.to(dev), float("-inf")), -1) @ v).transpose(0, 1)
        got = o[q0:q0 + n].double()
        worst = (got - want).norm(dim=-1) / want.norm(dim=-1)  # p and the result rounded to bf16, as above
        assert torch.isfinite(got).all() and worst.max() < 0.03, (i, worst.max())


def test_division_is_made_for_models_that_use_it(monkeypatch):
    """Neither for the hybrid designs, whose mixers plan their own steps, nor where the kernels do not apply."""
    from hcache_deepspeed_amd.inference.v2 import build_engine_from_model
    from hcache_deepspeed_amd.models.llama import LlamaForCausalLM, tiny
    from hcache_deepspeed_amd.ops import paged_prefill

    from .test_gofasun import engine
    made = []
    monkeypatch.setattr(paged_prefill, "divide_step", lambda *a: made.append(a) or divide_step(*a))
    cpu = torch.device("cpu")
    dense = build_engine_from_model(LlamaForCausalLM(tiny()).eval(), {"dtype": "fp32"}, device=cpu, num_kv_blocks=8)
    for eng in (engine("mixed", (cpu, torch.float32)), dense):
        eng.put([1, 2], [torch.arange(20) % 7, torch.arange(3)], capture_latents=False)
    assert not made
    dense._batch.set_attention_geometry(4, 2, 128)
    dense.put([1, 2], [torch.arange(20) % 7, torch.arange(3)], capture_latents=False)
    assert len(made) == 1


@pytest.mark.gpu
def test_engine_steps_in_pieces_match_whole_prompts():
    """A prompt taken in pieces beside decoding sequences gives the logits of the prompt taken whole."""
    from hcache_deepspeed_amd.inference.v2.engine import build_engine_from_model
    from hcache_deepspeed_amd.models.llama import LlamaForCausalLM, tiny
    torch.manual_seed(0)
    m = LlamaForCausalLM(tiny(vocab_size=211)).eval()
    conf = dict(dtype="bf16", state_manager={"max_context": 1024, "kv_block_size": 64, "max_ragged_batch_size": 1024})
    g = torch.Generator().manual_seed(3)
    prompt, other = (torch.randint(0, 211, (n, ), generator=g) for n in (700, 90))
    step = [torch.randint(0, 211, (1, ), generator=g) for _ in range(3)]
    dev = torch.device("cuda")
    eng = build_engine_from_model(m, conf, device=dev, num_kv_blocks=40)
    eng.put([1], [other], capture_latents=False)
    got = [eng.put([1, 2], [t, p], capture_latents=False)[0].float() for t, p in zip(step, prompt.split(256))]
    ref = build_engine_from_model(m, conf, device=dev, num_kv_blocks=40)
    ref.put([1], [other], capture_latents=False)
    for i, t in enumerate(step):
        a = ref.put([1], [t], capture_latents=False)[0].float()
        b = ref.put([2], [prompt[:256 * (i + 1)]], capture_latents=False)[0].float()
        ref.flush(2)
        want = torch.cat([a, b])
        assert (got[i] - want).norm() < 2e-2 * want.norm()
