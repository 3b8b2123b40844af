"""What a decode step does around its layers: embedding rows, the rows whose logits are wanted, the step's description."""
import pytest
import torch
import torch.nn.functional as F

from hcache_deepspeed_amd.inference.v2.modules import DSUnembedConfig, instantiate_unembed
from hcache_deepspeed_amd.ops.embedding import lookup_rows


@pytest.mark.gpu
@pytest.mark.parametrize("dtype,W", [(torch.bfloat16, 8), (torch.bfloat16, 2056), (torch.float32, 4096), (torch.bfloat16, 12)])
@pytest.mark.parametrize("n", [0, 1, 16, 700])
def test_lookup_rows_gpu(dtype, W, n):
    table = torch.randn(301, W, device="cuda").to(dtype)
    ids = torch.randint(0, 301, (n, ), device="cuda")
    ids[:1] = 300
    assert torch.equal(lookup_rows(table, ids), F.embedding(ids, table))
    if W % 8 == 0 and n > 1:
        ids[1] = 301
        out = lookup_rows(table, ids)
        assert out[1].isnan().all() and torch.equal(out[0], table[300])


def _unembed(norm, dev, W, n, T, seed=0):
    g = torch.Generator().manual_seed(seed)
    r = lambda *s: torch.randn(*s, generator=g).to(dev, torch.bfloat16)  # noqa: E731
    h, res, w, b, lm = r(T, W), r(T, W), r(W), r(W) if norm == "layer" else None, r(48, W)
    mod = instantiate_unembed(DSUnembedConfig(model_dim=W, vocab_size=48, norm_type=norm))
    return mod, h, res, w, b, lm


def _plain(norm, h, res, w, b, lm, idx, final=True):
    x = (h[idx].float() + res[idx].float()).to(h.dtype)
    if final:
        xf = x.float()
        if norm == "layer":
            y = F.layer_norm(xf, xf.shape[-1:], w.float(), b.float(), 1e-5)
        else:
            y = xf * torch.rsqrt((xf * xf).mean(-1, keepdim=True) + 1e-5) * w.float()
        x = y.to(h.dtype)
    return x.float() @ lm.float().t()


class _Batch:
    pass


@pytest.mark.parametrize("dev", ["cpu", pytest.param("cuda", marks=pytest.mark.gpu)])
@pytest.mark.parametrize("norm", ["rms", "layer"])
@pytest.mark.parametrize("W", [512, 4096, 648])
@pytest.mark.parametrize("pick,new,last,dtype", [
    ([0, 1, 2], 1, True, torch.int32),      # single tokens: every row
    ([2, 6, 6, 0], 4, True, torch.int32),   # last tokens of portions, in any order
    ([2, -1, 0], 4, False, torch.int32),    # rows of the caller's choice
    ([2, 6, 0], 4, True, torch.int64),
])
@pytest.mark.parametrize("final", [True, False])
def test_wanted_rows(dev, norm, W, pick, new, last, dtype, final):
    T = 3 if new == 1 else 7
    mod, h, res, w, b, lm = _unembed(norm, dev, W, len(pick), T)
    batch = _Batch()
    batch.last_token_idx = torch.tensor(pick, dtype=dtype, device=dev)
    batch.logits_of_last_tokens, batch.max_new, batch.current_sequences = last, new, len(pick)
    with torch.no_grad():
        got = mod(h, res, batch, lm, None, w if final else None, b, 1e-5)
    want = _plain(norm, h.cpu(), res.cpu(), w.cpu(), None if b is None else b.cpu(), lm.cpu(), batch.last_token_idx.cpu().long(),
                  final)
    # two roundings to bf16 of the row (2^-9 each) through W products of unit variance, and the logit's own
    bound = 6 * 2**-8 * lm.cpu().float().norm(dim=1) * (w.abs().max().item() if final else 2) + 2**-8 * want.abs()
    assert (got.cpu().float() - want).abs().le(bound).all()


def test_step_description_on_the_host():
    """Ids, metadata and the division of a mixed step are views of one buffer."""
    from hcache_deepspeed_amd.inference.v2.ragged import (BlockedKVCache, DSStateManager, DSStateManagerConfig,
                                                          RaggedBatchWrapper)
    cfg = DSStateManagerConfig(max_context=256)
    kv = BlockedKVCache(1, 2, 16, 64, torch.float32, torch.device("cpu"), cfg.memory_config, num_blocks=8)
    sm = DSStateManager(cfg, kv)
    b = RaggedBatchWrapper(cfg, torch.device("cpu"), sm.max_blocks_per_seq)
    b.set_attention_geometry(4, 2, 128)
    for lens in ([1], [1, 1, 1], [3, 1, 20], [5]):
        b.clear()
        toks = [torch.arange(n) + 2**33 * (i + 1) for i, n in enumerate(lens)]
        for i, t in enumerate(toks):
            seq = sm.get_or_create_sequence(i)
            sm.maybe_allocate_kv(seq, len(t))
            b.insert_sequence(seq, t)
        b.finalize()
        assert torch.equal(b.input_ids, torch.cat(toks)) and b.input_ids.dtype == torch.int64
        T, S = sum(lens), len(lens)
        assert b.tok_seq.tolist() == [i for i, n in enumerate(lens) for _ in range(n)]
        assert b.tok_pos.tolist() == [j for n in lens for j in range(n)]
        assert b.last_token_idx.tolist() == [sum(lens[:i + 1]) - 1 for i in range(S)]
        assert torch.equal(b.tables_host, b.block_tables) and b.block_tables.shape == (S, sm.max_blocks_per_seq)
        for i in range(S):
            blocks = sm.get_sequence(i).kv_blocks
            assert b.block_tables[i, :len(blocks)].tolist() == blocks
        assert b.slots.tolist() == [sm.get_sequence(i).tracking_id for i in range(S)] and b.current_tokens == T


def test_step_description_of_any_tokens():
    """Ids of other types and strides, more of them than the first buffer holds, wanted places, an empty step, refused ids."""
    from hcache_deepspeed_amd.inference.v2.ragged import (BlockedKVCache, DSStateManager, DSStateManagerConfig,
                                                          RaggedBatchWrapper)
    cfg = DSStateManagerConfig(max_context=8192, max_ragged_batch_size=8192)
    kv = BlockedKVCache(1, 2, 16, 64, torch.float32, torch.device("cpu"), cfg.memory_config, num_blocks=200)
    sm = DSStateManager(cfg, kv)
    b = RaggedBatchWrapper(cfg, torch.device("cpu"), sm.max_blocks_per_seq)
    assert not hasattr(b, "seq_meta")
    b.set_attention_geometry(4, 2, 128)
    steps = [[torch.arange(5, dtype=torch.int32), torch.arange(12)[::3]], [torch.arange(6000) % 100, torch.tensor(7)],
             [torch.arange(8).view(2, 4), torch.tensor([99], dtype=torch.uint8)], []]
    for toks in steps:
        for where in (None, [[0, t.numel() - 1] for t in toks]):
            b.clear()
            for u in range(2):
                sm.flush_sequence(u)
            for i, t in enumerate(toks):
                seq = sm.get_or_create_sequence(i)
                sm.maybe_allocate_kv(seq, t.numel())
                b.insert_sequence(seq, t, logits_at=None if where is None else where[i])
            b.finalize(100)
            flat = [t.reshape(-1).long() for t in toks]
            ends = [sum(t.numel() for t in flat[:i + 1]) for i in range(len(flat))]
            if toks:
                assert torch.equal(b.input_ids, torch.cat(flat)) and b.seq_meta[:, 0].tolist() == [0] + ends[:-1]
                last = [e - 1 for e in ends] if where is None else [e - t.numel() + i for e, t, w in zip(ends, flat, where) for i in w]
                assert b.last_token_idx.tolist() == last and b.atoms.shape[0] == b.n_atoms
                for i in range(len(toks)):
                    blocks = sm.get_sequence(i).kv_blocks
                    assert b.tables_host[i, :len(blocks)].tolist() == blocks and b.tables_host[i, len(blocks):].eq(0).all()
            else:
                assert b.seq_meta.shape == (1, 3) and b.input_ids.numel() == 0 and b.tables_host.shape[0] == 1
    for bad in (-1, 100, 2**40):
        b.clear()
        b.insert_sequence(sm.get_or_create_sequence(0), torch.tensor([3, bad]))
        with pytest.raises(IndexError, match=str(bad)):
            b.finalize(100)


def test_a_step_that_may_replay_makes_no_views():
    """Whether a decode step can replay its graph is known without a view of the step's buffer."""
    import types
    from hcache_deepspeed_amd.inference.v2.model import RaggedTransformer
    from hcache_deepspeed_amd.inference.v2.ragged import (BlockedKVCache, DSStateManager, DSStateManagerConfig,
                                                          RaggedBatchWrapper)
    cfg = DSStateManagerConfig(max_context=256)
    sm = DSStateManager(cfg, BlockedKVCache(1, 2, 16, 64, torch.float32, torch.device("cpu"), cfg.memory_config, num_blocks=8))
    b = RaggedBatchWrapper(cfg, torch.device("cpu"), sm.max_blocks_per_seq)
    model = types.SimpleNamespace(device=torch.device("cuda"), tp=1, decode_graph_max_batch=4, decode_graph_latents=True,
                                  spec=types.SimpleNamespace(moe=None), layers=[])
    assert not RaggedTransformer.decode_graph_eligible(model, b, False)
    for geometry in (False, True):
        b.clear()
        seq = sm.get_or_create_sequence(0)
        sm.maybe_allocate_kv(seq, 1)
        b.insert_sequence(seq, torch.tensor([3]))
        if geometry:
            b.set_attention_geometry(4, 2, 128)
        b.finalize(100)
        assert RaggedTransformer.decode_graph_eligible(model, b, False) == geometry
    assert not set(b.__dict__) & set(b._layout)


def test_staging_buffers_outlive_their_copies():
    """A wrapper that is dropped while its step's copy is queued: the pinned buffers stay until their events have passed."""
    import gc
    import weakref
    from hcache_deepspeed_amd.inference.v2 import ragged

    class Event:
        passed = False

        def query(self):
            return self.passed

        synchronize = record = None  # not to be called here

    def step(events=None):
        b = ragged.RaggedBatchWrapper(ragged.DSStateManagerConfig(), torch.device("cpu"), 4)
        b.finalize()
        if events:
            b.finalize()
            b._slot_events[:] = events
        return [weakref.ref(t) for t in b._slots if t is not None]

    events = [Event(), Event()]
    held = step(events)
    gc.collect()
    assert all(r() is not None for r in held)
    step()
    assert all(r() is not None for r in held)
    events[1].passed = True
    step()
    assert held[0]() is not None and held[1]() is None
    events[0].passed = True
    step()
    gc.collect()
    assert held[0]() is None and not ragged._IN_FLIGHT


def test_only_plain_tensors_pass_autograd_by():
    from hcache_deepspeed_amd.ops import native
    x = torch.ones(2)
    assert not native.plain(x)
    with torch.no_grad():
        assert native.plain(x, None, torch.nn.Parameter(x))
        seen = []
        torch.func.vmap(lambda t: seen.append(native.plain(x)) or t)(x)
        with torch.autograd.forward_ad.dual_level():
            seen.append(native.plain(x))

        class Sub(torch.Tensor):
            pass

        seen.append(native.plain(x.as_subclass(Sub)))
        torch.jit.trace(lambda t: seen.append(native.plain(x)) or t, (x, ), check_trace=False)
        assert seen == [False, False, False, False]


@pytest.mark.gpu
def test_traced_norms_and_gated_units_run_again():
    """A graph recorded without gradients computes them for its own inputs."""
    from hcache_deepspeed_amd.ops.activations import glu
    from hcache_deepspeed_amd.ops.norm import layer_norm, rms_norm
    w = torch.rand(256, device="cuda").bfloat16()
    with torch.no_grad():
        x, y = (torch.randn(64, 256, device="cuda").bfloat16() for _ in range(2))
        for f in (lambda t: rms_norm(t, w), lambda t: rms_norm(t, w, residual=t)[0], lambda t: layer_norm(t, w, w), glu):
            assert torch.equal(torch.jit.trace(f, (x, ), check_trace=False)(y), f(y))


@pytest.mark.gpu
@pytest.mark.parametrize("rows", [1, 5])
def test_traced_few_row_products_run_again(rows):
    """A graph recorded without gradients computes few-row products for its own inputs: they are torch's in it."""
    from hcache_deepspeed_amd.ops.gemv import glu_linear, linear
    w = torch.randn(512, 256, device="cuda").bfloat16()
    with torch.no_grad():
        x, y = (torch.randn(rows, 256, device="cuda").bfloat16() for _ in range(2))
        for f in (lambda t: linear(t, w), lambda t: (lambda z: linear(t, w) if z is None else z)(glu_linear(t, w, None, "silu"))):
            g = torch.jit.trace(f, (x, ), check_trace=False)
            assert torch.equal(g(y), torch.nn.functional.linear(y, w))


@pytest.mark.gpu
def test_graph_after_the_buffer_grew_gpu():
    """A graph reads the batch's device buffer; when a larger step has replaced that, later steps reach the graph's own."""
    from hcache_deepspeed_amd.inference.v2.arch import ArchSpec
    from hcache_deepspeed_amd.inference.v2.engine import InferenceEngineV2, RaggedInferenceEngineConfig
    H, I, V = 256, 512, 211
    g = torch.Generator().manual_seed(0)
    dev = torch.device("cuda")
    mat = lambda *s: (torch.randn(*s, generator=g) * s[-1]**-0.5).bfloat16().to(dev)  # noqa: E731
    one = torch.ones(H, dtype=torch.bfloat16, device=dev)
    layers = [{"ln1.w": one, "ln2.w": one, "qkv.w": mat(4 * 128, H), "o.w": mat(H, 256), "up.w": mat(2 * I, H),
               "down.w": mat(H, I)} for _ in range(2)]
    w = {"embed": mat(V, H) * 16, "final.w": one, "lm_head.w": mat(V, H), "layers": layers}
    spec = ArchSpec("llama", V, H, 2, 2, 1, 128, I, max_position_embeddings=8192)
    conf = RaggedInferenceEngineConfig.from_dict(dict(dtype="bf16", state_manager=dict(max_context=4096,
                                                                                       max_ragged_batch_size=8192)))
    engs = {k: InferenceEngineV2(spec, w, conf, device=dev, num_kv_blocks=200) for k in ("graph", "eager")}
    engs["eager"]._model.decode_graph_max_batch = 0
    draw = lambda n: torch.randint(0, V, (n, ), generator=g)  # noqa: E731
    step = lambda uids, toks: {k: e.put(uids, toks, capture_latents=False)[0] for k, e in engs.items()}  # noqa: E731
    step([1, 2], [draw(40), draw(65)])
    sizes = set()
    for i in range(9):
        if i in (3, 6):  # more tokens than the buffer holds, twice
            step([10 + i], [draw(1500 * i // 3)])
        out = step([1, 2], [draw(1), draw(1)])
        assert torch.equal(out["graph"], out["eager"]), i
        sizes.add(engs["graph"]._batch._dev_meta.numel())
    assert len(sizes) == 3 and engs["graph"]._model._decode_graphs[2, False].graph is not None


@pytest.mark.gpu
def test_graphs_of_several_sizes_share_memory_gpu():
    """Smaller batch sizes' graphs use the memory that the largest one's capture took: beside their logits and what the
    captures themselves round up to, nothing is reserved for them."""
    from hcache_deepspeed_amd.inference.v2.arch import ArchSpec
    from hcache_deepspeed_amd.inference.v2.engine import InferenceEngineV2, RaggedInferenceEngineConfig
    H, I, V = 512, 32768, 211  # activations of 3 MB a step
    g = torch.Generator().manual_seed(0)
    dev = torch.device("cuda")
    mat = lambda *s: (torch.randn(*s, generator=g) * s[-1]**-0.5).bfloat16().to(dev)  # noqa: E731
    one = torch.ones(H, dtype=torch.bfloat16, device=dev)
    layer = {"ln1.w": one, "ln2.w": one, "qkv.w": mat(4 * 128, H), "o.w": mat(H, 256), "up.w": mat(2 * I, H),
             "down.w": mat(H, I)}
    spec = ArchSpec("llama", V, H, 2, 2, 1, 128, I, max_position_embeddings=8192)
    eng = InferenceEngineV2(spec, {"embed": mat(V, H), "final.w": one, "lm_head.w": mat(V, H), "layers": [layer, layer]},
                            RaggedInferenceEngineConfig.from_dict(dict(dtype="bf16")), device=dev, num_kv_blocks=40)
    toks = torch.randint(0, V, (24, 1), generator=g)
    used = {}
    for n in range(24, 16, -1):  # (library products, which take a workspace of their own for each stream)
        for _ in range(3):
            eng.put(list(range(n)), list(toks[:n]), capture_latents=False)
        torch.cuda.synchronize()
        used[n] = torch.cuda.memory_reserved()
    assert all(eng._model._decode_graphs[n, False].graph is not None for n in used)
    assert used[17] - used[24] <= 24 << 20, used


@pytest.mark.gpu
@pytest.mark.parametrize("W", [512, 1024, 2048, 3072, 4096, 5120, 6144, 8192, 648])
@pytest.mark.parametrize("rows", [1, 2, 3, 5, 130])
@pytest.mark.parametrize("is_ln,res,dtype,wdtype", [(False, True, torch.bfloat16, torch.bfloat16),
                                                    (True, True, torch.float32, torch.float32),
                                                    (True, False, torch.bfloat16, torch.float32)])
def test_norm_rows_over_waves_gpu(W, rows, is_ln, res, dtype, wdtype):
    """Rows shared by one, two and four waves, workgroups with a row too many, against 64 bits."""
    from hcache_deepspeed_amd.ops.norm import layer_norm, rms_norm
    g = torch.Generator(device="cuda").manual_seed(W + rows)
    x, r = (torch.randn(rows, W, device="cuda", generator=g).to(dtype) for _ in range(2))
    w, b = (torch.randn(W, device="cuda", generator=g).to(wdtype) for _ in range(2))
    r = r if res else None
    y = layer_norm(x, w, b, 1e-5, r) if is_ln else rms_norm(x, w, 1e-5, r)
    y, h = y if res else (y, x)
    want_h = (x.float() + r.float()).to(dtype) if res else x
    assert torch.equal(h, want_h)
    hd = want_h.double()
    m = hd.mean(-1, keepdim=True) if is_ln else 0.0
    want = (hd - m) * torch.rsqrt(((hd - m)**2).mean(-1, keepdim=True) + 1e-5) * w.double() + (b.double() if is_ln else 0.0)
    # 32-bit sums of W squares, then one rounding of a product and a sum
    last = 2**-8 if dtype == torch.bfloat16 else 2**-22
    mag = want.abs() + (2 * b.double().abs() if is_ln else 0.0)
    assert ((y.double() - want).abs() <= (last + 2**-19) * mag + 1e-6).all()
