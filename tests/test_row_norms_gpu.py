"""Norms of decode rows inside the products around them (ops/gemv.py ``norm_linear``, ``scaled_linear``), against the separate
operations and float64."""
import pytest
import torch

from hcache_deepspeed_amd.ops import gemv, native
from hcache_deepspeed_amd.ops.norm import rms_norm

EPS = 1e-5


def _rows(g, *shape, scale=1.0):
    return (torch.randn(*shape, device="cuda", generator=g) * scale).bfloat16()


@pytest.mark.gpu
@pytest.mark.parametrize("M,K,N,out,act", [
    (2, 128, 128, 24, None), (3, 256, 2048, 3072, None), (8, 1024, 128, 40, "relu"), (9, 5632, 2048, 1000, "gelu_tanh"),
    (13, 512, 4096, 6144, None), (16, 4096, 4096, 14336, "silu"), (16, 256, 4096, 32000, None), (16, 256, 8320, 512, "silu"),
    (5, 256, 9216, 264, None)])
def test_norm_between_products(cuda, M, K, N, out, act):
    """One row block and the last row of it, widths of one and several parts a thread (and beyond four of them), the skinny
    kernel with four and eight waves and the tiled one (16 rows of large weights), gated units of odd halves."""
    g = torch.Generator(device="cuda").manual_seed(M * N + out)
    x, w = _rows(g, M, K), _rows(g, N, K, scale=K**-0.5)
    res, gamma = _rows(g, M, N), (1 + 0.1 * torch.randn(N, device="cuda", generator=g)).bfloat16()
    w2 = _rows(g, out * (1 if act is None else 2), N, scale=N**-0.5)
    with torch.no_grad():
        assert gemv.scaled_rows_ok(M) and gemv.scaled_weight_ok(w, True) and gemv.scaled_weight_ok(w2)
        rows, r = gemv.norm_linear(x, w, res, gamma, EPS)
        y = gemv.scaled_linear(rows, w2, act)
        _, want_r = rms_norm(gemv.skinny(x, w), gamma, EPS, res)
        assert torch.equal(r, want_r)  # the same sums, rounded at the same places
        d = r.double()
        assert torch.equal(rows.x, (r.float() * gamma.float()).bfloat16())
        ssq = rows.ssq.double().sum(0)[:M]
        assert ((ssq - d.square().sum(1)).abs() <= N * 2**-24 * d.square().sum(1)).all()
        z = rows.x.double() * torch.rsqrt(d.square().mean(1, keepdim=True) + EPS) @ w2.double().T
        if act is not None:
            h, u = z.chunk(2, 1)
            f = {"silu": torch.nn.functional.silu, "relu": torch.relu, "gelu_tanh": lambda t: torch.nn.functional.gelu(t, approximate="tanh")}[act]
            z = f(h) * u
        # the result is rounded to bf16 (2^-9 each, a gated unit's two inputs as well)
        assert (y.double() - z).norm() <= (2 if act else 1) * 2**-8 * z.norm()
        assert torch.equal(y, gemv.scaled_linear(rows, w2, act))


@pytest.mark.gpu
@pytest.mark.parametrize("fmt", ["fp6", "int8", "int4"])
@pytest.mark.parametrize("M,K,N,out,act", [(2, 256, 2048, 3072, None), (8, 4096, 4096, 6144, None), (3, 5632, 2048, 8192, "silu"),
                                           (8, 128, 4096, 8192, "relu"), (16, 8192, 4096, 4096, "gelu_tanh"), (13, 2048, 1024, 1536, None)])
def test_norm_between_packed_products(cuda, fmt, M, K, N, out, act):
    """The same on packed weights, through each of the stream's kernels: whole lines, resident rows, one and two tiles."""
    from hcache_deepspeed_amd.ops import quantizer as q
    g = torch.Generator(device="cuda").manual_seed(M * N + out)
    res, gamma = _rows(g, M, N), (1 + 0.1 * torch.randn(N, device="cuda", generator=g)).bfloat16()
    x, w, w2 = _rows(g, M, K), _rows(g, N, K, scale=K**-0.5), _rows(g, out * (1 if act is None else 2), N, scale=N**-0.5)

    def pack(w):
        return q.quantize_minifloat(w, 128, 6, 2)[:2] if fmt == "fp6" else q.quantize(w, 128, int(fmt[3:]), True)[:2]
    with torch.no_grad():
        a, b = pack(w), pack(w2)
        rows, r = q.packed_norm_linear(x, *a, N, K, 128, fmt, res, gamma, EPS)
        y = q.packed_scaled_linear(rows, *b, out, N, 128, fmt, act)
        plain = torch.empty(M, N, device="cuda", dtype=torch.bfloat16)
        native.check(native.kernels().hds_wmix_skinny(x.data_ptr(), a[0].data_ptr(), a[1].data_ptr(), None, plain.data_ptr(), M, N, K,
                                                      128, q._FMTS[fmt], 3, 0, native.stream()), "wmix_skinny")
        _, want_r = rms_norm(plain, gamma, EPS, res)
        assert torch.equal(r, want_r) and torch.equal(rows.x, (r.float() * gamma.float()).bfloat16())
        # the same weights against rows that are normed beforehand: both round the rows, the sums' factor and the result once
        xn = (rows.x.double() * torch.rsqrt(r.double().square().mean(1, keepdim=True) + EPS))
        stored = q.dequantize_minifloat(*b, 128, 6, 2, torch.float32) if fmt == "fp6" else q.dequantize(*b, None, 128, int(fmt[3:]), True, torch.float32)
        z = xn @ stored.double().view(w2.shape).T
        if act is not None:
            h, u = z.chunk(2, 1)
            f = {"silu": torch.nn.functional.silu, "relu": torch.relu, "gelu_tanh": lambda t: torch.nn.functional.gelu(t, approximate="tanh")}[act]
            z = f(h) * u
        assert (y.double() - z).norm() <= (2 if act else 1) * 2**-8 * z.norm()


@pytest.mark.gpu
@pytest.mark.parametrize("fmt", ["fp6", "int8", "int4"])
@pytest.mark.parametrize("M,K,N", [(9, 2048, 16384), (12, 2048, 16400), (16, 512, 16400), (16, 8320, 16400), (5, 4096, 16400), (16, 2048, 32784)])
def test_norm_behind_packed_products_of_many_columns(cuda, fmt, M, K, N):
    """Two tiles a workgroup, the last of them with one, whole lines and resident rows: every column once, nothing behind."""
    from hcache_deepspeed_amd.ops import quantizer as q
    g = torch.Generator(device="cuda").manual_seed(M * N)
    res, gamma = _rows(g, M, N), (1 + 0.1 * torch.randn(N, device="cuda", generator=g)).bfloat16()
    x, w = _rows(g, M, K), _rows(g, N, K, scale=K**-0.5)
    packed, scales = q.quantize_minifloat(w, 128, 6, 2)[:2] if fmt == "fp6" else q.quantize(w, 128, int(fmt[3:]), True)[:2]
    y, r = (torch.full((M + 1, N), 7.0, device="cuda", dtype=torch.bfloat16) for _ in range(2))
    ssq = torch.full((N // 16 + 4, 16), 7.0, device="cuda")
    plain = torch.empty(M, N, device="cuda", dtype=torch.bfloat16)
    lib, end = native.kernels(), (K, 128, q._FMTS[fmt], 3, 0, native.stream())
    native.check(lib.hds_wmix_norm(x.data_ptr(), packed.data_ptr(), scales.data_ptr(), y.data_ptr(), None, 0.0, res.data_ptr(),
                                   gamma.data_ptr(), r.data_ptr(), ssq.data_ptr(), M, N, *end), "wmix_norm")
    native.check(lib.hds_wmix_skinny(x.data_ptr(), packed.data_ptr(), scales.data_ptr(), None, plain.data_ptr(), M, N, *end), "wmix_skinny")
    _, want = rms_norm(plain, gamma, EPS, res)
    assert torch.equal(r[:M], want) and torch.equal(y[:M], (want.float() * gamma.float()).bfloat16())
    parts = want.double().square().view(M, N // 16, 16).sum(-1).T
    assert ((ssq[:N // 16, :M].double() - parts).abs() <= 16 * 2**-24 * parts).all()
    assert (y[M] == 7).all() and (r[M] == 7).all() and (ssq[N // 16:] == 7).all()


@pytest.mark.gpu
def test_norm_rows_out_of_range(cuda):
    """Rows with an infinity or a NaN become NaN, as a norm's do; others beside them do not; an all-zero row stays zero."""
    g = torch.Generator(device="cuda").manual_seed(1)
    x, w, w2 = _rows(g, 4, 256), _rows(g, 512, 256, scale=1 / 16), _rows(g, 48, 512, scale=0.05)
    res, gamma = _rows(g, 4, 512), torch.ones(512, device="cuda", dtype=torch.bfloat16)
    res[1, 3], res[2, 5], x[3], res[3] = float("inf"), float("nan"), 0, 0
    with torch.no_grad():
        rows, r = gemv.norm_linear(x, w, res, gamma, EPS)
        y = gemv.scaled_linear(rows, w2)
    assert torch.isfinite(y[0]).all() and y[1].isnan().all() and y[2].isnan().all() and not y[3].any()


@pytest.mark.gpu
def test_scaled_steps_are_asked_for(cuda, monkeypatch):
    """Where nothing may watch the separate operations, and where the switches leave the rows to the skinny kernel."""
    with torch.no_grad():
        assert [gemv.scaled_rows_ok(m) for m in (1, 2, 16, 17)] == [False, True, True, False]
        with torch.autocast("cuda"):
            assert not gemv.scaled_rows_ok(4)
        monkeypatch.setattr(gemv, "SKINNY", False)
        assert not gemv.scaled_rows_ok(4)
    assert not gemv.scaled_rows_ok(4)
    w = torch.zeros(32, 256, device="cuda", dtype=torch.bfloat16)
    assert gemv.scaled_weight_ok(w, True) and not gemv.scaled_weight_ok(w[:, :192]) and not gemv.scaled_weight_ok(w.float())
    assert not gemv.scaled_weight_ok(w[:24], True) and gemv.scaled_weight_ok(w[:24]) and not gemv.scaled_weight_ok(w.t())


@pytest.mark.gpu
@pytest.mark.parametrize("seqs,vocab,quant", [(2, 512, ""), (7, 500, ""), (16, 512, ""), (5, 512, "wf6af16"), (3, 512, "int8"), (4, 512, "int4")])
def test_decode_steps_without_norm_launches(cuda, monkeypatch, seqs, vocab, quant):
    """Decode steps, first eager, then replayed, give the same logits as with the norms' own launches, to bf16 through the
    layers (0.3 to 0.7 % from 64 bits either)."""
    from hcache_deepspeed_amd.inference.v2 import model as v2
    from hcache_deepspeed_amd.inference.v2.arch import ArchSpec
    from hcache_deepspeed_amd.inference.v2.engine import InferenceEngineV2, RaggedInferenceEngineConfig
    W, ff, nq, nkv = 256, 384, 2, 1
    g = torch.Generator(device="cuda").manual_seed(seqs)
    layers = [{"ln1.w": 1 + _rows(g, W, scale=0.1), "ln2.w": 1 + _rows(g, W, scale=0.1), "qkv.w": _rows(g, (nq + 2 * nkv) * 128, W, scale=1 / 16),
               "o.w": _rows(g, W, nq * 128, scale=1 / 16), "up.w": _rows(g, 2 * ff, W, scale=1 / 16), "down.w": _rows(g, W, ff, scale=0.05)}
              for _ in range(3)]
    sd = {"embed": _rows(g, vocab, W), "final.w": 1 + _rows(g, W, scale=0.1), "lm_head.w": _rows(g, vocab, W, scale=1 / 16), "layers": layers}
    spec = ArchSpec("llama", vocab, W, 3, nq, nkv, 128, ff, norm_eps=EPS, rope_theta=10000.0, max_position_embeddings=512)
    conf = RaggedInferenceEngineConfig.from_dict(dict(dtype="bf16", quantization={"quantization_mode": quant} if quant else {}, state_manager=dict(
        max_context=256, max_ragged_batch_size=1024, max_tracked_sequences=16, kv_block_size=64)))
    calls, sides = [], []
    from hcache_deepspeed_amd.inference.v2.modules import implementations as m
    name = "packed_norm_linear" if quant else "norm_linear"
    plain = getattr(m, name)
    monkeypatch.setattr(m, name, lambda *a: calls.append(1) or plain(*a))
    for on in (True, False):
        if not on:
            monkeypatch.setattr(v2, "scaled_rows_ok", lambda m: False)
        eng = InferenceEngineV2(spec, sd, conf, device=torch.device("cuda", 0), num_kv_blocks=4 * seqs)
        uids = list(range(seqs))
        gen = torch.Generator().manual_seed(3)
        out = [eng.put(uids, [torch.randint(0, vocab, (5 + 3 * u, ), generator=gen) for u in uids], capture_latents=False)[0].clone()]
        for _ in range(4):
            out.append(eng.put(uids, [torch.randint(0, vocab, (1, ), generator=gen) for u in uids], capture_latents=False)[0].clone())
        sides.append(out)
        assert bool(calls) == on
        calls.clear()
    assert torch.equal(sides[0][0], sides[1][0])
    for a, b in zip(*(s[1:] for s in sides)):
        assert (a.double() - b.double()).norm() <= 0.02 * b.double().norm()


def _small_engine(g, layers=2):
    from hcache_deepspeed_amd.inference.v2.arch import ArchSpec
    from hcache_deepspeed_amd.inference.v2.engine import InferenceEngineV2, RaggedInferenceEngineConfig
    W, ff, nq, nkv, vocab = 256, 384, 2, 1, 512
    sd = {"embed": _rows(g, vocab, W), "final.w": 1 + _rows(g, W, scale=0.1), "lm_head.w": _rows(g, vocab, W, scale=1 / 16), "layers": [
        {"ln1.w": 1 + _rows(g, W, scale=0.1), "ln2.w": 1 + _rows(g, W, scale=0.1), "qkv.w": _rows(g, (nq + 2 * nkv) * 128, W, scale=1 / 16),
         "o.w": _rows(g, W, nq * 128, scale=1 / 16), "up.w": _rows(g, 2 * ff, W, scale=1 / 16), "down.w": _rows(g, W, ff, scale=0.05)}
        for _ in range(layers)]}
    spec = ArchSpec("llama", vocab, W, layers, nq, nkv, 128, ff, norm_eps=EPS, rope_theta=10000.0, max_position_embeddings=512)
    conf = RaggedInferenceEngineConfig.from_dict(dict(dtype="bf16", state_manager=dict(
        max_context=256, max_ragged_batch_size=1024, max_tracked_sequences=16, kv_block_size=64)))
    return InferenceEngineV2(spec, sd, conf, device=torch.device("cuda", 0), num_kv_blocks=32)


def _steps(eng, seqs, first=0, steps=3):
    """Logits of a prompt each and some decode steps: launched, captured and replayed ones."""
    gen = torch.Generator().manual_seed(3)
    uids = list(range(first, first + seqs))
    out = [eng.put(uids, [torch.randint(0, 512, (5 + 3 * u, ), generator=gen) for u in range(seqs)], capture_latents=False)[0].clone()]
    for _ in range(steps):
        out.append(eng.put(uids, [torch.randint(0, 512, (1, ), generator=gen) for _ in uids], capture_latents=False)[0].clone())
    return torch.stack(out)


@pytest.mark.gpu
@pytest.mark.parametrize("what", ["_mlp", "_attn", "_norm", "_allreduce", "own", "attention", "norm", "head"])
def test_decode_steps_of_models_of_their_own(cuda, monkeypatch, what):
    """What a derived model, an object or a registered attention has in the place of a stock part is what decode steps compute."""
    from hcache_deepspeed_amd.inference.v2 import model as v2
    from hcache_deepspeed_amd.inference.v2.modules.implementations import DSDenseBlockedAttention
    sides = []
    for off in (False, True):
        if off:
            monkeypatch.setattr(v2, "scaled_rows_ok", lambda m: False)
        eng = _small_engine(torch.Generator(device="cuda").manual_seed(5))
        m = eng._model
        if what == "attention":
            class Spread(DSDenseBlockedAttention):  # rows that are no plain matrix
                def forward(self, *a):
                    return torch.cat([super().forward(*a)] * 2, 1)[:, ::2].mul(2)
            m.attn_mod = Spread(m.attn_mod._config)
        elif what == "own":
            plain = m._mlp
            m._mlp = lambda L, x: plain(L, x) * 2
        elif what in ("norm", "head"):  # an object's own
            mod = m.norm_mod if what == "norm" else m.unembed_mod
            plain = mod.forward
            mod.forward = (lambda *a: tuple(t * 2 for t in plain(*a))) if what == "norm" else (lambda *a: plain(*a) + 1)
        else:
            def double(self, *a, **kw):
                y = getattr(v2.RaggedTransformer, what)(self, *a, **kw)
                return (y[0] * 2, y[1]) if isinstance(y, tuple) else y * 2
            m.__class__ = type("Own", (v2.RaggedTransformer, ), {what: double})
        sides.append(_steps(eng, 3))
    assert torch.equal(*sides)


@pytest.mark.gpu
@pytest.mark.parametrize("key", ["qkv.w", "o.w", "up.w", "down.w", "ln2.w"])
def test_decode_steps_after_an_exchange_of_weights(cuda, key):
    """Weights of another layout or alignment that come in the place of others, for a batch size that has decoded before too: the
    same values, the same logits to the rounding of bf16 layers."""
    eng = _small_engine(torch.Generator(device="cuda").manual_seed(5))
    eng._model.decode_graph_max_batch = 0  # (a graph keeps the weights that it was captured with)
    want = _steps(eng, 3)
    for u in range(3):
        eng.flush(u)
    for L in eng._model.layers:
        w = L.w[key]
        if w.dim() == 2:
            L.w[key] = w.t().contiguous().t()
        else:  # two bytes from where rows of 16 begin
            L.w[key] = torch.cat([w[:1], w])[1:]
    got = _steps(eng, 3)
    assert (got.double() - want.double()).norm() <= 0.02 * want.double().norm()
