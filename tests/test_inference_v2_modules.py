"""Inference-v2 module registry + heuristics (reference inference/v2/modules, tests/unit/inference/v2/modules
strategy: each implementation against a torch reference; quantized linears within their format's error)."""
import pytest
import torch

from hcache_deepspeed_amd.inference.v2 import build_engine_from_model
from hcache_deepspeed_amd.inference.v2.modules import (DSLinearBase, DSLinearConfig, DSLinearRegistry, DSMoEConfig,
                                                       DSNormConfig, ConfigBundle, instantiate_linear,
                                                       instantiate_moe, instantiate_pre_norm)
from hcache_deepspeed_amd.models.llama import LlamaForCausalLM, tiny


def test_registry_selection_and_errors():
    assert type(instantiate_linear(DSLinearConfig(64, 32))).__name__ == "BlasFPLinear"
    q = instantiate_linear(DSLinearConfig(64, 32), type("EC", (), {"quantization": {"quantization_mode": "wf6af16"}}))
    assert q.name() == "quantized_wf6af16_linear"
    assert instantiate_linear(DSLinearConfig(64, 32, quantization_mode="int4")).name() == "quantized_int_linear"
    # shapes the packed kernels cannot take fall back to bf16
    assert instantiate_linear(DSLinearConfig(40, 32, quantization_mode="int8")).name() == "blas_fp_linear"
    with pytest.raises(ValueError):
        instantiate_linear(DSLinearConfig(64, 32, quantization_mode="nf4"))
    with pytest.raises(KeyError):
        DSLinearRegistry.instantiate_config(ConfigBundle("nope", DSLinearConfig(8, 8)))
    with pytest.raises(TypeError):
        DSLinearRegistry.register_module(int)
    assert "blas_fp_linear" in DSLinearRegistry.supporting(DSLinearConfig(64, 64))

    @DSLinearRegistry.register_module
    class _Custom(DSLinearBase):

        @staticmethod
        def name():
            return "custom_test_linear"

        def forward(self, x, w, b=None):
            return x @ w.t() * 2

    m = DSLinearRegistry.instantiate_config(ConfigBundle("custom_test_linear", DSLinearConfig(4, 4)))
    assert torch.equal(m(torch.ones(1, 4), torch.eye(4)), 2 * torch.ones(1, 4))
    del DSLinearRegistry.registry["custom_test_linear"]


@pytest.mark.parametrize("act", ["identity", "gelu", "relu", "silu_glu"])
@pytest.mark.parametrize("mode,tol", [(None, 1e-5), ("wf6af16", 0.08), ("int8", 0.02), ("int4", 0.2)])
def test_linear_implementations(act, mode, tol):
    torch.manual_seed(0)
    out = 96 if act.endswith("_glu") else 48
    x, w, b = torch.randn(5, 64), torch.randn(out, 64) * 0.2, torch.randn(out) * 0.1
    lin = instantiate_linear(DSLinearConfig(64, out, activation=act, quantization_mode=mode, group_size=32))
    y = lin(x, lin.transform_param(w), b)
    ref = x @ w.t() + b
    if act == "silu_glu":
        g, u = ref.chunk(2, -1)
        ref = torch.nn.functional.silu(g) * u
    elif act != "identity":
        ref = getattr(torch.nn.functional, act)(ref)
    err = (y.float() - ref).norm() / ref.norm()
    assert err < tol, (mode, act, float(err))


@pytest.mark.gpu
@pytest.mark.parametrize("rows", [1, 8, 16])
@pytest.mark.parametrize("leaf", ["rows", "weight"])
def test_few_rows_keep_their_gradient_gpu(rows, leaf):
    """Logits, a projection and a gated one of as few rows as run on kernels without a backward, with gradients wanted of
    the rows or of the weight alone."""
    from hcache_deepspeed_amd.inference.v2.modules import DSUnembedConfig, instantiate_unembed
    torch.manual_seed(rows)
    x, w = (torch.randn(n, 256, device="cuda", dtype=torch.bfloat16) * 256**-0.25 for n in (rows, 64))
    t = (x if leaf == "rows" else w).requires_grad_()
    unembed = instantiate_unembed(DSUnembedConfig(model_dim=256, vocab_size=64))
    lin, glu = (instantiate_linear(DSLinearConfig(256, 64, activation=a)) for a in ("identity", "silu_glu"))
    gate, up = torch.nn.functional.linear(x.float(), w.float()).chunk(2, -1)
    full = torch.cat([gate, up], -1)
    for got, ref in ((unembed.project(x, w), full), (lin(x, w), full),
                     (glu(x, w), torch.nn.functional.silu(gate) * up)):
        assert got.requires_grad
        do = torch.randn_like(ref)
        a, b = torch.autograd.grad(got, t, do.bfloat16())[0], torch.autograd.grad(ref, t, do, retain_graph=True)[0]
        assert (a.float() - b).norm() <= 3 * 2**-8 * b.norm()
        with torch.no_grad():
            assert (got - (lin(x, w) if ref is full else glu(x, w))).norm() <= 2**-7 * ref.norm()


def test_pre_norm_and_moe_modules():
    torch.manual_seed(0)
    n = instantiate_pre_norm(DSNormConfig(32, "rms", 1e-6))
    r, h, g = torch.randn(4, 32), torch.randn(4, 32), torch.rand(32) + 0.5
    r2, y = n(r, h, g)
    s = r + h
    assert torch.allclose(r2, s) and torch.allclose(y, s * torch.rsqrt(s.pow(2).mean(-1, keepdim=True) + 1e-6) * g,
                                                    atol=1e-5)
    moe = instantiate_moe(DSMoEConfig(32, 16, 4, 2, "silu_glu", True))
    x = torch.randn(6, 32)
    rw, w13, w2 = torch.randn(4, 32), torch.randn(4, 32, 32) * 0.2, torch.randn(4, 32, 16) * 0.2
    y = moe(x, rw, w13, w2)
    p = torch.softmax(x @ rw.t(), -1)
    tw, ti = p.topk(2, -1)
    tw = tw / tw.sum(-1, keepdim=True)
    ref = torch.zeros_like(x)
    for t in range(6):
        for j in range(2):
            e = int(ti[t, j])
            gu = w13[e] @ x[t]
            ref[t] += tw[t, j] * (w2[e] @ (torch.nn.functional.silu(gu[:16]) * gu[16:]))
    assert torch.allclose(y, ref, atol=1e-4), (y - ref).abs().max()


@pytest.mark.parametrize("mode,tol", [("wf6af16", 0.15), ("int8", 0.05)])
def test_quantized_engine_matches_bf16(mode, tol, tmp_path):
    from hcache_deepspeed_amd.inference.v2.engine import build_engine_from_ds_checkpoint
    torch.manual_seed(0)
    m = LlamaForCausalLM(tiny(head_dim=64, hidden_size=128, intermediate_size=256, vocab_size=101,
                              num_attention_heads=2, num_key_value_heads=1, num_hidden_layers=2)).eval()
    base = dict(dtype="fp32", state_manager={"max_context": 256, "kv_block_size": 64})
    ids = torch.randint(0, 101, (20, ), generator=torch.Generator().manual_seed(2))
    ref, _ = build_engine_from_model(m, base, device=torch.device("cpu"), num_kv_blocks=8).put([1], [ids])
    eng = build_engine_from_model(m, {**base, "quantization": {"quantization_mode": mode}},
                                  device=torch.device("cpu"), num_kv_blocks=8)
    from hcache_deepspeed_amd.inference.v2.modules.implementations import _PackedWeight
    assert isinstance(eng._model.layers[0].w["qkv.w"], _PackedWeight)
    got, _ = eng.put([1], [ids])
    err = (got - ref).norm() / ref.norm()
    assert err < tol, float(err)
    # serialize / reload keeps the packed weights
    eng.serialize(str(tmp_path))
    eng2 = build_engine_from_ds_checkpoint(str(tmp_path), {**base, "quantization": {"quantization_mode": mode}},
                                           device=torch.device("cpu"), num_kv_blocks=8)
    got2, _ = eng2.put([1], [ids])
    assert torch.equal(got, got2)


@pytest.mark.gpu
@pytest.mark.parametrize("mode,tol", [(None, 0.03), ("wf6af16", 0.15), ("int8", 0.06)])
def test_quantized_engine_gpu(mode, tol):
    """bf16 engine on the MI355X: decode steps run the FP6 / INT8 HIP GEMVs, prefill the dequant + GEMM path."""
    torch.manual_seed(0)
    m = LlamaForCausalLM(tiny(head_dim=128, hidden_size=256, intermediate_size=512, vocab_size=211,
                              num_attention_heads=2, num_key_value_heads=1, num_hidden_layers=2)).eval()
    dev = torch.device("cuda")
    ids = torch.randint(0, 211, (40, ), generator=torch.Generator().manual_seed(2))
    with torch.no_grad():
        full = m(torch.cat([ids, ids[:3]])[None]).float()
    cfg = dict(dtype="bf16", state_manager={"max_context": 256, "kv_block_size": 64})
    if mode:
        cfg["quantization"] = {"quantization_mode": mode}
    eng = build_engine_from_model(m, cfg, device=dev, num_kv_blocks=8)
    lg, _ = eng.put([1], [ids])
    outs = [lg[0].float().cpu()]
    for j in range(3):
        lg, _ = eng.put([1], [ids[j:j + 1]], capture_latents=False)
        outs.append(lg[0].float().cpu())
    want = full[[39, 40, 41, 42]]
    err = (torch.stack(outs) - want).norm() / want.norm()
    assert err < tol, float(err)


def _moe_reference(x, rw, w13, w2, top, normalize, shared=None):
    """In float64; the choices and weights too."""
    x, rw, w13, w2 = (t.double() for t in (x, rw, w13, w2))
    p = torch.softmax(x @ rw.t(), -1)
    weight, chosen = p.topk(top, -1)
    if normalize:
        weight = weight / weight.sum(-1, keepdim=True)
    out = torch.zeros_like(x)
    for e in range(rw.shape[0]):
        t, j = (chosen == e).nonzero(as_tuple=True)
        g, u = (x[t] @ w13[e].t()).chunk(2, -1)
        out.index_add_(0, t, weight[t, j, None] * ((torch.nn.functional.silu(g) * u) @ w2[e].t()))
    if shared is not None:
        s13, s2, gate = (t.double() for t in shared)
        g, u = (x @ s13.t()).chunk(2, -1)
        out += torch.sigmoid(x @ gate.t()) * ((torch.nn.functional.silu(g) * u) @ s2.t())
    return out, weight, chosen


@pytest.mark.gpu
@pytest.mark.parametrize("T,E,top,normalize,has_shared", [
    (1, 8, 2, True, False), (16, 64, 6, False, True), (64, 8, 2, True, True), (64, 200, 33, True, False),
    (65, 8, 1, True, False), (300, 64, 4, False, True), (700, 130, 3, True, False)])
def test_routed_moe_module_gpu(T, E, top, normalize, has_shared):
    """Both sides of the line between the products straight from the choices (64 tokens, 2,048 choices) and the sorted
    ones; one, two and four router entries a lane. Inputs are integers / 4, so that router logits are exact and
    no choice depends on rounding; what is left is bf16: the hidden rows, the experts' outputs and the result, each 2^-9."""
    H, I, S = 256, 128, 384
    g = torch.Generator().manual_seed(T)
    dev = torch.device("cuda")
    x = (torch.randint(-8, 9, (T, H), generator=g) / 4).bfloat16().to(dev)
    rw = (torch.randint(-8, 9, (E, H), generator=g) / 64).bfloat16().to(dev)
    mat = lambda *s: (torch.randn(*s, generator=g) * s[-1]**-0.5).bfloat16().to(dev)  # noqa: E731
    w13, w2 = mat(E, 2 * I, H), mat(E, H, I)
    shared = (mat(2 * S, H), mat(H, S), mat(1, H)) if has_shared else None
    moe = instantiate_moe(DSMoEConfig(H, I, E, top, "silu_glu", normalize))
    laid = moe.lay_out(rw, w13, w2, shared)
    assert laid is not None
    y = moe(x, rw, w13, w2, laid)
    want, weight, _ = _moe_reference(x, rw, w13, w2, top, normalize and top > 1, shared)
    assert (y.double() - want).norm() / want.norm() < 3 * 2**-8
    if not has_shared:
        assert torch.equal(y, moe(x, rw, w13, w2))  # laid out on the way
    from hcache_deepspeed_amd.ops.experts import RouterShape, route
    z = x.float() @ rw.float().t()
    expert, got = route(z, None, RouterShape(E, top=top, normalize=normalize and top > 1))
    # 32-bit exponentials and one division
    assert torch.allclose(got.double(), weight, rtol=1e-5, atol=1e-9)
    assert torch.equal(z.gather(1, expert.long()), z.topk(top, -1).values)


@pytest.mark.gpu
@pytest.mark.parametrize("T", [5, 130])
@pytest.mark.parametrize("how", ["columns first", "odd row stride", "shifted rows", "shifted weights"])
def test_routed_moe_module_takes_any_layout_gpu(T, how):
    """Rows that are no whole 16-byte pieces in order give what a copy in order gives; weights that are not aligned are not
    laid out."""
    H, I, E = 256, 128, 8
    g = torch.Generator(device="cuda").manual_seed(T)
    mat = lambda *s: (torch.randn(*s, generator=g, device="cuda") * s[-1]**-0.5).bfloat16()  # noqa: E731
    x, rw, w13, w2 = mat(T, H) * 16, mat(E, H) * 4, mat(E, 2 * I, H), mat(E, H, I)
    moe = instantiate_moe(DSMoEConfig(H, I, E, 2, "silu_glu", True))
    want = moe(x, rw, w13, w2)
    shifted = lambda t: torch.cat([t.new_zeros(1), t.reshape(-1)])[1:].view(t.shape)  # noqa: E731
    if how == "shifted weights":
        assert moe.lay_out(rw, shifted(w13), w2) is None and moe.lay_out(shifted(rw), w13, w2) is None
        return
    if how == "columns first":
        v = x.t().contiguous().t()
    else:
        v = shifted(x) if how == "shifted rows" else torch.cat([x, x[:, :5]], 1)[:, :H]
    assert torch.equal(v, x) and torch.equal(moe(v, rw, w13, w2), want)


def test_route_normalizes():
    from hcache_deepspeed_amd.ops.experts import RouterShape, route
    z = torch.randn(5, 12, generator=torch.Generator().manual_seed(0))
    _, w = route(z, None, RouterShape(12, top=3, normalize=True, scale=2.0))
    p = torch.softmax(z, -1).topk(3, -1).values
    assert torch.allclose(w, 2.0 * p / p.sum(-1, keepdim=True))


@pytest.mark.gpu
@pytest.mark.parametrize("shared,normalize", [(True, False), (False, True)])
def test_moe_decode_graph_matches_eager_gpu(shared, normalize):
    """A batch size's first step runs eagerly over the graph's buffers, the second captures, later ones replay: each gives
    the logits of an engine without graphs, bit for bit (the same kernels)."""
    from hcache_deepspeed_amd.inference.v2.arch import ArchSpec
    from hcache_deepspeed_amd.inference.v2.engine import InferenceEngineV2, RaggedInferenceEngineConfig
    H, E, I, S, V = 256, 8, 128, 384, 211
    g = torch.Generator().manual_seed(0)
    dev = torch.device("cuda")
    mat = lambda *s: (torch.randn(*s, generator=g) * s[-1]**-0.5).bfloat16().to(dev)  # noqa: E731
    one = torch.ones(H, dtype=torch.bfloat16, device=dev)
    layers = []
    for _ in range(2):
        L = {"ln1.w": one, "ln2.w": one, "qkv.w": mat(4 * 128, H), "o.w": mat(H, 256), "router.w": mat(E, H),
             "w13": mat(E, 2 * I, H), "w2": mat(E, H, I)}
        if shared:
            L.update({"shared.w13": mat(2 * S, H), "shared.w2": mat(H, S), "shared_gate.w": mat(1, H)})
        layers.append(L)
    w = {"embed": mat(V, H) * 16, "final.w": one, "lm_head.w": mat(V, H), "layers": layers}
    spec = ArchSpec("qwen2_moe", V, H, 2, 2, 1, 128, I, max_position_embeddings=512,
                    moe=dict(num_experts=E, top_k=2, normalize=normalize, shared=shared))
    conf = RaggedInferenceEngineConfig.from_dict(dict(dtype="bf16", state_manager=dict(max_context=512)))
    engs = {k: InferenceEngineV2(spec, w, conf, device=dev, num_kv_blocks=32) for k in ("graph", "eager")}
    engs["eager"]._model.decode_graph_max_batch = 0
    prompts = [torch.randint(0, V, (n, ), generator=g) for n in (40, 65, 7)]
    for e in engs.values():
        e.put([1, 2, 3], prompts, capture_latents=False)
    for step in range(8):
        uids = [1, 2, 3] if step % 2 else [1, 3]
        toks = [torch.randint(0, V, (1, ), generator=g) for _ in uids]
        out = {k: e.put(uids, toks, capture_latents=False)[0] for k, e in engs.items()}
        assert torch.equal(out["graph"], out["eager"]), step
    assert set(engs["graph"]._model._decode_graphs) == {(2, False), (3, False)}
    assert all(x.graph is not None for x in engs["graph"]._model._decode_graphs.values())
