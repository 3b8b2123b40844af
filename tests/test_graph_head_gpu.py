"""Logits of replayed decode steps: in memory of their own, the same as launch by launch."""
import pytest
import torch


@pytest.mark.gpu
@pytest.mark.parametrize("rows", [1, 2, 16, 17])  # norms in the one-row products, between the products, as kernels
@pytest.mark.parametrize("routed", [False, True])
def test_logits_of_earlier_steps_stay(rows, routed):
    from hcache_deepspeed_amd.inference.v2.arch import ArchSpec
    from hcache_deepspeed_amd.inference.v2.engine import InferenceEngineV2, RaggedInferenceEngineConfig
    H, I, V = 256, 512, 211
    g = torch.Generator().manual_seed(rows)
    dev = torch.device("cuda")
    mat = lambda *s: (torch.randn(*s, generator=g) * s[-1]**-0.5).bfloat16().to(dev)  # noqa: E731
    one = torch.ones(H, dtype=torch.bfloat16, device=dev)
    layers = []
    for _ in range(2):
        L = {"ln1.w": one, "ln2.w": one, "qkv.w": mat(4 * 128, H), "o.w": mat(H, 256)}
        L.update({"router.w": mat(4, H), "w13": mat(4, 2 * I, H), "w2": mat(4, H, I)} if routed else
                 {"up.w": mat(2 * I, H), "down.w": mat(H, I)})
        layers.append(L)
    spec = ArchSpec("llama", V, H, 2, 2, 1, 128, I, max_position_embeddings=1024)
    if routed:
        spec.model_type = "mixtral"
        spec.moe = dict(num_experts=4, top_k=2, normalize=True, shared=False, shared_intermediate_size=0)
    w = {"embed": mat(V, H) * 16, "final.w": one, "lm_head.w": mat(V, H), "layers": layers}
    conf = RaggedInferenceEngineConfig.from_dict(dict(dtype="bf16", state_manager=dict(max_context=1024)))
    engs = {k: InferenceEngineV2(spec, w, conf, device=dev, num_kv_blocks=40) for k in ("graph", "eager")}
    engs["eager"]._model.decode_graph_max_batch = 0
    got = {k: [] for k in engs}
    for _ in range(5):
        toks = list(torch.randint(0, V, (rows, 1), generator=g))
        for k, e in engs.items():
            got[k].append(e.put(list(range(rows)), toks, capture_latents=False)[0])
        torch.cuda.synchronize()
    assert engs["graph"]._model._decode_graphs[rows, False].graph is not None
    assert len({t.data_ptr() for t in got["graph"]}) == 5
    for a, b in zip(got["graph"], got["eager"]):
        assert torch.equal(a, b)
