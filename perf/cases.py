"""Performance cases: what programs on this framework spend their time in, with the same work in plain torch and 64 bits.

Three kinds of work, each through the call that a program makes:

* ``serve``: the ragged serving engine (``InferenceEngineV2.put`` / ``flush``). Some sequences decode one token a step over
  their cached context, some prompts arrive, whole or in pieces that ride along with the decoding ones. Dense and routed
  layouts, bf16 or weight-only quantized weights, with or without the latents that HCache keeps on the host.
* ``train``: a whole step of the ZeRO-3 engine (forward, backward, clip, AdamW) on a Llama layout.
* ``evoformer``: ``DS4Sci_EvoformerAttention`` over MSA rows or triangles, forward alone or with its gradients.

Layer sizes are those of benchmarks/serving.py; weights and tokens are random, drawn from the seed."""
import math
import os

import torch
import torch.nn.functional as F

VOCAB, HEAD, EPS, THETA = 32000, 128, 1e-5, 10000.0
# width -> (feed-forward, query heads, KV heads)
SIZES = {2048: (5632, 16, 4), 4096: (14336, 32, 8)}
# (layout, width) -> (experts, chosen, expert feed-forward, shared feed-forward or 0, weights sum to one)
ROUTED = {("qwen2-moe", 2048): (64, 6, 1024, 2048, False), ("qwen2-moe", 4096): (64, 4, 2048, 4096, False),
          ("mixtral", 2048): (8, 2, 5632, 0, True), ("mixtral", 4096): (8, 2, 14336, 0, True)}
# Router rows this much above unit scale: a trained router is decided about most tokens
ROUTER_SCALE = 4.0
CONTEXT_LIMIT, BLOCK = 8192, 64
LR, BETAS, ADAM_EPS, DECAY, CLIP = 1e-4, (0.9, 0.95), 1e-8, 0.1, 1.0


def _serve(name=None, arch="llama", width=2048, layers=2, decodes=0, context=0, prompts=0, tokens=0, piece=0, quant="",
           latents=False):
    """decodes: sequences that get one token a step, the longest of them with ``context`` cached tokens. prompts: new
    sequences, the longest of ``tokens``; piece: the longest part of a prompt in one step (0: whole)."""
    c = dict(kind="serve", arch=arch, width=width, layers=layers, decodes=decodes, context=context, prompts=prompts,
             tokens=tokens, piece=piece, quant=quant, latents=latents)
    return c if name is None else dict(c, name=name)


def _train(name=None, width=2048, layers=2, batch=1, seq=512):
    c = dict(kind="train", width=width, layers=layers, batch=batch, seq=seq)
    return c if name is None else dict(c, name=name)


def _evoformer(name=None, rows=128, length=256, heads=8, dim=32, train=True):
    c = dict(kind="evoformer", rows=rows, length=length, heads=heads, dim=dim, train=train)
    return c if name is None else dict(c, name=name)


def listed():
    return [
        # one user of a chat model: the step that latency is about, a few hundred MB of weights and few bytes else
        _serve("decode-1", layers=4, decodes=1, context=1000),
        # a server's usual step: many users, contexts of all lengths
        _serve("decode-16", width=4096, decodes=16, context=4000),
        # a prompt of ordinary length before its first token
        _serve("prefill-2048", width=4096, prompts=1, tokens=2048),
        # a long document: attention is as much work as the projections
        _serve("prefill-16k", prompts=1, tokens=16000),
        # a prompt that arrives while others decode: it is taken in pieces beside their tokens, and the latents of all
        # new tokens go to host memory, so that an evicted sequence can be restored from them
        _serve("mixed-latents", width=4096, decodes=9, context=3000, prompts=1, tokens=1301, piece=512, latents=True),
        # routed experts with a shared one, a few users
        _serve("moe-decode-4", arch="qwen2-moe", layers=4, decodes=4, context=1000),
        # the same layout on prompts of odd lengths
        _serve("moe-prefill", arch="qwen2-moe", prompts=3, tokens=701),
        # few large experts, a batch of users: every expert is read in a step
        _serve("mixtral-decode-16", arch="mixtral", width=4096, layers=1, decodes=16, context=2000),
        # weight-only FP6 for a model that would not fit otherwise
        _serve("fp6-decode-8", width=4096, decodes=8, context=1000, quant="wf6af16"),
        # fine-tuning on short texts
        _train("train-short", batch=2, seq=509),
        # pre-training at the layer size of an 8B model
        _train("train-4096", width=4096, batch=2, seq=4096),
        # MSA row attention with mask and pair bias in a training step of a folding model
        _evoformer("evoformer-rows", rows=128, length=256, heads=8),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    what = rng.choice(["decode", "decode", "prefill", "mixed", "moe", "moe", "quant", "train", "evoformer", "evoformer"])
    width = rng.choice([2048, 4096])
    layers = rng.randint(1, 3)
    if what == "decode":
        return _serve(width=width, layers=layers, decodes=_log(rng, 1, 32), context=_log(rng, 20, 4000),
                      latents=rng.random() < 0.25)
    if what == "prefill":
        return _serve(width=width, layers=layers, prompts=rng.randint(1, 4), tokens=_log(rng, 30, 4000))
    if what == "mixed":
        return _serve(width=width, layers=layers, decodes=_log(rng, 1, 32), context=_log(rng, 100, 4000), prompts=1,
                      tokens=_log(rng, 100, 1500), piece=rng.choice([256, 512, 768]), latents=rng.random() < 0.5)
    if what == "moe":
        arch, layers = rng.choice(["qwen2-moe", "mixtral"]), rng.randint(1, 2)
        if rng.random() < 0.5:
            return _serve(arch=arch, width=width, layers=layers, decodes=_log(rng, 1, 32), context=_log(rng, 20, 2000))
        return _serve(arch=arch, width=width, layers=layers, prompts=rng.randint(1, 3), tokens=_log(rng, 30, 1500))
    if what == "quant":
        quant = rng.choice(["wf6af16", "int8", "int4"])
        if rng.random() < 0.7:
            return _serve(width=width, layers=layers, decodes=_log(rng, 1, 32), context=_log(rng, 20, 2000), quant=quant)
        return _serve(width=width, layers=layers, prompts=1, tokens=_log(rng, 30, 2000), quant=quant)
    if what == "train":
        return _train(width=width, layers=rng.randint(1, 2), batch=rng.randint(1, 3), seq=_log(rng, 64, 2500))
    heads = rng.choice([4, 8])
    length = _log(rng, 16, 384)
    rows = _log(rng, 1, 512 if length <= 256 else 256)
    return _evoformer(rows=rows, length=length, heads=heads, dim=rng.choice([32, 32, 64]), train=rng.random() < 0.6)


# ---------------------------------------------------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------------------------------------------------
def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed))


def _normal(gen, *shape, scale=None, mean=0.0):
    w = torch.empty(*shape, dtype=torch.bfloat16, device="cuda")
    return w.normal_(mean, shape[-1]**-0.5 if scale is None else scale, generator=gen)


def _lengths(count, longest, least=1):
    """Ragged lengths, the first the longest: spread over the upper part of the range."""
    return [max(least, int(longest * (1.0 - 0.8 * ((0.618 * i) % 1.0)))) for i in range(count)]


def _sequences(c, seed):
    """Decoding sequences: (context tokens, token of this step ...); prompts: their tokens. On the host, where requests
    come from."""
    g = torch.Generator().manual_seed(int(seed) + 1)
    draw_ids = lambda n: torch.randint(0, VOCAB, (n, ), generator=g)  # noqa: E731
    decoding = [(draw_ids(n), draw_ids(_steps(c))) for n in _lengths(c["decodes"], c["context"])]
    return decoding, [draw_ids(n) for n in _lengths(c["prompts"], c["tokens"])]


def _steps(c):
    """Forward steps of a pass."""
    return -(-c["tokens"] // c["piece"]) if c["piece"] else 1


def _weights(c, seed):
    W = c["width"]
    ff, nq, nkv = SIZES[W]
    g = _gen(seed)
    layers = []
    for _ in range(c["layers"]):
        L = {"ln1.w": _normal(g, W, scale=0.1, mean=1.0), "ln2.w": _normal(g, W, scale=0.1, mean=1.0),
             "qkv.w": _normal(g, (nq + 2 * nkv) * HEAD, W), "o.w": _normal(g, W, nq * HEAD)}
        if (c["arch"], W) in ROUTED:
            E, _, eff, sff, _ = ROUTED[c["arch"], W]
            L.update({"router.w": _normal(g, E, W, scale=ROUTER_SCALE * W**-0.5), "w13": _normal(g, E, 2 * eff, W),
                      "w2": _normal(g, E, W, eff)})
            if sff:
                L.update({"shared.w13": _normal(g, 2 * sff, W), "shared.w2": _normal(g, W, sff),
                          "shared_gate.w": _normal(g, 1, W)})
        else:
            L.update({"up.w": _normal(g, 2 * ff, W), "down.w": _normal(g, W, ff)})
        layers.append(L)
    return {"embed": _normal(g, VOCAB, W, scale=1.0), "final.w": _normal(g, W, scale=0.1, mean=1.0),
            "lm_head.w": _normal(g, VOCAB, W), "layers": layers}


def _prepare_serve(c, seed):
    from hcache_deepspeed_amd.inference.v2.arch import ArchSpec
    from hcache_deepspeed_amd.inference.v2.engine import InferenceEngineV2, RaggedInferenceEngineConfig
    W = c["width"]
    ff, nq, nkv = SIZES[W]
    limit = max(CONTEXT_LIMIT, c["tokens"])
    spec = ArchSpec("llama", VOCAB, W, c["layers"], nq, nkv, HEAD, ff, norm_eps=EPS, rope_theta=THETA,
                    max_position_embeddings=limit)
    if (c["arch"], W) in ROUTED:
        E, top, eff, sff, normalize = ROUTED[c["arch"], W]
        spec.model_type, spec.intermediate_size = c["arch"].replace("-", "_"), eff
        spec.moe = dict(num_experts=E, top_k=top, normalize=normalize, shared=bool(sff), shared_intermediate_size=sff)
    count = c["decodes"] + c["prompts"]
    conf = RaggedInferenceEngineConfig.from_dict(dict(
        dtype="bf16", quantization={"quantization_mode": c["quant"]} if c["quant"] else {},
        state_manager=dict(max_context=limit, max_ragged_batch_size=max(8192, c["prompts"] * c["tokens"] + 64),
                           max_tracked_sequences=max(4, count), kv_block_size=BLOCK)))
    blocks = c["decodes"] * (CONTEXT_LIMIT // BLOCK) + c["prompts"] * (-(-c["tokens"] // BLOCK) + 1)
    eng = InferenceEngineV2(spec, _weights(c, seed), conf, device=torch.device("cuda", 0), num_kv_blocks=blocks)
    decoding, prompts = _sequences(c, seed)
    s = dict(c, engine=eng, decoding=decoding, prompts=prompts, left=0)
    _begin(s)
    return s


def _begin(s):
    """The decoding sequences' contexts, in as few steps as the batch limit allows."""
    eng, uids, batch, room = s["engine"], [], [], 8192
    for u, (ctx, _) in enumerate(s["decoding"]):
        eng.flush(u)
        if uids and room < ctx.numel():
            eng.put(uids, batch, capture_latents=False)
            uids, batch, room = [], [], 8192
        uids.append(u)
        batch.append(ctx)
        room -= ctx.numel()
    if uids:
        eng.put(uids, batch, capture_latents=False)
    s["left"] = CONTEXT_LIMIT - max([c.numel() for c, _ in s["decoding"]], default=0) if uids else 1 << 60


def _run_serve(s):
    eng, n, steps = s["engine"], s["decodes"], _steps(s)
    s["left"] -= steps
    if s["left"] < 0:  # sequences have come to their longest: the next ones begin
        _begin(s)
    logits, latents = [], []
    for i in range(steps):
        uids = list(range(n))
        batch = [t[i:i + 1] for _, t in s["decoding"]]
        for j, p in enumerate(s["prompts"]):
            part = p if not s["piece"] else p[i * s["piece"]:(i + 1) * s["piece"]]
            if part.numel():
                uids.append(n + j)
                batch.append(part)
        z, lat = eng.put(uids, batch, capture_latents=s["latents"])
        logits.append(z)
        if s["latents"]:
            latents += lat
    for j in range(len(s["prompts"])):
        eng.flush(n + j)
    return {"logits": logits, "latents": latents}


def _train_config(c):
    from hcache_deepspeed_amd.models.llama import LlamaConfig
    ff, nq, nkv = SIZES[c["width"]]
    return LlamaConfig(vocab_size=VOCAB, hidden_size=c["width"], intermediate_size=ff, num_hidden_layers=c["layers"],
                       num_attention_heads=nq, num_key_value_heads=nkv, rms_norm_eps=EPS, rope_theta=THETA,
                       max_position_embeddings=4096)


def _train_weights(c, seed):
    """Names and values of the model's parameters."""
    W, g = c["width"], _gen(seed)
    ff, nq, nkv = SIZES[W]
    w = {"model.embed_tokens.weight": _normal(g, VOCAB, W, scale=1.0)}
    for i in range(c["layers"]):
        p = f"model.layers.{i}."
        w[p + "input_layernorm.weight"] = _normal(g, W, scale=0.1, mean=1.0)
        w[p + "self_attn.qkv_proj.weight"] = _normal(g, (nq + 2 * nkv) * HEAD, W)
        w[p + "self_attn.o_proj.weight"] = _normal(g, W, nq * HEAD)
        w[p + "post_attention_layernorm.weight"] = _normal(g, W, scale=0.1, mean=1.0)
        w[p + "mlp.gate_up_proj.weight"] = _normal(g, 2 * ff, W)
        w[p + "mlp.down_proj.weight"] = _normal(g, W, ff)
    w["model.norm.weight"] = _normal(g, W, scale=0.1, mean=1.0)
    w["lm_head.weight"] = _normal(g, VOCAB, W)
    return w


def _tokens(c, seed):
    return torch.randint(0, VOCAB, (c["batch"], c["seq"]), device="cuda", generator=_gen(seed + 1))


def _prepare_train(c, seed):
    import hcache_deepspeed_amd as hds
    from hcache_deepspeed_amd.models.llama import LlamaForCausalLM
    for k, v in dict(RANK="0", WORLD_SIZE="1", LOCAL_RANK="0", MASTER_ADDR="127.0.0.1", MASTER_PORT="29547").items():
        os.environ.setdefault(k, v)
    with torch.device("cuda"):
        model = LlamaForCausalLM(_train_config(c))
    model.load_state_dict(_train_weights(c, seed))
    names = [n for n, _ in model.named_parameters()]
    engine, _, _, _ = hds.initialize(model=model, config={
        "train_micro_batch_size_per_gpu": c["batch"], "bf16": {"enabled": True}, "gradient_clipping": CLIP,
        "optimizer": {"type": "AdamW", "params": {"lr": LR, "betas": list(BETAS), "eps": ADAM_EPS, "weight_decay": DECAY}},
        "zero_optimization": {"stage": 3}, "steps_per_print": 1000000})
    # the optimizer's own 32-bit weights and first moments, by parameter
    z = engine.optimizer
    state = {"master": {}, "exp_avg": {}}
    for name, p in zip(names, model.parameters()):
        u, i = z.param_to_unit[id(p)]
        for key, flat in (("master", z.store.master), ("exp_avg", z.store.states["exp_avg"])):
            state[key][name] = u.param_view(flat[u.store_off:u.store_off + u.shard], i)
    return dict(c, engine=engine, ids=_tokens(c, seed), state=state)


def _run_train(s):
    engine, ids = s["engine"], s["ids"]
    loss = engine(ids, labels=ids)
    engine.backward(loss)
    engine.step()
    return dict(s["state"], loss=loss.detach())


def _evoformer_inputs(c, seed):
    N, L, H, D = c["rows"], c["length"], c["heads"], c["dim"]
    g = _gen(seed)
    q, k, v, do = (_normal(g, 1, N, L, H, D, scale=1.0) for _ in range(4))
    # one residue in ten of a row is padding or a gap
    gone = torch.rand(1, N, 1, 1, L, device="cuda", generator=g) < 0.1
    gone[..., 0] = False
    mask = gone.to(torch.bfloat16) * -1e9
    return q, k, v, mask, _normal(g, 1, 1, H, L, L, scale=1.0), do


def prepare(case, seed):
    if case["kind"] == "serve":
        return _prepare_serve(case, seed)
    if case["kind"] == "train":
        return _prepare_train(case, seed)
    q, k, v, mask, pair, do = _evoformer_inputs(case, seed)
    for t in (q, k, v, pair):
        t.requires_grad_(case["train"])
    return dict(case, args=(q, k, v, [mask, pair]), do=do)


def run(state):
    if state["kind"] == "serve":
        return _run_serve(state)
    if state["kind"] == "train":
        return _run_train(state)
    from hcache_deepspeed_amd.ops.deepspeed4science import DS4Sci_EvoformerAttention
    q, k, v, biases = state["args"]
    if not state["train"]:
        with torch.no_grad():
            return [DS4Sci_EvoformerAttention(q, k, v, biases)]
    o = DS4Sci_EvoformerAttention(q, k, v, biases)
    return [o.detach()] + list(torch.autograd.grad(o, (q, k, v, biases[1]), state["do"]))


# ---------------------------------------------------------------------------------------------------------------------
# what a pass cannot do without
# ---------------------------------------------------------------------------------------------------------------------
def _layer_sizes(arch, width):
    """Parameters of a layer that every token meets, and of one expert."""
    ff, nq, nkv = SIZES[width]
    attn = width * (nq + 2 * nkv) * HEAD + width * nq * HEAD + 2 * width
    if (arch, width) not in ROUTED:
        return attn + 3 * width * ff, 0
    E, _, eff, sff, _ = ROUTED[arch, width]
    return attn + width * E + 3 * width * sff + (width if sff else 0), 3 * width * eff


def _work_serve(c):
    W = c["width"]
    _, nq, nkv = SIZES[W]
    common, expert = _layer_sizes(c["arch"], W)
    E, top = ROUTED[c["arch"], W][:2] if expert else (0, 0)
    per = {"": 2.0, "int8": 1.0 + 4 / 128, "wf6af16": 0.75 + 4 / 128, "int4": 0.5 + 4 / 128}[c["quant"]]
    kv = 2 * nkv * HEAD * 2
    nbytes = flops = 0.0
    ctx = _lengths(c["decodes"], c["context"])
    lens = _lengths(c["prompts"], c["tokens"])
    for i in range(_steps(c)):
        pieces = [(0, n) if not c["piece"] else (i * c["piece"], min(n, (i + 1) * c["piece"])) for n in lens]
        new = [(n + i, n + i + 1) for n in ctx] + [(a, b) for a, b in pieces if b > a]
        T = sum(b - a for a, b in new)
        touched = E * (1 - (1 - top / E)**T) if E else 0
        nbytes += c["layers"] * (per * common + 2.0 * touched * expert + kv * sum(b for _, b in new) + kv * T)
        nbytes += 2.0 * VOCAB * W + 2.0 * T * W + 2.0 * len(new) * VOCAB
        if c["latents"]:
            nbytes += c["layers"] * T * W * 2
        flops += c["layers"] * (2.0 * T * (common + top * expert) +
                                sum(4.0 * nq * HEAD * (b - a) * (a + b + 1) / 2 for a, b in new))
        flops += 2.0 * len(new) * VOCAB * W
    return {"bytes": nbytes, "flops": flops}


def work(case):
    c = case
    if c["kind"] == "serve":
        return _work_serve(c)
    if c["kind"] == "train":
        W, T = c["width"], c["batch"] * c["seq"]
        _, nq, _ = SIZES[W]
        N = c["layers"] * _layer_sizes("llama", W)[0] + VOCAB * W
        # weights read twice, gradients written and read, weights, both moments and the 16-bit copy updated; the
        # embedding's rows likewise; activations that the backward needs, at least the input of each product
        nbytes = (N + VOCAB * W) * (2 * 2 + 2 * 2 + 6 * 4 + 2) + c["layers"] * T * 2 * 2 * (8 * W)
        return {"bytes": float(nbytes), "flops": 6.0 * T * N + c["layers"] * c["batch"] * 3 * 2.0 * nq * HEAD * c["seq"] *
                (c["seq"] + 1)}
    N, L, H, D = c["rows"], c["length"], c["heads"], c["dim"]
    x, pair = 2.0 * N * L * H * D, 2.0 * H * L * L
    return {"bytes": (4 + (8 if c["train"] else 0)) * x + (3 if c["train"] else 1) * pair + 2.0 * N * L,
            "flops": (14 if c["train"] else 4) * 1.0 * N * H * L * L * D}


def tolerance(case):
    # about four times the distance from 64 bits: 0.3 - 0.7 % through two to four bf16 layers, 0.9 - 1.1 % with routed
    # experts (a token near a tie goes to another expert), 0.6 - 0.9 % in gradients, 0.3 % in one attention
    if case["kind"] == "serve":
        return {"rel": 0.03, "max": 0.4} if case["arch"] != "llama" else {"rel": 0.025, "max": 0.2}
    if case["kind"] == "train":
        return {"rel": 0.03, "max": 0.5}
    return {"rel": 0.01, "max": 0.1}


# ---------------------------------------------------------------------------------------------------------------------
# the same in 64 bits
# ---------------------------------------------------------------------------------------------------------------------
def _rms(x, w):
    return x * torch.rsqrt((x * x).mean(-1, keepdim=True) + EPS) * w


def _rotate(x):
    """x: [T, heads, HEAD], halves of a head are the pairs."""
    T, half = x.shape[0], HEAD // 2
    inv = THETA**(-torch.arange(half, dtype=torch.float64, device=x.device) / half)
    a = torch.arange(T, dtype=torch.float64, device=x.device)[:, None] * inv
    cos, sin = a.cos()[:, None], a.sin()[:, None]
    x1, x2 = x[..., :half], x[..., half:]
    return torch.cat([x1 * cos - x2 * sin, x2 * cos + x1 * sin], -1)


def _attend(q, k, v):
    """Causal attention, q: [T, nq, HEAD], k and v: [T, nkv, HEAD]."""
    T, nq, _ = q.shape
    G = nq // k.shape[1]
    k, v = (x.repeat_interleave(G, 1).transpose(0, 1) for x in (k, v))
    out, step = [], max(1, (1 << 28) // T)
    rows = max(1, step // nq)
    at = torch.arange(T, device=q.device)
    for r in range(0, T, rows):
        n = min(T, r + rows)
        s = q[r:n].transpose(0, 1) @ k[:, :n].transpose(1, 2) * HEAD**-0.5
        s = s.masked_fill(at[None, :n] > at[r:n, None], -math.inf)
        out.append((torch.softmax(s, -1) @ v[:, :n]).transpose(0, 1))
    return torch.cat(out).reshape(T, nq * HEAD)


def _swiglu(x, up):
    g, u = (x @ up.T).chunk(2, -1)
    return F.silu(g) * u


def _experts(x, L, c):
    E, top, _, sff, normalize = ROUTED[c["arch"], c["width"]]
    p = torch.softmax(x @ L["router.w"].double().T, -1)
    weight, chosen = p.topk(top, -1)
    if normalize:
        weight = weight / weight.sum(-1, keepdim=True)
    y = torch.zeros_like(x)
    for e in range(E):
        t, j = (chosen == e).nonzero(as_tuple=True)
        if t.numel():
            y.index_add_(0, t, weight[t, j, None] * (_swiglu(x[t], L["w13"][e].double()) @ L["w2"][e].double().T))
    if sff:
        y += torch.sigmoid(x @ L["shared_gate.w"].double().T) * (
            _swiglu(x, L["shared.w13"].double()) @ L["shared.w2"].double().T)
    return y


def _stored(w, mode):
    """The values that a weight-only quantized matrix stands for: groups of 128 along its rows."""
    if not mode:
        return w.double()
    g = w.float().reshape(-1, 128)
    top = g.abs().amax(1, keepdim=True)
    if mode == "wf6af16":  # e3m2: largest value 28, steps of 2^(e - 2), the smallest exponent -2
        s = top / 28
        a = (g / s).abs()
        step = torch.exp2(torch.floor(torch.log2(a.clamp_min(2.0**-2))) - 2)
        q = torch.sign(g) * (torch.round(a / step) * step).clamp_max(28)
    else:
        most = 127 if mode == "int8" else 7
        s = top / most
        q = torch.round(g / s).clamp(-most - 1, most)
    return (q * s).double().view(w.shape)


def _exact_serve(c, seed):
    w = _weights(c, seed)
    ff, nq, nkv = SIZES[c["width"]]
    decoding, prompts = _sequences(c, seed)
    seqs = [torch.cat([a, b]).cuda() for a, b in decoding] + [p.cuda() for p in prompts]
    xs = [w["embed"][ids].double() for ids in seqs]
    normed = [[] for _ in seqs]
    for L in w["layers"]:
        qkv_w, o_w = _stored(L["qkv.w"], c["quant"]), _stored(L["o.w"], c["quant"])
        dense = "up.w" in L
        if dense:
            up, down = _stored(L["up.w"], c["quant"]), _stored(L["down.w"], c["quant"])
        for n, x in enumerate(xs):
            h = _rms(x, L["ln1.w"].double())
            if c["latents"]:
                normed[n].append(h)
            q, k, v = (h @ qkv_w.T).view(-1, nq + 2 * nkv, HEAD).split([nq, nkv, nkv], 1)
            x = x + _attend(_rotate(q), _rotate(k), v) @ o_w.T
            h = _rms(x, L["ln2.w"].double())
            xs[n] = x + (_swiglu(h, up) @ down.T if dense else _experts(h, L, c))
    head = w["lm_head.w"].double()
    logits, latents = [], []
    for i in range(_steps(c)):
        rows = []
        for n, x in enumerate(xs):
            if n < c["decodes"]:
                a = x.shape[0] - _steps(c) + i
                b = a + 1
            else:
                a, b = (0, x.shape[0]) if not c["piece"] else (i * c["piece"], min(x.shape[0], (i + 1) * c["piece"]))
            if b <= a:
                continue
            rows.append(_rms(x[b - 1], w["final.w"].double()) @ head.T)
            if c["latents"]:
                latents.append(torch.stack([h[a:b] for h in normed[n]]))
        logits.append(torch.stack(rows))
    return {"logits": logits, "latents": latents}


def _exact_train(c, seed):
    W = c["width"]
    ff, nq, nkv = SIZES[W]
    w = {k: v.double().requires_grad_() for k, v in _train_weights(c, seed).items()}
    ids = _tokens(c, seed)
    total = 0.0
    count = c["batch"] * (c["seq"] - 1)
    for row in ids:  # one sequence after the other: the loss is a sum over them
        x = F.embedding(row, w["model.embed_tokens.weight"])
        for i in range(c["layers"]):
            p = f"model.layers.{i}."
            h = _rms(x, w[p + "input_layernorm.weight"])
            q, k, v = (h @ w[p + "self_attn.qkv_proj.weight"].T).view(-1, nq + 2 * nkv, HEAD).split([nq, nkv, nkv], 1)
            x = x + _attend(_rotate(q), _rotate(k), v) @ w[p + "self_attn.o_proj.weight"].T
            h = _rms(x, w[p + "post_attention_layernorm.weight"])
            x = x + _swiglu(h, w[p + "mlp.gate_up_proj.weight"]) @ w[p + "mlp.down_proj.weight"].T
        z = _rms(x, w["model.norm.weight"])[:-1] @ w["lm_head.weight"].T
        loss = F.cross_entropy(z, row[1:], reduction="sum") / count
        loss.backward()
        total += loss.item()
    norm = math.sqrt(sum(p.grad.square().sum().item() for p in w.values()))
    coef = min(1.0, CLIP / (norm + 1e-6))
    out = {"master": {}, "exp_avg": {}, "loss": torch.tensor(total, dtype=torch.float64)}
    for name, p in w.items():
        g, p = p.grad * coef, p.detach()
        out["exp_avg"][name] = (1 - BETAS[0]) * g
        out["master"][name] = p - LR * (g / (g.abs() + ADAM_EPS) + DECAY * p)
    return out


def _exact_evoformer(c, seed):
    q, k, v, mask, pair, do = (t[0].double() for t in _evoformer_inputs(c, seed))
    D = c["dim"]
    o, dq, dk, dv = (torch.empty_like(q) for _ in range(4))
    dpair = torch.zeros_like(pair)
    for n in range(c["rows"]):
        a, b, e = (t[n].transpose(0, 1) for t in (q, k, v))  # [H, L, D]
        p = torch.softmax(a @ b.transpose(1, 2) * D**-0.5 + mask[n] + pair[0], -1)
        o[n] = (p @ e).transpose(0, 1)
        if c["train"]:
            d = do[n].transpose(0, 1)
            dp = d @ e.transpose(1, 2)
            ds = p * (dp - (p * dp).sum(-1, keepdim=True))
            dq[n] = (ds @ b * D**-0.5).transpose(0, 1)
            dk[n] = (ds.transpose(1, 2) @ a * D**-0.5).transpose(0, 1)
            dv[n] = (p.transpose(1, 2) @ d).transpose(0, 1)
            dpair[0] += ds
    return [t[None] for t in ([o, dq, dk, dv, dpair] if c["train"] else [o])]


def exact(case, seed):
    if case["kind"] == "train":
        return _exact_train(case, seed)
    with torch.no_grad():
        return _exact_serve(case, seed) if case["kind"] == "serve" else _exact_evoformer(case, seed)
