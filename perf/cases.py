"""Workloads of the Qwen3.5-2B decoder path, timed one pass at a time.

Every case goes through the entry points a program uses: the modules of a
fused model (``layer.mlp``, ``layer.linear_attn``, ``layer.self_attn``, the
model itself, the vision tower), ``integration.decode_layer`` for decode, and
``kernels.lm_head_argmax`` for the greedy head. Shapes are those of
``ppu_amd.synth.config_2b`` and of Transformers' default vision config; prompt
lengths, contexts and image sizes span what the tests and the benchmark use.

``captured`` cases replay a captured graph, as the generator does for a prompt
length it has seen and for every decode step; the others launch eagerly, as a
first-seen length does. Prefill passes start by resetting the cache, as each
prompt does.

``exact`` restates each path in 64-bit torch, without the package.
"""

from __future__ import annotations

import inspect
import math

import torch

from ppu_amd import integration, kernels, synth
from ppu_amd.generate import cache_bucket, reset_cache

DEV = "cuda"
BF16 = torch.bfloat16
HID, INTER, QH, KVH, HD, LH, LD = 2048, 6144, 8, 2, 256, 16, 128
VOCAB = 248320
PERIOD = ["linear_attention"] * 3 + ["full_attention"]
CAPTURE_BELOW = 2000  # prompt tokens: shorter prompts replay a captured graph


# ------------------------------------------------------------------ cases
def listed():
    return [
        # one generated token through a period of the decoder (3 DeltaNet
        # layers, 1 attention layer) at the benchmark's context
        {"name": "decode bf16 ctx 1040", "kind": "decode", "int8": False, "context": 1040},
        # int8 linears (one DeltaNet and one attention layer), a long document
        # in the cache
        {"name": "decode int8 ctx 8000", "kind": "decode", "int8": True, "context": 8000},
        # the greedy token of one step: the whole vocabulary's head
        {"name": "head 248320", "kind": "head", "vocab": VOCAB},
        # a short chat turn through an MLP
        {"name": "mlp bf16 37", "kind": "mlp", "int8": False, "tokens": 37},
        # a question of ordinary length, int8
        {"name": "mlp int8 333", "kind": "mlp", "int8": True, "tokens": 333},
        # a long document, bf16
        {"name": "mlp bf16 4096", "kind": "mlp", "int8": False, "tokens": 4096},
        # an image-and-question prompt through a DeltaNet mixer
        {"name": "delta bf16 340", "kind": "delta", "int8": False, "tokens": 340},
        # a ragged long prompt, int8
        {"name": "delta int8 2003", "kind": "delta", "int8": True, "tokens": 2003},
        # the benchmark's prompt through an attention mixer
        {"name": "attention bf16 1024", "kind": "attention", "int8": False, "tokens": 1024},
        # the longest document the benchmark's contexts cover
        {"name": "attention bf16 8192", "kind": "attention", "int8": False, "tokens": 8192},
        # one 448 x 448 image through the vision tower
        {"name": "vision 28x28", "kind": "vision", "images": 1, "height": 28, "width": 28},
        # a whole prefill call of a period-deep decoder, logits of the last token
        {"name": "model bf16 1000", "kind": "model", "int8": False, "tokens": 1000},
    ]


def draw(rng):
    def log(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    kind = rng.choice(["decode", "head", "mlp", "mlp", "mlp", "delta", "delta", "attention", "attention",
                       "vision", "model"])
    if kind == "head":
        return {"kind": kind, "vocab": rng.randrange(50001, VOCAB, 2)}
    if kind == "vision":
        images = rng.choice([1, 1, 2, 3])
        most = 784 // images  # patches of one image
        height = 2 * rng.randint(5, most // 20)
        return {"kind": kind, "images": images, "height": height,
                "width": 2 * rng.randint(5, max(5, most // height // 2))}
    int8 = rng.random() < 0.5
    if kind == "decode":
        return {"kind": kind, "int8": int8, "context": log(100, 16000)}
    tokens = {"mlp": log(2, 6000), "delta": log(17, 8000), "attention": log(17, 8000),
              "model": log(17, 2000)}[kind]
    return {"kind": kind, "int8": int8, "tokens": tokens}


# ------------------------------------------------------------------ inputs
def _generator(seed):
    return torch.Generator(device=DEV).manual_seed(seed)


def _normal(g, *shape, std=1.0, mean=0.0, dtype=BF16):
    return (torch.randn(shape, generator=g, device=DEV, dtype=torch.float32) * std + mean).to(dtype)


def _layers(case):
    # int8: fewer layers, as a rounding that moves a quantised activation by
    # one step travels through every layer after it
    if case["kind"] == "decode":
        return PERIOD[2:] if case["int8"] else PERIOD
    if case["kind"] == "model":
        return PERIOD[:1] if case["int8"] else PERIOD
    return ["full_attention"] if case["kind"] == "attention" else ["linear_attention"]


def _config(case):
    layers = _layers(case)
    return synth.config_2b(num_hidden_layers=len(layers), layer_types=list(layers),
                           vocab_size=VOCAB if case["kind"] == "model" else 512)


def _on_meta(cls, cfg):
    old = torch.get_default_dtype()
    torch.set_default_dtype(BF16)
    try:
        with torch.device("meta"):
            return cls(cfg)
    finally:
        torch.set_default_dtype(old)


def _text_weight(g, name, shape):
    # projections, embeddings and the (1 + w) norms ~N(0, 0.02); the gated
    # norm multiplies directly, so it sits around one
    return _normal(g, *shape, std=0.02, mean=1.0 if name.endswith("linear_attn.norm.weight") else 0.0)


def _text_shapes(case):
    model = _on_meta(integration.qwen_impl.Qwen3_5ForCausalLM, _config(case))
    return model, [(n, tuple(p.shape)) for n, p in model.named_parameters()]


def _vision_weight(g, name, shape):
    if name.endswith(("norm.weight", "norm1.weight", "norm2.weight")):
        return _normal(g, *shape, std=0.02, mean=1.0)
    return _normal(g, *shape, std=0.02)


def _vision_tower():
    cfg = integration.qwen_impl.Qwen3_5VisionConfig()
    cfg._attn_implementation = "sdpa"
    tower = _on_meta(integration.qwen_impl.Qwen3_5VisionModel, cfg)
    return cfg, tower, [(n, tuple(p.shape)) for n, p in tower.named_parameters()]


def _patches(case):
    return case["images"] * case["height"] * case["width"]


def _data(case, seed):
    """The random tensors of a case, the same for ``prepare`` and ``exact``:
    (weights by parameter name, inputs by name)."""
    g = _generator(seed)
    kind, weights, inputs = case["kind"], {}, {}
    if kind == "head":
        weights["w"] = _normal(g, case["vocab"], HID, std=0.02)
        inputs["hidden"] = _normal(g, 1, HID)
        return weights, inputs
    if kind == "vision":
        cfg, _, shapes = _vision_tower()
        for name, shape in shapes:
            weights[name] = _vision_weight(g, name, shape)
        width = cfg.in_channels * cfg.temporal_patch_size * cfg.patch_size**2
        inputs["pixels"] = _normal(g, _patches(case), width)
        return weights, inputs
    for name, shape in _text_shapes(case)[1]:
        weights[name] = _text_weight(g, name, shape)
    if kind == "model":
        inputs["ids"] = torch.randint(0, VOCAB, (1, case["tokens"]), generator=g, device=DEV)
    elif kind == "decode":
        inputs["residual"] = _normal(g, 1, 1, HID)
        inputs["update"] = _normal(g, 1, 1, HID, std=0.5)
        cache_len = cache_bucket(case["context"], 64)
        for i, layer in enumerate(_layers(case)):
            if layer == "full_attention":
                inputs[f"keys{i}"] = _normal(g, 1, KVH, cache_len, HD)
                inputs[f"values{i}"] = _normal(g, 1, KVH, cache_len, HD)
            else:
                inputs[f"conv{i}"] = _normal(g, 1, 3 * LH * LD, 4)
                inputs[f"rec{i}"] = _normal(g, 1, LH, LD, LD, std=0.1, dtype=torch.float32)
    else:
        inputs["x"] = _normal(g, 1, case["tokens"], HID)  # a normalised hidden state
    return weights, inputs


def _fused_model(case, weights):
    model, _ = _text_shapes(case)
    model = model.to_empty(device=DEV)
    model.tie_weights()
    with torch.no_grad():
        for name, p in model.named_parameters():
            p.copy_(weights[name])
        rot = model.model.rotary_emb
        inv_freq, _ = rot.compute_default_rope_parameters(model.config, torch.device(DEV))
        rot.inv_freq.copy_(inv_freq)
        rot.original_inv_freq.copy_(inv_freq)
    model.eval()
    config = integration.FusionConfig(a8w8=case["int8"], lm_head_screen=False)
    integration.apply_fusions(model, config)
    return model


def _static_cache(model, length):
    return inspect.getmodule(integration.DynamicCache).StaticCache(config=model.config, max_cache_len=length)


def _captured(step):
    """A graph of ``step`` (run once eagerly before, as every captured path is)."""
    step()
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = step()

    def replay():
        graph.replay()
        return out

    replay.step = step  # the graph reads the model's and the inputs' memory: they live as long as it does
    return replay


def prepare(case, seed):
    weights, inputs = _data(case, seed)
    kind = case["kind"]
    with torch.no_grad():
        if kind == "head":
            w, hidden = weights["w"], inputs["hidden"]
            screen = kernels.lm_head_screen_prep(w)
            return {"step": lambda: kernels.lm_head_argmax(hidden, w, screen=screen)}
        if kind == "vision":
            return {"step": _vision_step(case, weights, inputs)}
        model = _fused_model(case, weights)
        del weights
        step = {"mlp": _mlp_step, "delta": _mixer_step, "attention": _mixer_step, "decode": _decode_step,
                "model": _model_step}[kind](case, model, inputs)
        if kind == "decode":
            return {"step": step}
        if kind != "model" and case["tokens"] < CAPTURE_BELOW:
            step = _captured(step)
        else:
            step()  # the cache's buffers exist after a program's first prompt
    return {"step": step}


def run(state):
    with torch.no_grad():
        return state["step"]()


def _mlp_step(case, model, inputs):
    mlp, x = model.model.layers[0].mlp, inputs["x"]
    return lambda: {"y": mlp(x)}


def _mixer_step(case, model, inputs):
    layer, x, tokens = model.model.layers[0], inputs["x"], case["tokens"]
    cache = _static_cache(model, cache_bucket(tokens, 64))
    slot = cache.layers[0]
    if case["kind"] == "delta":
        def step():
            reset_cache(cache)
            y = layer.linear_attn(hidden_states=x, cache_params=cache)
            return {"y": y, "state": slot.recurrent_states[0], "conv": slot.conv_states[0]}
        return step
    rope = model.model.rotary_emb(x, torch.arange(tokens, device=DEV).view(1, -1))

    def step():
        reset_cache(cache)
        y, _ = layer.self_attn(hidden_states=x, position_embeddings=rope, attention_mask=None,
                               past_key_values=cache)
        return {"y": y, "keys": slot.keys, "values": slot.values}
    return step


def _decode_step(case, model, inputs):
    stack, context, layers = model.model, case["context"], _layers(case)
    cache = _static_cache(model, cache_bucket(context, 64))
    positions = torch.full((1, 1), context, device=DEV, dtype=torch.long)
    ctx = integration.DecodeContext(cache, positions, True)
    length = cache.layers[-1]  # the attention layer's

    def chain():
        residual, update = inputs["residual"], inputs["update"]
        for i in range(len(layers)):
            residual, update = integration.decode_layer(stack, i, residual, update, ctx)
        return residual, update

    chain()  # allocates the cache
    for i, layer in enumerate(layers):
        slot = cache.layers[i]
        if layer == "full_attention":
            slot.keys.copy_(inputs[f"keys{i}"])
            slot.values.copy_(inputs[f"values{i}"])

    def restore():
        for i, layer in enumerate(layers):
            if layer != "full_attention":
                cache.layers[i].conv_states[0].copy_(inputs[f"conv{i}"])
                cache.layers[i].recurrent_states[0].copy_(inputs[f"rec{i}"])

    def step():
        # every pass decodes the token after the same context
        length.cumulative_length.fill_(context)
        residual, update = chain()
        out = {"residual": residual, "update": update, "keys": length.keys, "values": length.values}
        for i, layer in enumerate(layers):
            if layer != "full_attention":
                out[f"rec{i}"] = cache.layers[i].recurrent_states[0]
                out[f"conv{i}"] = cache.layers[i].conv_states[0]
        return out

    replay = _captured(step)
    restore()
    return replay


def _model_step(case, model, inputs):
    ids, tokens, layers = inputs["ids"], case["tokens"], _layers(case)
    cache = _static_cache(model, cache_bucket(tokens, 64))
    positions = torch.arange(tokens, device=DEV).view(1, -1)

    def step():
        reset_cache(cache)
        out = model(input_ids=ids, position_ids=positions, past_key_values=cache, use_cache=True,
                    logits_to_keep=1)
        result = {"logits": out.logits}
        for i, layer in enumerate(layers):
            slot = cache.layers[i]
            if layer == "full_attention":
                result.update(keys=slot.keys, values=slot.values)
            else:
                result[f"rec{i}"] = slot.recurrent_states[0]
        return result
    return step


def _vision_step(case, weights, inputs):
    cfg, tower, _ = _vision_tower()
    tower = tower.to_empty(device=DEV)
    for name, p in tower.named_parameters():
        p.copy_(weights[name])
    tower.rotary_pos_emb.inv_freq = _vision_inv_freq(cfg).float()
    tower.eval()
    integration.install_vision(tower, integration.FusionConfig())
    grid = torch.tensor([[1, case["height"], case["width"]]] * case["images"], device=DEV)
    pixels = inputs["pixels"]

    def step():
        out = tower(pixels, grid_thw=grid)
        return {"hidden": out.last_hidden_state, "merged": out.pooler_output}

    step()  # a size's first image captures its graph
    return step


# ------------------------------------------------------------------ work
def work(case):
    kind = case["kind"]
    if kind == "head":
        v = case["vocab"]
        return {"bytes": v * HID + 8 * v + 2 * HID, "flops": 2 * v * HID}  # the int8 screen's rows
    if kind == "vision":
        t, per = _patches(case), case["height"] * case["width"]
        block = 4 * 1152 * 1152 + 2 * 1152 * 4304
        merged = 4608 * 4608 + 4608 * 2048  # weights of the merger; rows t / 4
        other = 1536 * 1152
        params = 27 * block + merged + other
        flops = 2 * t * (27 * block + other) + t // 2 * merged + 27 * 4 * t * per * 1152
        return {"bytes": 2 * params + 2 * t * (1536 + 1152 + 512), "flops": flops}
    es = 1 if case["int8"] else 2
    mlp, delta, attn = 3 * HID * INTER, (4 * HID + 2 * LH) * HID + HID * HID, 5120 * HID + HID * HID
    state = 2 * LH * LD * LD * 4 + 2 * 3 * LH * LD * 4 * 2
    if kind == "decode":
        n = case["context"] + 1
        deltas = len(_layers(case)) - 1
        weights = (deltas + 1) * mlp + deltas * delta + attn
        return {"bytes": es * weights + deltas * state + 4 * KVH * HD * n + 8 * HID,
                "flops": 2 * weights + 4 * QH * HD * n + deltas * 6 * LH * LD * LD}
    m = case["tokens"]
    rows = 4 * m * HID  # hidden rows in and out
    recurrence, softmax = 6 * m * LH * LD * LD, 2 * QH * HD * m * (m + 1)
    if kind == "mlp":
        return {"bytes": es * mlp + rows, "flops": 2 * m * mlp}
    if kind == "delta":
        return {"bytes": es * delta + rows + state // 2, "flops": 2 * m * delta + recurrence}
    if kind == "attention":
        return {"bytes": es * attn + rows + 4 * KVH * HD * m, "flops": 2 * m * attn + softmax}
    layers = _layers(case)
    attns = layers.count("full_attention")
    deltas = len(layers) - attns
    weights = len(layers) * mlp + deltas * delta + attns * attn
    return {"bytes": es * weights + 2 * VOCAB * HID + 2 * m * HID + attns * 4 * KVH * HD * m + deltas * state // 2,
            "flops": 2 * m * weights + deltas * recurrence + attns * softmax + 2 * VOCAB * HID}


def tolerance(case):
    kind = case["kind"]
    if kind == "head":
        return "exact"
    # about four times what the path measures against exact(): 0.004 for a
    # bf16 block, 0.014 where a step of an int8 activation may move, 0.013
    # through the 27 vision blocks
    if kind == "vision" or case["int8"]:
        return {"rel": 0.03}
    return {"rel": 0.03 if kind == "model" else 0.02}


# ------------------------------------------------------------------ exact
def _linear(x, w, int8):
    """x @ w.T in 64 bits; int8: on the path's quantised operands (per-row
    weights, per-token activations), exact integer products."""
    w = w.double()
    if not int8:
        return x @ w.t()
    sw = w.abs().amax(-1) / 127.0
    qw = torch.round(w / torch.where(sw > 0, sw, 1.0)[:, None]).clamp(-127, 127)
    top = x.abs().amax(-1, keepdim=True)
    qx = torch.round(x * torch.where(top > 0, 127.0 / top, 0.0)).clamp(-128, 127)
    return (qx @ qw.t()) * (top / 127.0) * sw


def _rms(x, w):
    return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + 1e-6) * (1.0 + w.double())


def _silu(x):
    return x * torch.sigmoid(x)


def _mlp64(w, p, x, int8):
    gate = _linear(x, w[p + "mlp.gate_proj.weight"], int8)
    return _linear(_silu(gate) * _linear(x, w[p + "mlp.up_proj.weight"], int8), w[p + "mlp.down_proj.weight"], int8)


def _delta64(w, p, x, int8, rec=None, conv=None):
    """x [T, HID] -> (y, state, conv state); one token continues from ``conv``."""
    p = p + "linear_attn."
    t = x.shape[0]
    qkv = _linear(x, w[p + "in_proj_qkv.weight"], int8)
    z = _linear(x, w[p + "in_proj_z.weight"], int8).view(t, LH, LD)
    a = _linear(x, w[p + "in_proj_a.weight"], int8)
    b = _linear(x, w[p + "in_proj_b.weight"], int8)
    taps = w[p + "conv1d.weight"].double()[:, 0, :]
    before = qkv.new_zeros(3, qkv.shape[1]) if conv is None else conv[0].double().t()[1:]
    rows = torch.cat((before, qkv))
    mixed = _silu(sum(rows[i : i + t] * taps[:, i] for i in range(4)))
    q, k, v = mixed.view(t, 3, LH, LD).unbind(1)
    q = q * torch.rsqrt(q.square().sum(-1, keepdim=True) + 1e-6) / math.sqrt(LD)
    k = k * torch.rsqrt(k.square().sum(-1, keepdim=True) + 1e-6)
    decay = torch.exp(-torch.exp(w[p + "A_log"].double())
                      * torch.nn.functional.softplus(a + w[p + "dt_bias"].double()))
    beta = torch.sigmoid(b)
    s = q.new_zeros(LH, LD, LD) if rec is None else rec[0].double()
    core = torch.empty_like(q)
    for i in range(t):
        s = s * decay[i, :, None, None]
        d = (v[i] - torch.einsum("hkv,hk->hv", s, k[i])) * beta[i, :, None]
        s = s + k[i][:, :, None] * d[:, None, :]
        core[i] = torch.einsum("hkv,hk->hv", s, q[i])
    core = core * torch.rsqrt(core.square().mean(-1, keepdim=True) + 1e-6) * w[p + "norm.weight"].double() * _silu(z)
    return _linear(core.reshape(t, HID), w[p + "out_proj.weight"], int8), s[None], rows[-4:].t()[None]


def _rope64(x, positions):
    """x [T, heads, HD], the first 64 dims rotated."""
    inv = 1e7 ** (-torch.arange(0, 64, 2, device=DEV, dtype=torch.float64) / 64)
    ang = (positions.double()[:, None] * inv)[:, None, :]
    lo, hi = x[..., :32], x[..., 32:64]
    return torch.cat((lo * ang.cos() - hi * ang.sin(), hi * ang.cos() + lo * ang.sin(), x[..., 64:]), -1)


def _attention64(w, p, x, int8, start=0, keys=None, values=None):
    """x [T, HID] -> (y, all keys [KVH, n, HD], all values)."""
    p = p + "self_attn."
    t = x.shape[0]
    q, gate = _linear(x, w[p + "q_proj.weight"], int8).view(t, QH, 2 * HD).chunk(2, -1)
    k = _linear(x, w[p + "k_proj.weight"], int8).view(t, KVH, HD)
    v = _linear(x, w[p + "v_proj.weight"], int8).view(t, KVH, HD).transpose(0, 1)
    pos = torch.arange(start, start + t, device=DEV)
    q = _rope64(_rms(q, w[p + "q_norm.weight"]), pos)
    k = _rope64(_rms(k, w[p + "k_norm.weight"]), pos).transpose(0, 1)
    if start:
        k = torch.cat((keys.double()[:, :start], k), 1)
        v = torch.cat((values.double()[:, :start], v), 1)
    out = torch.empty_like(q)
    for h in range(QH):
        for a in range(0, t, 2048):  # rows at a time
            n = start + min(a + 2048, t)
            s = q[a : a + 2048, h] @ k[h // (QH // KVH), :n].t() / math.sqrt(HD)
            s.masked_fill_(torch.arange(n, device=DEV)[None] > pos[a : a + 2048, None], -math.inf)
            out[a : a + 2048, h] = torch.softmax(s, -1) @ v[h // (QH // KVH), :n]
    y = (out * torch.sigmoid(gate)).reshape(t, QH * HD)
    return _linear(y, w[p + "o_proj.weight"], int8), k, v


def _filled(rows, into):
    """The cache tensor with the first rows replaced."""
    out = into.double().clone()
    out[0, :, : rows.shape[1]] = rows
    return out


def exact(case, seed):
    weights, inputs = _data(case, seed)
    kind = case["kind"]
    if kind == "head":
        return None  # a token: compared as it is
    if kind == "vision":
        return _vision64(case, weights, inputs)
    int8, p = case["int8"], "model.layers.0."
    if kind == "mlp":
        return {"y": _mlp64(weights, p, inputs["x"][0].double(), int8)[None]}
    if kind == "delta":
        y, s, conv = _delta64(weights, p, inputs["x"][0].double(), int8)
        return {"y": y[None], "state": s, "conv": conv}
    if kind == "attention":
        y, k, v = _attention64(weights, p, inputs["x"][0].double(), int8)
        empty = torch.zeros(1, KVH, cache_bucket(case["tokens"], 64), HD, device=DEV)
        return {"y": y[None], "keys": _filled(k, empty), "values": _filled(v, empty)}
    out = {}
    if kind == "decode":
        residual, update, start = inputs["residual"][0].double(), inputs["update"][0].double(), case["context"]
    else:
        residual = weights["model.embed_tokens.weight"][inputs["ids"][0]].double()
        update, start = torch.zeros_like(residual), 0
    for i, layer in enumerate(_layers(case)):
        p = f"model.layers.{i}."
        residual = residual + update
        x = _rms(residual, weights[p + "input_layernorm.weight"])
        if layer == "full_attention":
            old = [inputs.get(f"{n}{i}") for n in ("keys", "values")]
            y, k, v = _attention64(weights, p, x, int8, start, *(None if o is None else o[0] for o in old))
            if old[0] is None:
                old = [torch.zeros(1, KVH, cache_bucket(case["tokens"], 64), HD, device=DEV)] * 2
            out["keys"], out["values"] = _filled(k, old[0]), _filled(v, old[1])
        else:
            y, s, conv = _delta64(weights, p, x, int8, inputs.get(f"rec{i}"), inputs.get(f"conv{i}"))
            out[f"rec{i}"] = s
            if kind == "decode":
                out[f"conv{i}"] = conv
        residual = residual + y
        update = _mlp64(weights, p, _rms(residual, weights[p + "post_attention_layernorm.weight"]), int8)
    if kind == "decode":
        return {"residual": residual[None], "update": update[None], **out}
    last = _rms((residual + update)[-1:], weights["model.norm.weight"])
    return {"logits": (last @ weights["model.embed_tokens.weight"].double().t())[None], **out}


# ------------------------------------------------------------------ the vision tower in 64 bits
def _vision_inv_freq(cfg):
    half = cfg.hidden_size // cfg.num_heads // 2
    return 10000.0 ** (-torch.arange(0, half, 2, device=DEV, dtype=torch.float64) / half)


def _vision64(case, w, inputs):
    cfg = integration.qwen_impl.Qwen3_5VisionConfig()
    w = {n: t.double() for n, t in w.items()}
    heads, dim = cfg.num_heads, cfg.hidden_size // cfg.num_heads
    h, wd, merge = case["height"], case["width"], cfg.spatial_merge_size
    side = int(cfg.num_position_embeddings**0.5)

    # patches run in blocks of merge x merge
    at = torch.arange(h * wd, device=DEV).view(h // merge, wd // merge, merge, merge)
    flat = torch.empty(h, wd, device=DEV, dtype=torch.long)
    flat.view(h // merge, merge, wd // merge, merge).copy_(at.permute(0, 2, 1, 3))
    order = torch.empty(h * wd, device=DEV, dtype=torch.long)
    order[flat.reshape(-1)] = torch.arange(h * wd, device=DEV)
    row, col = order // wd, order % wd

    def taps(i, n):  # align_corners
        x = i.double() * ((side - 1) / max(n - 1, 1))
        lo = x.floor().clamp(max=side - 1)
        return lo.long(), (lo + 1).clamp(max=side - 1).long(), x - lo

    r0, r1, fr = taps(row, h)
    c0, c1, fc = taps(col, wd)
    table = w["pos_embed.weight"]
    fr, fc = fr[:, None], fc[:, None]
    pos = ((1 - fr) * ((1 - fc) * table[r0 * side + c0] + fc * table[r0 * side + c1])
           + fr * ((1 - fc) * table[r1 * side + c0] + fc * table[r1 * side + c1]))
    inv = _vision_inv_freq(cfg)
    ang = torch.cat((row.double()[:, None] * inv, col.double()[:, None] * inv), -1)
    cos, sin = (torch.cat((f, f), -1)[:, None, :] for f in (ang.cos(), ang.sin()))

    def ln(x, p):
        return torch.nn.functional.layer_norm(x, x.shape[-1:], w[p + "weight"], w[p + "bias"], 1e-6)

    def lin(x, p):
        return x @ w[p + "weight"].t() + w[p + "bias"]

    def rot(x):
        return x * cos + torch.cat((-x[..., dim // 2 :], x[..., : dim // 2]), -1) * sin

    hidden = []
    for pixels in inputs["pixels"].double().view(case["images"], h * wd, -1):
        kernel = w["patch_embed.proj.weight"]
        x = pixels @ kernel.reshape(kernel.shape[0], -1).t() + w["patch_embed.proj.bias"] + pos
        for i in range(cfg.depth):
            p = f"blocks.{i}."
            q, k, v = lin(ln(x, p + "norm1."), p + "attn.qkv.").view(-1, 3, heads, dim).unbind(1)
            q, k, v = (t.transpose(0, 1).contiguous() for t in (rot(q), rot(k), v))
            a = torch.softmax(q @ k.transpose(1, 2).contiguous() / math.sqrt(dim), -1) @ v
            x = x + lin(a.transpose(0, 1).reshape(-1, heads * dim), p + "attn.proj.")
            y = torch.nn.functional.gelu(lin(ln(x, p + "norm2."), p + "mlp.linear_fc1."), approximate="tanh")
            x = x + lin(y, p + "mlp.linear_fc2.")
        hidden.append(x)
    hidden = torch.cat(hidden)
    y = ln(hidden, "merger.norm.").reshape(hidden.shape[0] // merge**2, -1)
    merged = lin(torch.nn.functional.gelu(lin(y, "merger.linear_fc1.")), "merger.linear_fc2.")
    return {"hidden": hidden, "merged": merged}
