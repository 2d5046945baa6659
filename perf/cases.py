"""What this framework's speed is measured on: the work a program has it do, through its public entry points.

Six kinds of case, each over a range of sizes:

* ``linear``       a quantized layer's forward on rows that lie on the GPU: one token, a batch of sequences decoded together, a
                   short prompt, a whole prompt.  W4A16-g128 and W8A16.
* ``quantize``     a dense fp32 weight made into a quantized layer, as a program does for every layer of a model it loads.
* ``attention``    causal attention of a prompt against its cache, fp32 or bf16.
* ``transformer``  a request to the quantized Transformer: prompts through the library's kernels, then greedy tokens.
* ``prompt``       prompts through one of the dense decoders (latent attention; hybrid of attention and selective scans), which leaves
                   the next token's logits and the filled cache.
* ``generate``     a request to one of them: prompts, then greedy tokens.

Models have random weights of the sizes that this repository's benchmarks use, with a head that reads the embedding back (a
trained model is sure of most of its tokens; one whose logits are noise would turn rounding into other tokens).
"""

import math

import torch
import torch.nn.functional as F

DEVICE = "cuda"
VOCAB = 32000
EPS = 1e-5
KEEP = 4          # first positions that stay visible in the hybrid decoder's windows


# ------------------------------------------------------------------ the cases
def listed():
    return [
        # one token through one projection of a 7-billion-parameter model: the smallest call, and the most frequent one
        dict(name="linear_w4_token", kind="linear", scheme="w4a16_g128", rows=1, inputs=4096, outputs=4096),
        # an odd number of sequences decoded together through the widest reduction of such a model
        dict(name="linear_w8_batch", kind="linear", scheme="w8a16", rows=37, inputs=14336, outputs=4096),
        # a short prompt, no multiple of any tile
        dict(name="linear_w4_prompt", kind="linear", scheme="w4a16_g128", rows=500, inputs=4096, outputs=14336),
        # four prompts of 2048 tokens at once
        dict(name="linear_w8_large", kind="linear", scheme="w8a16", rows=8192, inputs=4096, outputs=14336),
        # loading a model: one feed-forward matrix
        dict(name="quantize_w4", kind="quantize", scheme="w4a16_g128", inputs=4096, outputs=14336),
        # the attention of the same prompts, grouped heads, bf16 cache
        dict(name="attention_prompt", kind="attention", batch=4, heads=32, kv_heads=8, seq=2048, start=0, dim=128, cache="bfloat16"),
        # one user's request to the 12-layer int4 model, fp32 cache (the model's own dtype)
        dict(name="transformer_single", kind="transformer", scheme="w4a16_g128", layers=12, width=2048, heads=16, kv_heads=16, ff=5632,
             batch=1, prompt=512, new=65, cache="float32"),
        # a batch of requests to layers of an int8 model with grouped heads, bf16 cache
        dict(name="transformer_batch", kind="transformer", scheme="w8a16", layers=4, width=4096, heads=32, kv_heads=8, ff=14336,
             batch=16, prompt=333, new=33, cache="bfloat16"),
        # prompts of the latent-attention decoder
        dict(name="latent_prompt", kind="prompt", model="latent", width=2048, heads=16, ff=5632, layers=8, looped=4, window=1024, batch=4,
             prompt=2048),
        # a batch of requests to it, wide layers
        dict(name="latent_generate", kind="generate", model="latent", width=4096, heads=32, ff=14336, layers=4, looped=2, window=1024,
             batch=8, prompt=512, new=65),
        # one user's prompt to the hybrid decoder, wide layers
        dict(name="hybrid_prompt", kind="prompt", model="hybrid", width=4096, heads=32, ff=16384, layers=4, looped=2, window=1024, batch=1,
             prompt=1500),
        # a few users' requests to it
        dict(name="hybrid_generate", kind="generate", model="hybrid", width=2048, heads=16, ff=8192, layers=8, looped=4, window=1024,
             batch=4, prompt=700, new=65),
    ]


def _log(rng, low, high):
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def _drawn(rng):
    kind = rng.choice(["linear", "linear", "linear", "quantize", "attention", "transformer", "prompt", "generate"])
    scheme = rng.choice(["w4a16_g128", "w8a16"])
    if kind == "linear":
        return dict(kind=kind, scheme=scheme, rows=_log(rng, 1, 8192), inputs=128 * _log(rng, 8, 112), outputs=8 * _log(rng, 128, 4000))
    if kind == "quantize":
        return dict(kind=kind, scheme=scheme, inputs=128 * _log(rng, 8, 112), outputs=8 * _log(rng, 64, 2048))
    if kind == "attention":
        kv_heads = rng.choice([4, 8, 16])
        return dict(kind=kind, batch=_log(rng, 1, 8), heads=kv_heads * rng.choice([1, 2, 4]), kv_heads=kv_heads, seq=_log(rng, 64, 4096),
                    start=rng.choice([0, 0, rng.randrange(1, 1024)]), dim=rng.choice([128, 128, 64]), cache=rng.choice(["bfloat16", "float32"]))
    if kind == "transformer":
        heads = rng.choice([8, 16, 32])
        return dict(kind=kind, scheme=scheme, layers=rng.randrange(2, 5), width=128 * heads, heads=heads, kv_heads=heads // rng.choice([1, 2, 4]),
                    ff=128 * rng.randrange(2 * heads, 4 * heads), batch=_log(rng, 1, 32), prompt=_log(rng, 16, 1024), new=1 + 8 * rng.randrange(1, 9),
                    cache=rng.choice(["bfloat16", "float32"]))
    heads = rng.choice([8, 16, 32])
    case = dict(kind=kind, model=rng.choice(["latent", "hybrid"]), width=128 * heads, heads=heads, ff=128 * rng.randrange(2 * heads, 4 * heads),
                layers=4, looped=rng.choice([0, 2]), window=rng.choice([512, 1024]))
    if kind == "prompt":
        return dict(case, batch=_log(rng, 1, 4), prompt=_log(rng, 32, 2048))
    return dict(case, batch=_log(rng, 1, 32), prompt=_log(rng, 16, 1024), new=1 + 8 * rng.randrange(1, 9))


def draw(rng):
    def cost(case):
        w = work(case)
        return max(w["bytes"], w["flops"] / 50)

    most = max(cost(c) for c in listed()) / 2
    while True:
        case = _drawn(rng)
        if cost(case) <= most:
            return case


# ------------------------------------------------------------------ weights and inputs
def _generator(seed):
    return torch.Generator(device=DEVICE).manual_seed(seed)


def _randn(gen, *shape, std=1.0):
    return torch.randn(shape, generator=gen, device=DEVICE) * std


def _weight(gen, outputs, inputs):
    return _randn(gen, outputs, inputs, std=math.sqrt(2.0 / (inputs + outputs)))


def _tokens(gen, batch, count):
    return torch.randint(0, VOCAB, (batch, count), generator=gen, device=DEVICE)


def _rows(gen, case):
    """Activations with a few outliers, as a decoder's are."""
    x = _randn(gen, case["rows"], case["inputs"])
    return torch.where(torch.rand(x.shape, generator=gen, device=DEVICE) < 0.001, x * 20.0, x).to(torch.bfloat16)


def _transformer_weights(case, gen):
    d, ff, kv = case["width"], case["ff"], case["width"] // case["heads"] * case["kv_heads"]
    w = {"token_embeddings.weight": _randn(gen, VOCAB, d), "final_norm.weight": 1 + _randn(gen, d, std=0.1)}
    for i in range(case["layers"]):
        p = f"layers.{i}."
        w.update({p + "norm1.weight": 1 + _randn(gen, d, std=0.1), p + "norm2.weight": 1 + _randn(gen, d, std=0.1),
                  p + "attention.q_proj.weight": _weight(gen, d, d), p + "attention.k_proj.weight": _weight(gen, kv, d),
                  p + "attention.v_proj.weight": _weight(gen, kv, d), p + "attention.output_proj.weight": _weight(gen, d, d),
                  p + "feed_forward.w1.weight": _weight(gen, ff, d), p + "feed_forward.w2.weight": _weight(gen, d, ff),
                  p + "feed_forward.w3.weight": _weight(gen, ff, d)})
    w["lm_head.weight"] = w["token_embeddings.weight"].roll(1, 0) * d ** -0.5   # after token t, t + 1
    return w


def _dense_config(case):
    """What a ``config.json`` of the model holds."""
    d, heads = case["width"], case["heads"]
    length = case["prompt"] + case.get("new", 0) + 1
    config = {"vocab": VOCAB, "width": d, "norm": {"eps": EPS}}
    if case["looped"]:
        config["loop"] = {"start": 1, "stop": 1 + case["looped"], "times": 2}
    if case["model"] == "latent":
        mixer = {"heads": heads, "dim": 128, "rot_dim": 64, "vdim": 128, "kv_rank": 512, "scale": 192 ** -0.5, "rot": {"dims": 64, "base": 1e4},
                 "mask": {"size": case["window"]}}
        layer = {"type": "latent_attention", "mixer": mixer, "mlp": {"kind": "dense", "ff": case["ff"]}}
        return dict(config, architecture="Dorutar", max_positions=length, layers=[layer] * case["layers"])
    scan = {"inner": 2 * d, "state": 16, "dt_rank": d // 16, "conv": 4}
    attention = {"heads": heads, "kv_heads": heads // 4, "dim": 128, "scale": 128 ** -0.5, "rot": {"dims": 64, "base": 1e4},
                 "mask": {"size": case["window"], "keep_first": KEEP}}
    kinds = [("attention", attention) if i % 2 else ("mamba1", scan) for i in range(case["layers"])]
    return dict(config, architecture="Purusun", streams=2,
                layers=[{"type": t, "mixer": m, "mlp": {"kind": "dense", "ff": case["ff"]}} for t, m in kinds])


def _dense_weights(case, gen):
    """bf16 parameters by their names in the model."""
    config = _dense_config(case)
    d, ff, heads = case["width"], case["ff"], case["heads"]
    latent = case["model"] == "latent"
    w = {"token_embeddings.weight": _randn(gen, VOCAB, d), "final_norm.weight": _randn(gen, d, std=0.1) + (1 if latent else 0)}
    if latent:
        w["position_embeddings.weight"] = _randn(gen, config["max_positions"], d, std=0.3)
        w["lm_head.weight"] = w["token_embeddings.weight"].roll(1, 0) * d ** -0.5
        if case["looped"]:
            w["loop_step"] = _randn(gen, 2, d, std=0.1)
    for i, layer in enumerate(config["layers"]):
        m = {}
        if latent:
            m = {"q_proj": _weight(gen, heads * 192, d), "dkv_proj": _weight(gen, 576, d), "dkv_norm": 1 + _randn(gen, 512, std=0.1),
                 "uk_proj": _weight(gen, heads * 128, 512), "uv_proj": _weight(gen, heads * 128, 512), "gate_proj": _weight(gen, heads, d),
                 "output_proj": _weight(gen, d, heads * 128)}
            m = {f"mixer.{k}.weight": v for k, v in m.items()} | {"mixer.sink": _randn(gen, heads)}
            m |= {"norm1.weight": 1 + _randn(gen, d, std=0.1), "norm2.weight": 1 + _randn(gen, d, std=0.1),
                  "feed_forward.w1.weight": _weight(gen, ff, d), "feed_forward.w2.weight": _weight(gen, d, ff),
                  "feed_forward.w3.weight": _weight(gen, ff, d)}
        else:
            s = layer["mixer"]
            if layer["type"] == "attention":
                m = {"q_proj.weight": _weight(gen, heads * 128, d), "k_proj.weight": _weight(gen, heads // 4 * 128, d),
                     "q_norm.weight": 1 + _randn(gen, 128, std=0.1), "k_norm.weight": 1 + _randn(gen, 128, std=0.1),
                     "gate_proj.weight": _weight(gen, heads * 128, d), "output_proj.weight": _weight(gen, d, heads * 128)}
            else:
                n, r, inner = s["state"], s["dt_rank"], s["inner"]
                m = {"in_proj.weight": _weight(gen, 2 * inner, d), "conv_weight": _randn(gen, inner, 4, std=0.5), "conv_bias": _randn(gen, inner, std=0.1),
                     "x_proj.weight": _weight(gen, r + 2 * n, inner), "dt_proj.weight": _weight(gen, inner, r),
                     "dt_bias": -4.6 + _randn(gen, inner, std=0.5), "skip": 1 + _randn(gen, inner, std=0.1),
                     "a_log": torch.log(torch.arange(1, n + 1, device=DEVICE)).repeat(inner, 1), "output_proj.weight": _weight(gen, d, inner)}
            m = {"mixer." + k: v for k, v in m.items()}
            m |= {"feed_forward.w1.weight": _weight(gen, ff, d), "feed_forward.w2.weight": _weight(gen, d, ff)}
            for q in "12":
                m |= {f"norm{q}.weight": _randn(gen, d, std=0.1), f"scale{q}": 1 + _randn(gen, d, std=0.1),
                      f"hyper{q}.reads": 0.5 + _randn(gen, 2, std=0.1), f"hyper{q}.writes": 1 + _randn(gen, 2, std=0.1),
                      f"hyper{q}.mix": torch.eye(2, device=DEVICE) + _randn(gen, 2, 2, std=0.1)}
        w.update({f"layers.{i}.{k}": v for k, v in m.items()})
    return {k: v.to(torch.bfloat16) for k, v in w.items()}


# ------------------------------------------------------------------ what a program has in hand, and one pass
def _loaded(model, weights):
    own = dict(model.named_parameters())
    assert own.keys() == weights.keys()
    with torch.no_grad():
        for k, v in weights.items():
            own[k].copy_(v)
    return model.eval()


def prepare(case, seed):
    gen, kind = _generator(seed), case["kind"]
    if kind == "linear":
        from ajllm_amd import QuantLinear
        layer = QuantLinear.from_weight(_randn(gen, case["outputs"], case["inputs"], std=0.02), case["scheme"])
        return kind, layer, _rows(gen, case)
    if kind == "quantize":
        return kind, _randn(gen, case["outputs"], case["inputs"], std=0.02), case["scheme"]
    if kind == "attention":
        return kind, *_attention_inputs(case, gen), case["start"]
    if kind == "transformer":
        from ajllm_amd import decoding, modeling, quantize_model_
        weights, prompt = _transformer_weights(case, gen), _tokens(gen, case["batch"], case["prompt"])
        length = case["prompt"] + case["new"]
        with torch.device(DEVICE):
            model = modeling.TransformerLM(VOCAB, length, case["width"], case["layers"], case["heads"], case["ff"], num_kv_heads=case["kv_heads"])
        model = quantize_model_(_loaded(model, weights), case["scheme"])
        decoder = decoding.FusedDecoder(model, case["batch"], length, getattr(torch, case["cache"]))
        state = kind, decoder, prompt, case["new"]
        run(state)   # a serving program's decoder has recorded its step
        return state
    from ajllm_amd import decoding, modeling
    with torch.device(DEVICE):
        model = modeling.build_model(_dense_config(case)).to(torch.bfloat16)
    _loaded(model, _dense_weights(case, gen)).prepare()
    prompt = _tokens(gen, case["batch"], case["prompt"])
    if kind == "prompt":
        return kind, model, model.new_cache(case["batch"], case["prompt"] + 1), prompt
    state = kind, decoding.DenseDecoder(model, case["batch"], case["prompt"] + case["new"] + 1), prompt, case["new"]
    run(state)
    return state


def run(state):
    kind = state[0]
    if kind == "linear":
        _, layer, x = state
        with torch.no_grad():
            return layer(x)
    if kind == "quantize":
        from ajllm_amd import QuantLinear
        layer = QuantLinear.from_weight(state[1], state[2])
        return {"qweight": layer.qweight, "scales": layer.scales, "zeros": layer.zeros, "wq": layer.wq, "meta": layer.meta}
    if kind == "attention":
        from ajllm_amd.attention import flash_prefill
        _, q, keys, values, start = state
        return flash_prefill(q, keys, values, start, out_dtype=torch.bfloat16)
    if kind == "prompt":
        _, model, cache, prompt = state
        cache.reset()
        logits = model(prompt, cache, last_token_only=True)[:, -1]
        return {"logits": logits, "rings": list(cache.rings), "states": [s for s in cache.states if s is not None]}
    _, decoder, prompt, new = state
    if kind == "transformer":
        decoder.prefill(prompt, fused=True)
        tokens = decoder.generate(new)
        return {"tokens": tokens, "logits": decoder.logits_full[:, :VOCAB]}   # those of the last token
    decoder.prefill(prompt)
    tokens = decoder.generate(new)
    return {"tokens": tokens, "logits": decoder.model(decoder.token, decoder.cache)[:, -1]}   # what would come next


# ------------------------------------------------------------------ what a pass cannot do without
def _linear_bytes(scheme, outputs, inputs):
    return outputs * inputs + 2 * outputs if scheme == "w8a16" else outputs * inputs / 2 + 2.5 * outputs * inputs / 128


def _seen(seq, start=0, window=None, keep=0):
    """Pairs (query, visible key) of ``seq`` new positions."""
    if window is None or start + seq <= window:
        return seq * (start + (seq + 1) / 2)
    return sum(min(start + t + 1, window + keep) for t in range(seq))


def work(case):
    kind = case["kind"]
    if kind == "linear":
        m, k, n = case["rows"], case["inputs"], case["outputs"]
        return {"bytes": _linear_bytes(case["scheme"], n, k) + 2 * m * (n + k), "flops": 2 * m * n * k}
    if kind == "quantize":
        n, k = case["outputs"], case["inputs"]
        stored = n * k + 2 * n if case["scheme"] == "w8a16" else n * k / 2 + 3 * n * k / 128
        packed = n * k + 2 * n if case["scheme"] == "w8a16" else n * k / 2 + 4 * n * k / 128
        return {"bytes": 4 * n * k + stored + packed, "flops": 4 * n * k}
    b, heads = case["batch"], case["heads"]
    if kind == "attention":
        t, total, hd = case["seq"], case["start"] + case["seq"], case["dim"]
        size = 2 if case["cache"] == "bfloat16" else 4
        return {"bytes": b * hd * (heads * t * 6 + 2 * case["kv_heads"] * total * size), "flops": 4 * b * heads * hd * _seen(t, case["start"])}
    d, ff, t, new = case["width"], case["ff"], case["prompt"], case.get("new", 1)
    if kind == "transformer":
        hd = d // heads
        shapes = [(d + 2 * hd * case["kv_heads"], d), (d, d), (2 * ff, d), (d, ff)]
        layer = sum(_linear_bytes(case["scheme"], n, k) for n, k in shapes)
        row = 2 * hd * case["kv_heads"] * (2 if case["cache"] == "bfloat16" else 4)
        per_token = case["layers"] * sum(2 * n * k for n, k in shapes)
        head, seen, length = _linear_bytes(case["scheme"], VOCAB, d), _seen(t), t + new / 2
        return {"bytes": new * (case["layers"] * layer + head) + case["layers"] * b * row * (t + new * length) + 8 * b * t * d,
                "flops": b * (per_token * (t + new) + 4 * d * case["layers"] * (seen + new * length) + 2 * new * VOCAB * d)}
    runs = case["layers"] + case["looped"]
    reach = min(t + new / 2, case["window"])
    if case["model"] == "latent":
        once = d * (heads * 192 + 576 + heads + 2 * ff) + d * (heads * 128 + ff)
        expand, seen = 512 * heads * 256, _seen(t, 0, case["window"])
        prompt = runs * (t * 2 * (once + expand) + 2 * heads * 320 * seen)
        step = runs * (2 * (once + expand) + 2 * heads * 1088 * reach)
        weights, row = runs * 2 * (once + expand), runs * 2 * 576 * reach
    else:
        attends = sum(layer % 2 for layer in _order(case))
        scans = runs - attends
        once = d * (2 * heads * 128 + heads // 4 * 128) + d * heads * 128
        low = d // 16 + 32
        scan = d * 4 * d + 2 * d * low + 2 * d * (d // 16) + 2 * d * d
        seen = _seen(t, 0, case["window"], KEEP)
        every = attends * once + scans * scan + runs * 2 * d * ff
        prompt = 2 * t * every + attends * 4 * heads * 128 * seen + scans * t * 2 * d * 16 * 7
        step = 2 * every + attends * 4 * heads * 128 * reach + scans * 2 * d * 16 * 7
        weights, row = 2 * every, attends * heads // 4 * 512 * reach + scans * 2 * d * (16 * 8 + 6)
    if kind == "prompt":
        return {"bytes": weights + 2 * VOCAB * d + 8 * b * t * d + b * row, "flops": b * (prompt + 2 * VOCAB * d)}
    return {"bytes": new * (weights + 2 * VOCAB * d + b * row) + 8 * b * t * d, "flops": b * (prompt + new * (step + 2 * VOCAB * d))}


def tolerance(case):
    kind = case["kind"]
    if kind == "quantize":
        return "exact"
    if kind in ("linear", "attention"):
        return {"rel": 1e-2, "max": 0.1}
    # whole models: bf16 products one behind the other, through up to 24 sublayers
    return {"rel": 2e-2, "max": 0.5, "differ": 0.005}


# ------------------------------------------------------------------ the same in 64 bits
def _dequantized(weight, scheme):
    """The weight a quantized layer stands for, in 64 bits (the codes are defined by 32-bit arithmetic)."""
    n, k = weight.shape
    if scheme == "w8a16":
        scales = (weight.abs().amax(1) / 127).half()
        d = torch.where(scales == 0, 1.0, scales.float())[:, None]
        return (weight / d).round().clamp(-127, 127).double() * scales.double()[:, None]
    g = weight.view(n, -1, 128)
    low, high = g.amin(2), g.amax(2)
    scales = ((high - low) / 15).half()
    d = torch.where(scales == 0, 1.0, scales.float())
    zeros = (-low / d).round().clamp(0, 15)
    codes = ((g / d[..., None]).round() + zeros[..., None]).clamp(0, 15)
    return ((codes - zeros[..., None]).double() * scales.double()[..., None]).view(n, k)


def _rms(x):
    return x / torch.sqrt(x.square().mean(-1, keepdim=True) + EPS)


def _layer_norm(x, gain):
    return F.layer_norm(x, x.shape[-1:], gain, None, EPS)


def _angles(count, dims, base):
    f = base ** (-torch.arange(0, dims, 2, device=DEVICE, dtype=torch.float64) / dims)
    a = torch.arange(count, device=DEVICE, dtype=torch.float64)[:, None] * f
    return a.cos(), a.sin()


def _halves_rotated(x, dims):
    """Rows ``[B, heads, T, dim]``: component i against i + dims / 2, the rest passes."""
    c, s = _angles(x.shape[-2], dims, 1e4)
    a, b = x[..., : dims // 2], x[..., dims // 2: dims]
    return torch.cat((a * c - b * s, b * c + a * s, x[..., dims:]), -1)


def _pairs_rotated(x):
    c, s = _angles(x.shape[-2], x.shape[-1], 1e4)
    a, b = x[..., ::2], x[..., 1::2]
    return torch.stack((a * c - b * s, a * s + b * c), -1).flatten(-2)


def _attended(q, k, v, scale, window=None, keep=0, sink=None):
    """Causal attention of the last positions, ``[B, H, T, dim]`` with grouped heads, a sequence at a time."""
    t, total = q.shape[2], k.shape[2]
    i, j = torch.arange(total - t, total, device=DEVICE)[:, None], torch.arange(total, device=DEVICE)[None]
    hidden = (j > i) if window is None else (j > i) | ((i - j >= window) & (j >= keep))
    out = []
    for n in range(q.shape[0]):
        kn, vn = (x[n].repeat_interleave(q.shape[1] // k.shape[1], 0) for x in (k, v))
        scores = (q[n] @ kn.transpose(1, 2).contiguous() * scale).masked_fill_(hidden, float("-inf"))
        if sink is not None:
            scores = torch.cat((scores, sink[:, None, None].expand(-1, t, 1)), -1)
        out.append(scores.softmax(-1)[..., :total] @ vn)
    return torch.stack(out)


def _split_heads(x, count):
    return x.unflatten(-1, (count, -1)).transpose(1, 2)


def _joined(x):
    return x.transpose(1, 2).flatten(2)


def _attention_inputs(case, gen):
    b, total, hd, dtype = case["batch"], case["start"] + case["seq"], case["dim"], getattr(torch, case["cache"])
    q = _randn(gen, b, case["heads"], case["seq"], hd)
    return q, *(_randn(gen, b, case["kv_heads"], total, hd).to(dtype) for _ in range(2))


def _transformer_exact(case, w, tokens):
    """Logits ``[B, T, vocab]`` of the last positions, from the first new one on."""
    heads, kv = case["heads"], case["kv_heads"]
    x = w["token_embeddings.weight"][tokens]
    for i in range(case["layers"]):
        p = f"layers.{i}."
        h = _rms(x) * w[p + "norm1.weight"]
        q, k, v = (_split_heads(h @ w[f"{p}attention.{n}_proj.weight"].T, c) for n, c in (("q", heads), ("k", kv), ("v", kv)))
        mixed = _attended(_pairs_rotated(q), _pairs_rotated(k), v, q.shape[-1] ** -0.5)
        x = x + _joined(mixed) @ w[p + "attention.output_proj.weight"].T
        h = _rms(x) * w[p + "norm2.weight"]
        x = x + (F.silu(h @ w[p + "feed_forward.w1.weight"].T) * (h @ w[p + "feed_forward.w3.weight"].T)) @ w[p + "feed_forward.w2.weight"].T
    return (_rms(x[:, case["prompt"] - 1:]) * w["final_norm.weight"]) @ w["lm_head.weight"].T, None


def _order(case):
    inner = list(range(1, 1 + case["looped"]))
    return [0] + 2 * inner + list(range(1 + case["looped"], case["layers"])) if inner else list(range(case["layers"]))


def _ring(rows, capacity, kept=0):
    """The last rows of ``[.., T, width]`` where a ring of that capacity keeps them, and the first ``kept``."""
    t, out = rows.shape[-2], rows.new_zeros(*rows.shape[:-2], capacity, rows.shape[-1])
    if t <= capacity:
        out[..., :t, :] = rows
        return out
    out[..., :kept, :] = rows[..., :kept, :]
    p = torch.arange(t - (capacity - kept), t, device=DEVICE)
    out[..., kept + (p - kept) % (capacity - kept), :] = rows[..., p, :]
    return out


def _latent_exact(case, w, tokens):
    heads, t = case["heads"], tokens.shape[1]
    x = embedded = w["token_embeddings.weight"][tokens] + w["position_embeddings.weight"][:t]
    rings, begun = [], 0
    for i in _order(case):
        if case["looped"] and i == 1:
            x = x + w["loop_step"][begun] + (embedded if begun else 0)
            begun += 1
        m = {k[len(f"layers.{i}."):]: v for k, v in w.items() if k.startswith(f"layers.{i}.")}
        h, g = _layer_norm(x, m["norm1.weight"]), _layer_norm(x, m["norm2.weight"])
        q = _split_heads(h @ m["mixer.q_proj.weight"].T, heads)
        q = torch.cat((q[..., :128], _halves_rotated(q[..., 128:], 64)), -1)
        down = h @ m["mixer.dkv_proj.weight"].T
        latent = _rms(down[..., :512]) * m["mixer.dkv_norm.weight"]
        turned = _halves_rotated(down[:, None, :, 512:], 64)
        rings.append(_ring(torch.cat((latent, turned[:, 0]), -1), min(case["window"], t + 1)))
        k = torch.cat((_split_heads(latent @ m["mixer.uk_proj.weight"].T, heads), turned.expand(-1, heads, -1, -1)), -1)
        v = _split_heads(latent @ m["mixer.uv_proj.weight"].T, heads)
        mixed = _attended(q, k, v, 192 ** -0.5, case["window"], 0, m["mixer.sink"])
        mixed = mixed * torch.sigmoid(h @ m["mixer.gate_proj.weight"].T).transpose(1, 2)[..., None]
        x = x + _joined(mixed) @ m["mixer.output_proj.weight"].T + (
            torch.relu(g @ m["feed_forward.w1.weight"].T) * (g @ m["feed_forward.w3.weight"].T)) @ m["feed_forward.w2.weight"].T
    return _layer_norm(x[:, case["prompt"] - 1:], w["final_norm.weight"]) @ w["lm_head.weight"].T, {"rings": rings, "states": []}


def _scan_exact(h, m):
    """A selective scan's output, its ring and its last state."""
    inner, n, r = m["skip"].shape[0], m["a_log"].shape[1], m["dt_proj.weight"].shape[1]
    both = h @ m["in_proj.weight"].T
    padded = F.pad(both[..., :inner], (0, 0, 3, 0))
    x = F.silu(m["conv_bias"] + sum(padded[:, j: j + h.shape[1]] * m["conv_weight"][:, j] for j in range(4)))
    low = x @ m["x_proj.weight"].T
    dt = F.softplus(low[..., :r] @ m["dt_proj.weight"].T + m["dt_bias"])
    a, state, y = -m["a_log"].exp(), h.new_zeros(h.shape[0], inner, n), torch.empty_like(x)
    for t in range(h.shape[1]):
        state = torch.exp(dt[:, t, :, None] * a) * state + (dt[:, t] * x[:, t])[..., None] * low[:, t, None, r: r + n]
        y[:, t] = (state * low[:, t, None, r + n:]).sum(-1)
    y = (y + m["skip"] * x) * F.silu(both[..., inner:])
    return y @ m["output_proj.weight"].T, _ring(both[..., :inner], 3), state.unflatten(-1, (n // 4, 4)).transpose(1, 2).contiguous()


def _hybrid_exact(case, w, tokens):
    heads, t = case["heads"], tokens.shape[1]
    e = w["token_embeddings.weight"][tokens]
    streams, rings, states = [e, e], [], []

    def sublayer(m, q, body):
        nonlocal streams
        u = sum(m[f"hyper{q}.reads"][s] * streams[s] for s in range(2))
        y = body(_rms(u) * (1 + m[f"norm{q}.weight"])) * m[f"scale{q}"]
        mix = m[f"hyper{q}.mix"]
        streams = [mix[0, s] * streams[0] + mix[1, s] * streams[1] + m[f"hyper{q}.writes"][s] * y for s in range(2)]

    def attention(h, m):
        q = _halves_rotated(_rms(_split_heads(h @ m["q_proj.weight"].T, heads)) * m["q_norm.weight"], 64)
        v = _split_heads(h @ m["k_proj.weight"].T, heads // 4)
        k = _halves_rotated(_rms(v) * m["k_norm.weight"], 64)
        reach = min(case["window"] + KEEP, t + 1)
        rings.append(_ring(torch.cat((v, k), -1), reach, KEEP if reach > KEEP else 0))
        mixed = _joined(_attended(q, k, v, 128 ** -0.5, case["window"], KEEP))
        return (mixed * torch.sigmoid(h @ m["gate_proj.weight"].T)) @ m["output_proj.weight"].T

    def scan(h, m):
        y, ring, state = _scan_exact(h, m)
        rings.append(ring)
        states.append(state)
        return y

    for i in _order(case):
        m = {k[len(f"layers.{i}."):]: v for k, v in w.items() if k.startswith(f"layers.{i}.")}
        mixer = {k[len("mixer."):]: v for k, v in m.items() if k.startswith("mixer.")}
        sublayer(m, 1, lambda h: (attention if i % 2 else scan)(h, mixer))
        sublayer(m, 2, lambda h: torch.relu(h @ m["feed_forward.w1.weight"].T).square() @ m["feed_forward.w2.weight"].T)
    x = (streams[0] + streams[1])[:, case["prompt"] - 1:]
    return (_rms(x) * (1 + w["final_norm.weight"])) @ w["token_embeddings.weight"].T, {"rings": rings, "states": states}


@torch.no_grad()
def exact(case, seed):
    gen, kind = _generator(seed), case["kind"]
    if kind == "linear":
        weight = _dequantized(_randn(gen, case["outputs"], case["inputs"], std=0.02), case["scheme"])
        return _rows(gen, case).double() @ weight.T
    if kind == "quantize":
        w = _randn(gen, case["outputs"], case["inputs"], std=0.02).double()
        if case["scheme"] == "w8a16":
            scales = w.abs().amax(1) / 127
            return {"qweight": None, "scales": scales, "zeros": None, "wq": None, "meta": F.pad(scales, (0, -len(scales) % 16))}
        g = w.view(w.shape[0], -1, 128)
        return {"qweight": None, "scales": (g.amax(2) - g.amin(2)) / 15, "zeros": None, "wq": None, "meta": None}
    if kind == "attention":
        q, keys, values = _attention_inputs(case, gen)
        return _joined(_attended(q.double(), keys.double(), values.double(), case["dim"] ** -0.5))
    if kind == "transformer":
        w = {k: (_dequantized(v, case["scheme"]) if v.dim() == 2 and k != "token_embeddings.weight" else v.double())
             for k, v in _transformer_weights(case, gen).items()}
        model = _transformer_exact
    else:
        w = {k: v.double() for k, v in _dense_weights(case, gen).items()}
        model = _latent_exact if case["model"] == "latent" else _hybrid_exact
    prompt = _tokens(gen, case["batch"], case["prompt"])
    if kind == "prompt":
        logits, cache = model(case, w, prompt)
        return {"logits": logits[:, -1], **cache}
    # the new tokens are guessed, and guessed again from the logits at their places until nothing changes
    new = prompt[:, -1:] + torch.arange(1, case["new"] + 1, device=DEVICE) * int(kind == "transformer" or case["model"] == "latent")
    new = new % VOCAB
    for _ in range(8):
        logits, _ = model(case, w, torch.cat((prompt, new), 1))
        again = logits[:, : case["new"]].argmax(-1)
        if torch.equal(again, new):
            return {"tokens": new, "logits": logits[:, -1 if kind == "generate" else -2]}
        new = again
    return None
