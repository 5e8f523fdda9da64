"""What the framework's speed is measured on: the paths a user of it has it run, through its public entry points.

Kinds of case, and the calls they stand for:

* ``events``   an event recording on the host -> CLIP pixels on the GPU (``ops.event_ops.event_frames_gpu``)
* ``voxel``    events on the GPU -> polarity histograms and voxel grid (``ops.event_ops.voxel_grid_gpu``)
* ``vision``   event frames -> spatio-temporal features (``EventChatModel.encode_event_frames``)
* ``chat``     one EventGPT-7B answer along given tokens: prompt, then one decode step a token (``GenerationEngine.score``),
  with bf16 or 4-bit weights
* ``prompt``   one long EventGPT-7B prompt into the cache (``GenerationEngine.prefill``)
* ``layered_prompt``, ``layered_chat``   the layered decoders (``LayeredEngine.extend``): packs of prompts; prompts followed
  by single tokens of every stream
* ``adapter``  one training step of the attention adapter (loss, backward, optimizer step)
* ``tune``     one instruction-tuning step of EventGPT-7B with low-rank adapters over right-padded samples

Text is given as random tokens and the weights are random at the real sizes: nothing on these paths depends on values,
except which expert of a mixture a token uses and where events fall on the image."""
import math

import numpy as np
import torch

DEV = "cuda:0"
WIDTH, FF, LAYERS, HEADS, VOCAB = 4096, 11008, 32, 32, 32003          # EventGPT-7B's decoder with the event tokens
EPS, THETA = 1e-6, 10000.0
VIT, VIT_FF, VIT_LAYERS, VIT_HEADS, IMAGE, PATCH, VIT_EPS = 1024, 4096, 24, 16, 336, 14, 1e-5
VIT_TOKENS = (IMAGE // PATCH) ** 2 + 1
EVENT_TOKEN, IGNORE = -200, -100
CLIP_MEAN = (0.48145466, 0.4578275, 0.40821073)
CLIP_STD = (0.26862954, 0.26130258, 0.27577711)
ADAPTER_FF, ADAPTER_HEADS, ADAPTER_LR, ADAPTER_DECAY = 2048, 8, 1e-5, 0.01
LORA_RANK, LORA_SCALE = 16, 2.0
LAYERED_VOCAB, LAYERED_PAIRS = 32000, 4
LAYERED = {                                                            # benchmarks/layered_bench.py
    "1b": dict(width=2048, ff=5632, heads=16, kv_heads=4, memory_heads=4, mamba_heads=64, groups=4, q_rank=768, expert_ff=2816),
    "7b": dict(width=4096, ff=11008, heads=32, kv_heads=8, memory_heads=8, mamba_heads=128, groups=8, q_rank=1536, expert_ff=5504),
}


def listed():
    return [
        # the smallest call: a short recording of a small sensor, latency of the upload and of three launches
        dict(name="events_20k", kind="events", events=20000, width=160, height=120, frames=5),
        # 50 ms of a busy 640 x 480 sensor as a voxel grid, binned by time
        dict(name="voxel_10m", kind="voxel", events=10_000_000, width=640, height=480, bins=5, by="time"),
        # the tower as a chat uses it with one event frame: 577 rows through 24 narrow blocks
        dict(name="vision_1", kind="vision", frames=1),
        # the headline: one event frame's prompt of 636 tokens and a short answer, one stream
        dict(name="chat_bf16", kind="chat", prompt=636, new=32, weights="bf16"),
        # the same on 4-bit weights
        dict(name="chat_nf4", kind="chat", prompt=636, new=32, weights="nf4"),
        # eight video frames of 577 tokens and a question: the verifier's prompt, the largest matrix products
        dict(name="prompt_4643", kind="prompt", tokens=4643),
        # a long document through recurrent and chunk-attention layers
        dict(name="nusitar_prompt", kind="layered_prompt", design="nusitar", size="7b", sequences=1, tokens=4096),
        # one interactive stream on the small size: launches and latency count
        dict(name="nusitar_chat", kind="layered_chat", design="nusitar", size="1b", streams=1, prompt=100, new=64),
        # several prompts admitted together, lengths as they come, through latent attention and experts
        dict(name="zapipel_prompt", kind="layered_prompt", design="zapipel", size="7b", sequences=8, tokens=512),
        # a serving batch in the middle of its answers
        dict(name="zapipel_chat_32", kind="layered_chat", design="zapipel", size="1b", streams=32, prompt=200, new=32),
        # one step of adapter training at the trainer's default batch
        dict(name="adapter_64", kind="adapter", batch=64, tokens=50),
        # one micro-batch of low-rank instruction tuning, five event frames a sample
        dict(name="tune_lora_8", kind="tune", samples=8, frames=5, text=255),
    ]


def _log(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["events", "voxel", "vision", "chat", "prompt", "layered_prompt", "layered_chat", "adapter", "tune"])
    c = dict(kind=kind)
    if kind == "events":
        c.update(events=_log(rng, 5000, 500_000), width=rng.randint(120, 640), height=rng.randint(90, 480), frames=rng.randint(1, 8))
    elif kind == "voxel":
        c.update(events=_log(rng, 20_000, 10_000_000), width=rng.randint(120, 640), height=rng.randint(90, 480),
                 bins=rng.randint(1, 10), by=rng.choice(["time", "count"]))
    elif kind == "vision":
        c.update(frames=rng.randint(1, 8))
    elif kind == "chat":
        c.update(prompt=_log(rng, 40, 2100), new=rng.randint(8, 32), weights=rng.choice(["bf16", "nf4"]))
    elif kind == "prompt":
        c.update(tokens=_log(rng, 300, 4643))
    elif kind == "layered_prompt":
        n = _log(rng, 1, 8)
        c.update(design=rng.choice(["nusitar", "zapipel"]), size=rng.choice(["1b", "7b"]), sequences=n, tokens=_log(rng, 64, 4096 // n))
    elif kind == "layered_chat":
        c.update(design=rng.choice(["nusitar", "zapipel"]), size=rng.choice(["1b", "7b"]), streams=_log(rng, 1, 32),
                 prompt=rng.randint(33, 256), new=rng.randint(16, 48))
    elif kind == "adapter":
        c.update(batch=_log(rng, 4, 64), tokens=rng.randint(9, 64))
    else:
        c.update(samples=_log(rng, 1, 8), frames=rng.choice([1, 5]), text=rng.randint(80, 255))
    return c


# ------------------------------------------------------------------------------------------------------- random inputs
def _gen(seed, device=DEV):
    return torch.Generator(device=device).manual_seed(int(seed) * 7919 + 17)


def _normal(g, *shape, std=1.0, dtype=torch.bfloat16):
    return torch.empty(shape, device=g.device, dtype=dtype).normal_(0.0, std, generator=g)


def _near_one(g, *shape, dtype=torch.bfloat16):
    return torch.empty(shape, device=g.device, dtype=dtype).normal_(1.0, 0.1, generator=g)


def _ints(g, lo, hi, *shape, dtype=torch.int64):
    return torch.randint(lo, hi, shape, generator=g, device=g.device, dtype=dtype)


def _decoder_weights(g, layers=LAYERS):
    """Checkpoint names -> tensors of the decoder.  Matrices are scaled by fan-in and what a sublayer adds to the residual
    stream is a fraction of it, as in a trained model: rounding is then not amplified from layer to layer."""
    w = {"model.embed_tokens.weight": _normal(g, VOCAB, WIDTH), "lm_head.weight": _normal(g, VOCAB, WIDTH, std=WIDTH ** -0.5),
         "model.norm.weight": _near_one(g, WIDTH)}
    for i in range(layers):
        p = f"model.layers.{i}."
        for n in ("q", "k", "v", "o"):
            w[p + f"self_attn.{n}_proj.weight"] = _normal(g, WIDTH, WIDTH, std=WIDTH ** -0.5)
        w[p + "mlp.gate_proj.weight"] = _normal(g, FF, WIDTH, std=WIDTH ** -0.5)
        w[p + "mlp.up_proj.weight"] = _normal(g, FF, WIDTH, std=WIDTH ** -0.5)
        w[p + "mlp.down_proj.weight"] = _normal(g, WIDTH, FF, std=0.5 * FF ** -0.5)
        w[p + "input_layernorm.weight"] = _near_one(g, WIDTH)
        w[p + "post_attention_layernorm.weight"] = _near_one(g, WIDTH)
    return w


def _vision_weights(g):
    v = "model.visual_tower.visual_tower.vision_model."
    w = {v + "embeddings.class_embedding": _normal(g, VIT, std=0.02),
         v + "embeddings.patch_embedding.weight": _normal(g, VIT, 3, PATCH, PATCH, std=0.02),
         v + "embeddings.position_embedding.weight": _normal(g, VIT_TOKENS, VIT, std=0.02)}

    def norm(n):
        w[n + ".weight"], w[n + ".bias"] = _near_one(g, VIT), _normal(g, VIT, std=0.02)

    def lin(n, a, b):
        w[n + ".weight"], w[n + ".bias"] = _normal(g, a, b, std=0.02), _normal(g, a, std=0.02)
    norm(v + "pre_layrnorm")
    norm(v + "post_layernorm")
    for i in range(VIT_LAYERS):
        p = v + f"encoder.layers.{i}."
        for n in ("q", "k", "v", "out"):
            lin(p + f"self_attn.{n}_proj", VIT, VIT)
        lin(p + "mlp.fc1", VIT_FF, VIT)
        lin(p + "mlp.fc2", VIT, VIT_FF)
        norm(p + "layer_norm1")
        norm(p + "layer_norm2")
    lin("model.visual_projector.0", WIDTH, VIT)
    lin("model.visual_projector.2", WIDTH, WIDTH)
    lin("model.feature_adaptor", WIDTH, WIDTH)
    return w


def _events(case, seed):
    """Events of a few moving edges over uniform noise, sorted by time; host arrays."""
    g = _gen(seed, DEV)
    n, w, h = case["events"], case["width"], case["height"]
    t = torch.sort(_ints(g, 0, 50_000, n)).values
    c = torch.rand(8, 2, device=DEV, generator=g) * torch.tensor([w, h], device=DEV)
    edge = torch.rand(n, device=DEV, generator=g) < 0.8
    at = c[_ints(g, 0, 8, n)] + torch.randn(n, 2, device=DEV, generator=g) * torch.tensor([w / 50.0, h / 12.0], device=DEV)
    noise = torch.rand(n, 2, device=DEV, generator=g) * torch.tensor([w, h], device=DEV)
    at = torch.where(edge[:, None], at, noise)
    x, y = at[:, 0].clamp(0, w - 1).to(torch.int32), at[:, 1].clamp(0, h - 1).to(torch.int32)
    x[0], y[0] = w - 1, h - 1                              # the sensor's extent is seen
    return {"x": x, "y": y, "t": t, "p": _ints(g, 0, 2, n, dtype=torch.int32)}


def _layered_config(case):
    s = LAYERED[case["size"]]
    layers = []
    if case["design"] == "nusitar":
        rec = {"heads": s["memory_heads"], "dim": 256, "vdim": 512, "gate_cap": 15.0}
        att = {"heads": s["heads"], "kv_heads": s["kv_heads"], "dim": 128, "vdim": 128, "scale": 128 ** -0.5,
               "rot": {"dims": 128, "base": 10000.0}, "mask": {"size": 2048}}
        mam = {"heads": s["mamba_heads"], "groups": s["groups"], "state": 128, "vdim": 64, "conv": 4, "norm_groups": s["groups"]}
        for _ in range(LAYERED_PAIRS):
            layers.append({"type": "mamba2", "mlp": None, "mixer": mam})
            layers.append({"type": "parallel", "mixer": {"left": att, "right": rec}, "mlp": {"kind": "dense", "ff": s["ff"]}})
        return {"architecture": "Nusitar", "vocab": LAYERED_VOCAB, "width": s["width"], "norm": {"eps": EPS},
                "embedding": {"scale": 1.0}, "layers": layers}
    mix = {"heads": s["heads"], "dim": 128, "vdim": 128, "kv_rank": 512, "q_rank": s["q_rank"], "scale": 128 ** -0.5}
    for i in range(LAYERED_PAIRS):
        layers.append({"type": "latent_attention", "mixer": mix, "mlp": {"kind": "dense", "ff": s["ff"]}})
        layers.append({"type": "latent_attention", "mixer": {**mix, "kv_from": 2 * i},
                       "mlp": {"kind": "moe", "expert": {"ff": s["expert_ff"]}, "router": {"experts": 8, "top": 2}}})
    return {"architecture": "Zapipel", "vocab": LAYERED_VOCAB, "width": s["width"], "norm": {"eps": EPS}, "logit_scale": 1.0,
            "logit_softcap": 30.0, "layers": layers}


def _layered_weights(cfg, g):
    d, w = cfg["width"], {}

    def mat(n, rows, cols):
        w[n] = _normal(g, rows, cols, std=cols ** -0.5)

    def one(n, size):
        w[n] = _near_one(g, size)
    mat("embed", cfg["vocab"], d)
    if cfg["architecture"] == "Zapipel":
        # what a token is about decides its experts: a first and a second topic in its embedding, a router row a topic
        topics = _normal(g, 8, d)
        first, step = _ints(g, 0, 8, cfg["vocab"]), _ints(g, 1, 8, cfg["vocab"])
        w["embed"] = _normal(g, cfg["vocab"], d) + 0.5 * topics[first] + 0.25 * topics[(first + step) % 8]
    mat("head", cfg["vocab"], d)
    one("final.norm", d)
    for i, layer in enumerate(cfg["layers"]):
        p, m, mlp = f"l{i}.", layer["mixer"], layer["mlp"]
        zap = cfg["architecture"] == "Zapipel"
        for n in ("norm1",) + (("norm1b",) if zap else ()) + (() if mlp is None else ("norm2",) + (("norm2b",) if zap else ())):
            one(p + n, d)
        q = p + "mix."
        if layer["type"] == "mamba2":
            h, inner, ch = m["heads"], m["heads"] * m["vdim"], m["heads"] * m["vdim"] + 2 * m["groups"] * m["state"]
            mat(q + "in", inner + ch + h, d)
            mat(q + "conv", ch, m["conv"])
            w[q + "conv.b"], w[q + "dt_bias"] = _normal(g, ch), _normal(g, h) - 2
            w[q + "A_log"] = _normal(g, h, std=0.5)
            one(q + "D", h)
            one(q + "norm", inner)
            mat(q + "o", d, inner)
        elif layer["type"] == "parallel":
            a, r = m["left"], m["right"]
            hq, hk, hv = a["heads"] * a["dim"], a["kv_heads"] * a["dim"], a["kv_heads"] * a["vdim"]
            for n, rows in (("q", hq), ("k", hk), ("v", hv)):
                mat(q + "left." + n, rows, d)
            one(q + "left.q.norm", hq)
            one(q + "left.k.norm", hk)
            mat(q + "left.o", d, a["heads"] * a["vdim"])
            qk, v, h = r["heads"] * r["dim"], r["heads"] * r["vdim"], r["heads"]
            for n, rows in (("q", qk), ("k", qk), ("v", v), ("g", v), ("i", h), ("f", h)):
                mat(q + "right." + n, rows, d)
            mat(q + "right.o", d, v)
            one(q + "right.norm", v)
            w[q + "right.i.b"], w[q + "right.f.b"] = _normal(g, h) - 3, _normal(g, h) + 3
            one(q + "left.out", d)
            one(q + "right.out", d)
        else:
            h = m["heads"]
            mat(q + "dq", m["q_rank"], d)
            one(q + "dq.norm", m["q_rank"])
            mat(q + "uq", h * m["dim"], m["q_rank"])
            mat(q + "uk", h * m["dim"], m["kv_rank"])
            mat(q + "uv", h * m["vdim"], m["kv_rank"])
            mat(q + "g", h, d)
            mat(q + "o", d, h * m["vdim"])
            if m.get("kv_from") is None:
                mat(q + "dkv", m["kv_rank"], d)
                one(q + "dkv.norm", m["kv_rank"])
        if mlp is None:
            continue
        units = [(p + "mlp.", mlp["ff"])] if mlp["kind"] == "dense" else \
            [(f"{p}mlp.e{e}.", mlp["expert"]["ff"]) for e in range(mlp["router"]["experts"])]
        for u, ff in units:
            mat(u + "gate", ff, d)
            mat(u + "up", ff, d)
            mat(u + "down", d, ff)
        if mlp["kind"] == "moe":
            w[p + "mlp.router"] = topics * d ** -0.5
            w[p + "mlp.router.b"] = _normal(g, mlp["router"]["experts"], std=0.1)
    return w


def _lengths(case):
    """Prompt lengths of a pack: spread by a third around the named one; the total is the same for every seed."""
    n, t = case["sequences"], case["tokens"]
    return [max(1, t + (2 * i - n + 1) * t // (3 * n)) for i in range(n)]


def _layered_inputs(case, seed):
    """``(config, weights, prompts, [new, streams] tokens or None)``."""
    cfg, g = _layered_config(case), _gen(seed)
    w = _layered_weights(cfg, g)
    if case["kind"] == "layered_prompt":
        return cfg, w, [_ints(g, 0, LAYERED_VOCAB, n, dtype=torch.int32) for n in _lengths(case)], None
    prompts = [_ints(g, 0, LAYERED_VOCAB, case["prompt"], dtype=torch.int32) for _ in range(case["streams"])]
    return cfg, w, prompts, _ints(g, 0, LAYERED_VOCAB, case["new"], case["streams"], dtype=torch.int32)


def _adapter_inputs(case, seed):
    g, d, f32 = _gen(seed), WIDTH, torch.float32
    w, p = {"alpha": torch.tensor(0.1, device=DEV)}, "layers.0."
    for n in (p + "attn_norm", p + "ffn_norm", "output_proj.0"):
        w[n + ".weight"], w[n + ".bias"] = _near_one(g, d, dtype=f32), _normal(g, d, std=0.02, dtype=f32)
    for n, a, b in ((p + "attn.in_proj_", 3 * d, d), (p + "attn.out_proj.", d, d), (p + "ffn.0.", ADAPTER_FF, d),
                    (p + "ffn.3.", d, ADAPTER_FF), ("output_proj.1.", d, d)):
        w[n + "weight"], w[n + "bias"] = _normal(g, a, b, std=b ** -0.5, dtype=f32), _normal(g, a, std=0.02, dtype=f32)
    b, s = case["batch"], case["tokens"]
    src = _normal(g, b, s, d, dtype=f32)
    lens = torch.clamp(s - _ints(g, 0, max(1, s // 3), b), min=1)
    mask = (torch.arange(s, device=DEV)[None] < lens[:, None]).to(f32)
    return w, src, src + 0.3 * _normal(g, b, s, d, dtype=f32), mask


def _tune_inputs(case, seed):
    g = _gen(seed)
    w = {**_decoder_weights(g), **_vision_weights(g)}
    lora = {}
    for i in range(LAYERS):
        for n in ("q", "k", "v", "o"):
            p = f"model.layers.{i}.self_attn.{n}_proj."
            lora[p + "lora_A.weight"] = _normal(g, LORA_RANK, WIDTH, std=WIDTH ** -0.5)
            lora[p + "lora_B.weight"] = _normal(g, WIDTH, LORA_RANK, std=0.01)
    n, text = case["samples"], case["text"]
    ids = _ints(g, 3, VOCAB, n, text).cpu()
    mask = torch.ones(n, text, dtype=torch.long)
    labels = torch.full((n, text), IGNORE)
    for i in range(n):
        k = text - (i * text) // (4 * n)                   # answers of different lengths, right-padded
        ids[i, 35], ids[i, k:], mask[i, k:] = EVENT_TOKEN, 0, 0
        labels[i, 60:k] = ids[i, 60:k]                     # prompt of 60 tokens, answer after it
    frames = _normal(g, n, case["frames"], 3, IMAGE, IMAGE)
    return w, lora, ids, mask, labels, frames


# ------------------------------------------------------------------------------------------------------------- prepare
def _event_model(weights, layers, vision):
    from eventgpt_amd.models import ClipVisionConfig, EventChatConfig, EventChatModel
    cfg = EventChatConfig.eventgpt_7b(vocab_size=VOCAB)
    cfg.num_hidden_layers = layers
    if not vision:                                         # text paths: the tower is not used
        cfg.vision_config = ClipVisionConfig(hidden_size=64, intermediate_size=128, num_hidden_layers=1, num_attention_heads=1,
                                             image_size=28, patch_size=14)
    model = EventChatModel.from_config(cfg, torch.bfloat16, torch.device(DEV), seed=None)
    own = model.state_dict()
    with torch.no_grad():
        for n, t in weights.items():
            own[n].copy_(t)
    return model


def _chat_inputs(case, seed):
    g = _gen(seed)
    w = _decoder_weights(g)
    rows = case["prompt"] if case["kind"] == "chat" else case["tokens"]
    embeds = _normal(g, rows, WIDTH)
    tokens = _ints(g, 3, VOCAB, case["new"]).cpu() if case["kind"] == "chat" else None
    return w, embeds, tokens


def prepare(case, seed):
    kind = case["kind"]
    if kind == "events":
        return dict(case=case, events={k: v.cpu().numpy() for k, v in _events(case, seed).items()})
    if kind == "voxel":
        return dict(case=case, events=_events(case, seed))
    if kind == "vision":
        g = _gen(seed)
        weights = _vision_weights(g)
        frames = [_normal(g, 3, IMAGE, IMAGE) for _ in range(case["frames"])]
        model = _event_model(weights, 1, True)
        with torch.no_grad():
            model.encode_event_frames(frames)              # a server's first call: the tower is captured
        return dict(case=case, model=model, frames=frames)
    if kind in ("chat", "prompt"):
        weights, embeds, tokens = _chat_inputs(case, seed)
        model = _event_model(weights, LAYERS, False)
        del weights
        kw = dict(weight_format=case["weights"]) if kind == "chat" else {}
        engine = model.engine(max_len=embeds.shape[0] + 64, max_new_tokens=64, **kw)
        if kind == "chat":
            engine.ensure_graphs(-1, greedy=False)
        return dict(case=case, engine=engine, embeds=embeds, tokens=tokens)
    if kind in ("layered_prompt", "layered_chat"):
        from eventgpt_amd.models import LayeredConfig, LayeredDecoder
        cfg, weights, prompts, tokens = _layered_inputs(case, seed)
        model = LayeredDecoder(LayeredConfig(cfg), torch.bfloat16, DEV)
        for n, t in weights.items():
            model.tensors[n].copy_(t)
        del weights
        longest = max(p.numel() for p in prompts)
        engine = model.engine(max_len=longest + 64, max_batch=len(prompts))
        if tokens is not None:
            engine.ensure_graphs(-1, greedy=False)
        return dict(case=case, engine=engine, prompts=prompts, tokens=tokens)
    if kind == "adapter":
        from eventgpt_amd.align.adapters import create_adapter
        from eventgpt_amd.parallel.dp import ShardedAdamW
        weights, src, tgt, mask = _adapter_inputs(case, seed)
        model = create_adapter(4, WIDTH, num_heads=ADAPTER_HEADS, ffn_dim=ADAPTER_FF, dropout=0.0).to(DEV).train()
        with torch.no_grad():
            for n, p in model.named_parameters():
                p.copy_(weights[n])
        return dict(case=case, model=model, opt=ShardedAdamW(model.parameters(), lr=ADAPTER_LR, weight_decay=ADAPTER_DECAY),
                    src=src, tgt=tgt, mask=mask)
    from eventgpt_amd.cli.train_sft import select_trainable
    from eventgpt_amd.ops.differentiable import enable_transposed_dgrad
    weights, lora, ids, mask, labels, frames = _tune_inputs(case, seed)
    model = _event_model(weights, LAYERS, True)
    del weights
    params = select_trainable(model, "lora", lora_rank=LORA_RANK, lora_alpha=int(LORA_RANK * LORA_SCALE), lora_dropout=0.0)
    named = dict(model.named_parameters())
    with torch.no_grad():
        for n, t in lora.items():
            named[n].copy_(t)
    enable_transposed_dgrad(model.get_model().layers)
    from eventgpt_amd.parallel.dp import ShardedAdamW
    model.train()
    return dict(case=case, model=model, opt=ShardedAdamW(params, lr=1e-6, weight_decay=0.0, overlap=False),
                named={n: p for n, p in model.named_parameters() if p.requires_grad}, ids=ids, mask=mask, labels=labels,
                frames=[list(f) for f in frames])


# ----------------------------------------------------------------------------------------------------------------- run
TUNED_BRIDGE = ("model.visual_projector.0.weight", "model.visual_projector.0.bias", "model.visual_projector.2.weight",
                "model.visual_projector.2.bias", "model.feature_adaptor.weight", "model.feature_adaptor.bias")


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "events":
        from eventgpt_amd.ops.event_ops import event_frames_gpu
        size, pixels = event_frames_gpu(state["events"], DEV, case["frames"])
        return [size, pixels]
    if kind == "voxel":
        from eventgpt_amd.ops.event_ops import voxel_grid_gpu
        return list(voxel_grid_gpu(state["events"], case["bins"], (case["height"], case["width"]), by=case["by"]))
    if kind == "vision":
        with torch.no_grad():
            return state["model"].encode_event_frames(state["frames"])
    if kind == "chat":
        return state["engine"].score(state["embeds"], state["tokens"])
    if kind == "prompt":
        e = state["engine"]
        e.reset()
        hidden = e.prefill(state["embeds"], select="logits", return_hidden=True)
        return [hidden, e.logits[0].clone()]
    if kind in ("layered_prompt", "layered_chat"):
        e, prompts = state["engine"], state["prompts"]
        slots = list(range(len(prompts)))
        e.reset()
        out = [e.extend(slots, prompts, [[p.numel() - 1] for p in prompts])]
        if state["tokens"] is not None:
            want = [[0]] * len(slots)
            for row in state["tokens"]:
                out.append(e.extend(slots, list(row.split(1)), want))
        return torch.stack(out)
    if kind == "adapter":
        from eventgpt_amd.ops.intree_mode import InTreeLinear
        model, opt = state["model"], state["opt"]
        opt.zero_grad()
        with torch.autocast("cuda", dtype=torch.bfloat16), InTreeLinear():
            loss = model.compute_loss(state["src"], state["tgt"], state["mask"])["total_loss"]
        loss.backward()
        opt.step(max_grad_norm=1.0)
        p = dict(model.named_parameters())
        return {"loss": loss.detach(), "grad": {n: t.grad for n, t in p.items()}, "weight": {n: t.detach() for n, t in p.items()}}
    model, opt, named = state["model"], state["opt"], state["named"]
    opt.zero_grad()
    ids, mask, labels = (state[k].to(DEV) for k in ("ids", "mask", "labels"))
    loss = model(input_ids=ids, attention_mask=mask, labels=labels, event_tensors=state["frames"],
                 loss_reduction="sequence_mean").loss
    loss.backward()
    opt.step(max_grad_norm=1.0)
    out = {n: named[n].grad for n in TUNED_BRIDGE}
    for k in ("lora_A", "lora_B"):
        out[k] = torch.stack([p.grad for n, p in named.items() if k in n])
    out["loss"] = loss.detach()
    return out


# ---------------------------------------------------------------------------------------------------------------- work
def _layer_matrices(cfg, streams):
    """``(values of matrices a pass over `streams` rows has to read, values one token is multiplied by)`` of all layers."""
    read = used = 0
    d = cfg["width"]
    for layer in cfg["layers"]:
        m, mlp, n = layer["mixer"], layer["mlp"], 0
        if layer["type"] == "mamba2":
            inner = m["heads"] * m["vdim"]
            n += d * (3 * inner + 2 * m["groups"] * m["state"] + m["heads"])
        elif layer["type"] == "parallel":
            a, r = m["left"], m["right"]
            n += d * (2 * a["heads"] * a["dim"] + 2 * a["kv_heads"] * a["dim"])
            n += d * (2 * r["heads"] * r["dim"] + 3 * r["heads"] * r["vdim"] + 2 * r["heads"])
        else:
            h = m["heads"]
            n += d * (m["q_rank"] + h + h * m["vdim"]) + h * m["dim"] * m["q_rank"] + h * (m["dim"] + m["vdim"]) * m["kv_rank"]
            n += 0 if m.get("kv_from") is not None else d * m["kv_rank"]
        read, used = read + n, used + n
        if mlp is not None and mlp["kind"] == "dense":
            read, used = read + 3 * d * mlp["ff"], used + 3 * d * mlp["ff"]
        elif mlp is not None:
            e, top, ff = mlp["router"]["experts"], mlp["router"]["top"], mlp["expert"]["ff"]
            hit = e * (1 - (1 - top / e) ** streams)       # experts that some row of the pass uses
            read, used = read + 3 * d * ff * hit, used + 3 * d * ff * top
    return read, used


def _layered_attention(cfg, n):
    """Multiplications of token mixing over a prompt of ``n``, all layers (chunk-masked, latent or linear)."""
    total = 0
    for layer in cfg["layers"]:
        m = layer["mixer"]
        if layer["type"] == "mamba2":
            total += n * m["heads"] * m["vdim"] * m["state"] * 2
        elif layer["type"] == "parallel":
            a, r, c = m["left"], m["right"], m["left"]["mask"]["size"]
            total += sum(min(c, n - s) ** 2 / 2 for s in range(0, n, c)) * a["heads"] * (a["dim"] + a["vdim"])
            total += n * r["heads"] * r["dim"] * r["vdim"] * 2
        else:
            total += n * n / 2 * m["heads"] * (m["dim"] + m["vdim"])
    return total


VISION_VALUES = VIT_LAYERS * (4 * VIT * VIT + 2 * VIT * VIT_FF) + 3 * PATCH * PATCH * VIT
BRIDGE_VALUES = WIDTH * VIT + 2 * WIDTH * WIDTH
LAYER_VALUES = 4 * WIDTH * WIDTH + 3 * WIDTH * FF


def _vision_flops(frames):
    rows = frames * VIT_TOKENS
    return 2 * rows * VISION_VALUES + frames * VIT_LAYERS * 4 * VIT_TOKENS ** 2 * VIT


def _causal(n):
    """Operations of causal attention of the 7B decoder over ``n`` tokens, all layers."""
    return LAYERS * 4 * WIDTH * n * (n + 1) / 2


def work(case):
    kind = case["kind"]
    if kind == "events":
        pixels = 3 * IMAGE * IMAGE * case["frames"]
        return {"bytes": 20 * case["events"] + 2 * pixels, "flops": 2 * 8 * pixels}
    if kind == "voxel":
        return {"bytes": 20 * case["events"] + 12 * case["bins"] * case["width"] * case["height"], "flops": 0}
    if kind == "vision":
        t = case["frames"]
        return {"bytes": 2 * (VISION_VALUES + BRIDGE_VALUES + t * 3 * IMAGE * IMAGE + (t + VIT_TOKENS) * WIDTH),
                "flops": _vision_flops(t) + 2 * t * VIT_TOKENS * BRIDGE_VALUES}
    if kind == "chat":
        p, n = case["prompt"], case["new"]
        per = (LAYERS * LAYER_VALUES * (2 if case["weights"] == "bf16" else 0.5625)) + 2 * VOCAB * WIDTH
        first = 2 * LAYERS * LAYER_VALUES if case["weights"] == "nf4" else per
        cache = sum(p + i + 1 for i in range(n)) * LAYERS * 4 * WIDTH
        return {"bytes": first + n * per + cache + 4 * (n + 1) * VOCAB,
                "flops": 2 * (p + n) * LAYERS * LAYER_VALUES + 2 * (n + 1) * VOCAB * WIDTH + _causal(p + n)}
    if kind == "prompt":
        n = case["tokens"]
        return {"bytes": 2 * (LAYERS * LAYER_VALUES + VOCAB * WIDTH) + n * (LAYERS * 4 * WIDTH + 4 * WIDTH) + 4 * VOCAB,
                "flops": 2 * n * LAYERS * LAYER_VALUES + 2 * VOCAB * WIDTH + _causal(n)}
    if kind in ("layered_prompt", "layered_chat"):
        cfg = _layered_config(case)
        head = LAYERED_VOCAB * cfg["width"]
        lens = _lengths(case) if kind == "layered_prompt" else [case["prompt"]] * case["streams"]
        read, used = _layer_matrices(cfg, sum(lens))
        w = {"bytes": 2 * (read + head) + 4 * LAYERED_VOCAB * len(lens),
             "flops": 2 * sum(lens) * used + 2 * len(lens) * head + 2 * sum(_layered_attention(cfg, n) for n in lens)}
        if kind == "layered_chat":
            read, used = _layer_matrices(cfg, case["streams"])
            w["bytes"] += case["new"] * (2 * (read + head) + 4 * LAYERED_VOCAB * case["streams"])
            w["flops"] += case["new"] * case["streams"] * 2 * (used + head)
        return w
    if kind == "adapter":
        values = 5 * WIDTH * WIDTH + 2 * WIDTH * ADAPTER_FF
        rows = case["batch"] * case["tokens"]
        # weights and both moments read and written, gradients written and read, source and target read
        return {"bytes": 32 * values + 8 * rows * WIDTH, "flops": 6 * rows * values}
    n, t = case["samples"], case["frames"]
    rows = sum(case["text"] - (i * case["text"]) // (4 * n) - 1 + t + VIT_TOKENS for i in range(n))
    low = LAYERS * 8 * LORA_RANK * WIDTH
    answer = sum(case["text"] - (i * case["text"]) // (4 * n) - 60 for i in range(n))
    per = rows / n
    flops = rows * (4 * LAYERS * LAYER_VALUES + 6 * low) + n * 3.5 * _causal(per) + 4 * answer * VOCAB * WIDTH
    flops += _vision_flops(n * t) + 6 * n * t * VIT_TOKENS * BRIDGE_VALUES
    return {"bytes": 2 * (2 * LAYERS * LAYER_VALUES + 2 * VOCAB * WIDTH + VISION_VALUES) + 30 * (low + BRIDGE_VALUES), "flops": flops}


def tolerance(case):
    """bf16 rounding after every product and norm of up to 32 layers; measured against ``exact``: pixels 0.0017, 0.007 to 0.013
    for the towers, decoders and the adapter's gradients."""
    return {"events": {"rel": 0.007}, "voxel": "exact"}.get(case["kind"], {"rel": 0.03})


# --------------------------------------------------------------------------------------------------------------- exact
def _rms(x, w, eps=EPS):
    return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + eps) * w


def _ln(x, w, b=0.0, eps=EPS):
    x = x - x.mean(-1, keepdim=True)
    return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + eps) * w + b


def _silu(z):
    return z * torch.sigmoid(z)


def _rotate(x, base=THETA, pos0=0):
    """Rotate-half positions of ``x [T, H, D]``."""
    half = x.shape[-1] // 2
    f = base ** (-torch.arange(half, device=x.device, dtype=torch.float64) / half)
    a = (pos0 + torch.arange(x.shape[0], device=x.device, dtype=torch.float64))[:, None] * f
    c, s = a.cos()[:, None], a.sin()[:, None]
    u, v = x[..., :half], x[..., half:]
    return torch.cat([u * c - v * s, v * c + u * s], -1)


def _attend(q, k, v, scale, causal=True, chunk=None):
    """``q [T, H, D]``, ``k, v [T, G, D]``; positions see earlier ones (of their chunk)."""
    t, h, per = q.shape[0], q.shape[1], q.shape[1] // k.shape[1]
    i = torch.arange(t, device=q.device)
    hide = None
    if causal:
        hide = i[None] > i[:, None]
        if chunk is not None:
            hide = hide | (i[None] // chunk != i[:, None] // chunk)
    out = []
    for j in range(h):
        s = q[:, j] @ k[:, j // per].T * scale
        if hide is not None:
            s = s.masked_fill(hide, -math.inf)
        out.append(torch.softmax(s, -1) @ v[:, j // per])
    return torch.stack(out, 1)


def _decode_layer(x, w, lens, lora=None):
    """One decoder layer in 64 bits over rows ``x`` of sequences of ``lens`` rows; ``w(name)`` gives a weight."""
    h = _rms(x, w("input_layernorm.weight"))

    def proj(n, y):
        out = y @ w(f"self_attn.{n}_proj.weight").T
        if lora is not None:
            a, b = lora(n)
            out = out + LORA_SCALE * (y @ a.T) @ b.T
        return out
    q, k, v = (proj(n, h).view(-1, HEADS, WIDTH // HEADS) for n in ("q", "k", "v"))
    o, at = [], 0
    for n in lens:
        s = slice(at, at + n)
        o.append(_attend(_rotate(q[s]), _rotate(k[s]), v[s], (WIDTH // HEADS) ** -0.5))
        at += n
    x = x + proj("o", torch.cat(o).reshape(-1, WIDTH))
    h = _rms(x, w("post_attention_layernorm.weight"))
    return x + (_silu(h @ w("mlp.gate_proj.weight").T) * (h @ w("mlp.up_proj.weight").T)) @ w("mlp.down_proj.weight").T


NF4 = (-1.0, -0.6961928009986877, -0.5250730514526367, -0.39491748809814453, -0.28444138169288635, -0.18477343022823334,
       -0.09105003625154495, 0.0, 0.07958029955625534, 0.16093020141124725, 0.24611230194568634, 0.33791524171829224,
       0.44070982933044434, 0.5626170039176941, 0.7229568362236023, 1.0)        # Dettmers et al. 2023, appendix E


def _nf4(w):
    """The 4-bit image of a matrix: blocks of 64 scaled to their largest value, nearest of 16 bf16 levels."""
    levels = torch.tensor(NF4, device=w.device).to(torch.bfloat16).float()
    out = []
    for part in w.split(2048):
        b = part.float().reshape(part.shape[0], -1, 64)
        top = b.abs().amax(-1, keepdim=True)
        out.append((levels[((b / top)[..., None] - levels).abs().argmin(-1)].double() * top.double()).reshape(part.shape))
    return torch.cat(out)


def _exact_chat(case, seed):
    w, embeds, tokens = _chat_inputs(case, seed)
    x = embeds.double()
    if tokens is not None:
        x = torch.cat([x, w["model.embed_tokens.weight"][tokens.to(DEV)].double()])
    four = case.get("weights") == "nf4"
    for i in range(LAYERS):
        def layer(n, p=f"model.layers.{i}."):
            t = w[p + n]
            return _nf4(t) if four and t.dim() == 2 else t.double()
        x = _decode_layer(x, layer, [x.shape[0]])
    last = x[embeds.shape[0] - 1:]
    logits = _rms(last, w["model.norm.weight"].double()) @ w["lm_head.weight"].double().T
    return logits if tokens is not None else [x, logits[0]]


def _exact_tower(w, frames):
    """Tower output ``[T, 577, 1024]`` of ``frames [T, 3, S, S]``."""
    v = "model.visual_tower.visual_tower.vision_model."
    t, side = frames.shape[0], IMAGE // PATCH
    x = frames.double().reshape(t, 3, side, PATCH, side, PATCH).permute(0, 2, 4, 1, 3, 5).reshape(t, side * side, -1)
    x = x @ w[v + "embeddings.patch_embedding.weight"].double().reshape(VIT, -1).T
    x = torch.cat([w[v + "embeddings.class_embedding"].double().expand(t, 1, VIT), x], 1)
    x = x + w[v + "embeddings.position_embedding.weight"].double()

    def norm(n, y):
        return _ln(y, w[n + ".weight"].double(), w[n + ".bias"].double(), VIT_EPS)

    def lin(n, y):
        return y @ w[n + ".weight"].double().T + w[n + ".bias"].double()
    x = norm(v + "pre_layrnorm", x)
    for i in range(VIT_LAYERS):
        p = v + f"encoder.layers.{i}."
        h = norm(p + "layer_norm1", x)
        q, k, y = (lin(p + f"self_attn.{n}_proj", h).view(t, VIT_TOKENS, VIT_HEADS, -1) for n in ("q", "k", "v"))
        o = torch.stack([_attend(q[j], k[j], y[j], (VIT // VIT_HEADS) ** -0.5, causal=False) for j in range(t)])
        x = x + lin(p + "self_attn.out_proj", o.reshape(t, VIT_TOKENS, VIT))
        h = lin(p + "mlp.fc1", norm(p + "layer_norm2", x))
        x = x + lin(p + "mlp.fc2", h * torch.sigmoid(1.702 * h))
    return x


def _exact_bridge(w, tower):
    """Projector, adaptor and pooling of one sample's frames: ``[T + 577, 4096]``."""
    f = tower @ w["model.visual_projector.0.weight"].T + w["model.visual_projector.0.bias"]
    f = 0.5 * f * (1 + torch.erf(f / math.sqrt(2)))
    f = f @ w["model.visual_projector.2.weight"].T + w["model.visual_projector.2.bias"]
    f = f @ w["model.feature_adaptor.weight"].T + w["model.feature_adaptor.bias"]
    return torch.cat([f.mean(1), f.mean(0)])


def _gelu_tanh(z):
    return 0.5 * z * (1 + torch.tanh(math.sqrt(2 / math.pi) * (z + 0.044715 * z ** 3)))


def _exact_mamba(h, w, m):
    """Mamba-2 in its quadratic form: ``y_t = sum_s decay(s, t) dt_s (C_t . B_s) x_s + D x_t``."""
    t, hd, vd, n, gr = h.shape[0], m["heads"], m["vdim"], m["state"], m["groups"]
    inner = hd * vd
    z, xbc, dt = (h @ w("in").T).split([inner, inner + 2 * gr * n, hd], -1)
    taps = m["conv"]
    padded = torch.cat([xbc.new_zeros(taps - 1, xbc.shape[1]), xbc])
    xbc = _silu(w("conv.b") + sum(padded[j:j + t] * w("conv")[:, j] for j in range(taps)))
    x, b, c = xbc.split([inner, gr * n, gr * n], -1)
    x, b, c = x.view(t, hd, vd), b.view(t, gr, n), c.view(t, gr, n)
    dt = torch.nn.functional.softplus(dt + w("dt_bias"))
    cum = torch.cumsum(-torch.exp(w("A_log")) * dt, 0)
    seen = torch.tril(torch.ones(t, t, device=h.device, dtype=torch.bool))
    y = []
    for j in range(hd):
        g = j // (hd // gr)
        decay = (cum[:, j, None] - cum[None, :, j]).masked_fill(~seen, -math.inf).exp()
        y.append((decay * (c[:, g] @ b[:, g].T) * dt[None, :, j]) @ x[:, j] + w("D")[j] * x[:, j])
    y = torch.stack(y, 1).reshape(t, inner) * _silu(z)
    y = _rms(y.view(t, m["norm_groups"], -1), 1.0).reshape(t, inner) * w("norm")
    return y @ w("o").T


def _exact_parallel(h, w, m):
    a, r, t = m["left"], m["right"], h.shape[0]
    q = _rms(h @ w("left.q").T, w("left.q.norm")).view(t, a["heads"], -1)
    k = _rms(h @ w("left.k").T, w("left.k.norm")).view(t, a["kv_heads"], -1)
    v = (h @ w("left.v").T).view(t, a["kv_heads"], -1)
    left = _attend(_rotate(q), _rotate(k), v, a["scale"], True, a["mask"]["size"]).reshape(t, -1) @ w("left.o").T
    hd, n, vd, cap = r["heads"], r["dim"], r["vdim"], r["gate_cap"]
    q = (h @ w("right.q").T).view(t, hd, n) * n ** -0.5
    k, v = (h @ w("right.k").T).view(t, hd, n), (h @ w("right.v").T).view(t, hd, vd)
    gi = cap * torch.tanh((h @ w("right.i").T + w("right.i.b")) / cap)
    gf = torch.nn.functional.logsigmoid(cap * torch.tanh((h @ w("right.f").T + w("right.f.b")) / cap))
    cum = torch.cumsum(gf, 0)
    seen = torch.tril(torch.ones(t, t, device=h.device, dtype=torch.bool))
    out = []
    for j in range(hd):
        d = (cum[:, j, None] - cum[None, :, j] + gi[None, :, j]).masked_fill(~seen, -math.inf)
        top = torch.maximum(d.amax(1), cum[:, j])              # the running maximum starts from zero
        p = (d - top[:, None]).exp() * (q[:, j] @ k[:, j].T)
        out.append(p @ v[:, j] / (torch.maximum(p.sum(1).abs(), torch.exp(-top)) + 1e-6)[:, None])
    o = _rms(torch.stack(out, 1), 1.0).reshape(t, hd * vd) * w("right.norm") * torch.sigmoid(h @ w("right.g").T)
    return 0.5 * (_rms(left, w("left.out")) + _rms(o @ w("right.o").T, w("right.out")))


def _exact_latent(h, c, w, m):
    t, hd = h.shape[0], m["heads"]
    q = (_rms(h @ w("dq").T, w("dq.norm")) @ w("uq").T).view(t, hd, -1)
    o = _attend(q, (c @ w("uk").T).view(t, hd, -1), (c @ w("uv").T).view(t, hd, -1), m["scale"])
    return (o * torch.sigmoid(h @ w("g").T)[:, :, None]).reshape(t, -1) @ w("o").T


def _exact_mlp(h, w, mlp, act):
    if mlp["kind"] == "dense":
        return (act(h @ w("gate").T) * (h @ w("up").T)) @ w("down").T
    best, which = (h @ w("router").T + w("router.b")).topk(mlp["router"]["top"], -1)
    share, out = torch.softmax(best, -1), torch.zeros_like(h)
    for e in range(mlp["router"]["experts"]):
        rows, slot = (which == e).nonzero(as_tuple=True)
        y = (act(h[rows] @ w(f"e{e}.gate").T) * (h[rows] @ w(f"e{e}.up").T)) @ w(f"e{e}.down").T
        out.index_add_(0, rows, y * share[rows, slot, None])
    return out


def _exact_layered(cfg, weights, tokens):
    """Final residual rows, normed, of one sequence."""
    x, latents, zap = weights["embed"][tokens.long()].double(), {}, cfg["architecture"] == "Zapipel"
    norm = _ln if zap else _rms
    for i, layer in enumerate(cfg["layers"]):
        def w(n, p=f"l{i}."):
            return weights[p + n].double()

        def after(n, y):
            return norm(y, w(n)) if zap else y
        h, m = norm(x, w("norm1")), layer["mixer"]

        def mix(n):
            return w("mix." + n)
        if layer["type"] == "latent_attention":
            src = m.get("kv_from")
            if src is None:
                src, latents[i] = i, _rms(h @ mix("dkv").T, mix("dkv.norm"))
            y = _exact_latent(h, latents[src], mix, m)
        else:
            y = (_exact_mamba if layer["type"] == "mamba2" else _exact_parallel)(h, mix, m)
        x = x + after("norm1b", y)
        if layer["mlp"] is not None:
            y = _exact_mlp(norm(x, w("norm2")), lambda n: w("mlp." + n), layer["mlp"], _silu if zap else _gelu_tanh)
            x = x + after("norm2b", y)
    return norm(x, weights["final.norm"].double())


def _exact_layered_case(case, seed):
    cfg, weights, prompts, tokens = _layered_inputs(case, seed)
    out = []
    for b, p in enumerate(prompts):
        t = p if tokens is None else torch.cat([p, tokens[:, b]])
        out.append(_exact_layered(cfg, weights, t)[p.numel() - 1:] @ weights["head"].double().T)
    out = torch.stack(out, 1)                                  # [1 + new, streams, vocab]
    if cfg["architecture"] == "Zapipel":
        cap = cfg["logit_softcap"]
        out = cap * torch.tanh(out * cfg["logit_scale"] / cap)
    return out


def _clipped_adamw(w, grads, lr, decay):
    """Weights after the first AdamW step on gradients clipped to norm one."""
    clip = min(1.0, 1.0 / (math.sqrt(sum(float(g.square().sum()) for g in grads.values())) + 1e-6))
    return {n: t * (1 - lr * decay) - lr * (grads[n] * clip) / ((grads[n] * clip).abs() + 1e-8) for n, t in w.items()}


def _exact_adapter(case, seed):
    w, src, tgt, mask = _adapter_inputs(case, seed)
    w = {n: t.double().requires_grad_() for n, t in w.items()}
    src, tgt, mask, p = src.double(), tgt.double(), mask.double(), "layers.0."
    b, s, d = src.shape
    h = _ln(src, w[p + "attn_norm.weight"], w[p + "attn_norm.bias"], 1e-5)
    qkv = (h @ w[p + "attn.in_proj_weight"].T + w[p + "attn.in_proj_bias"]).view(b, s, 3, ADAPTER_HEADS, -1).permute(2, 0, 3, 1, 4)
    score = (qkv[0] @ qkv[1].transpose(-1, -2)) * (d // ADAPTER_HEADS) ** -0.5
    score = score.masked_fill(mask[:, None, None] == 0, -math.inf)
    o = (torch.softmax(score, -1) @ qkv[2]).transpose(1, 2).reshape(b, s, d)
    x = src + o @ w[p + "attn.out_proj.weight"].T + w[p + "attn.out_proj.bias"]
    h = _ln(x, w[p + "ffn_norm.weight"], w[p + "ffn_norm.bias"], 1e-5) @ w[p + "ffn.0.weight"].T + w[p + "ffn.0.bias"]
    h = 0.5 * h * (1 + torch.erf(h / math.sqrt(2)))
    x = x + h @ w[p + "ffn.3.weight"].T + w[p + "ffn.3.bias"]
    y = _ln(x, w["output_proj.0.weight"], w["output_proj.0.bias"], 1e-5) @ w["output_proj.1.weight"].T + w["output_proj.1.bias"]
    y = src + w["alpha"] * (y - src)
    cos = (y * tgt).sum(-1) / (y.norm(dim=-1) * tgt.norm(dim=-1))
    loss = ((y - tgt).square().sum(-1) * mask).sum() / (mask.sum() * d) + 0.5 * (1 - (cos * mask).sum() / mask.sum())
    loss.backward()
    grads = {n: t.grad for n, t in w.items()}
    with torch.no_grad():
        return {"loss": loss.detach(), "grad": grads, "weight": _clipped_adamw({n: t.detach() for n, t in w.items()}, grads,
                                                                                ADAPTER_LR, ADAPTER_DECAY)}


def _exact_tune(case, seed):
    from torch.utils.checkpoint import checkpoint
    w, lora, ids, mask, labels, frames = _tune_inputs(case, seed)
    bridge = {n: w[n].double().requires_grad_() for n in TUNED_BRIDGE}
    low = {n: t.double().requires_grad_() for n, t in lora.items()}
    rows, lens, targets = [], [], []
    for i in range(case["samples"]):
        with torch.no_grad():
            tower = _exact_tower(w, frames[i])
        f = _exact_bridge(bridge, tower)
        k = int(mask[i].sum())
        emb = w["model.embed_tokens.weight"][ids[i, :k].clamp(min=0).to(DEV)].double()
        rows.append(torch.cat([emb[:35], f, emb[36:]]))
        lens.append(rows[-1].shape[0])
        targets.append(torch.cat([labels[i, :35], torch.full((f.shape[0],), IGNORE), labels[i, 36:k]]))
    x = torch.cat(rows)
    for i in range(LAYERS):
        p = f"model.layers.{i}."

        def layer(y, p=p):
            return _decode_layer(y, lambda n: w[p + n].double(), lens,
                                 lambda n: (low[p + f"self_attn.{n}_proj.lora_A.weight"], low[p + f"self_attn.{n}_proj.lora_B.weight"]))
        x = checkpoint(layer, x, use_reentrant=False)
    x, head, loss, at = _rms(x, w["model.norm.weight"].double()), w["lm_head.weight"].double(), 0.0, 0
    for n, t in zip(lens, targets):
        pick = (t[1:] != IGNORE).nonzero()[:, 0]
        loss = loss + torch.nn.functional.cross_entropy(x[at + pick.to(DEV)] @ head.T, t[1:][pick].to(DEV)) / len(lens)
        at += n
    loss.backward()
    out = {n: bridge[n].grad for n in TUNED_BRIDGE}
    for k in ("lora_A", "lora_B"):
        out[k] = torch.stack([low[f"model.layers.{i}.self_attn.{n}_proj.{k}.weight"].grad for i in range(LAYERS) for n in ("q", "k", "v", "o")])
    out["loss"] = loss.detach()
    return out


def _exact_events(case, seed):
    """Rasters by the last event of every pixel, then an antialiased bicubic resize in 64 bits."""
    ev = {k: v.cpu().numpy() for k, v in _events(case, seed).items()}
    h, w, n, t = int(ev["y"].max()) + 1, int(ev["x"].max()) + 1, case["events"], case["frames"]
    pixels = []
    for i in range(t):
        img = np.full((h, w, 3), 255.0)
        lo, hi = i * (n // t), n if i == t - 1 else (i + 1) * (n // t)
        last = np.full(h * w, -1)
        np.maximum.at(last, ev["y"][lo:hi].astype(np.int64) * w + ev["x"][lo:hi], np.arange(lo, hi))
        hit = (last >= 0).nonzero()[0]
        on = ev["p"][last[hit]] != 0
        img.reshape(-1, 3)[hit] = np.where(on[:, None], [[255.0, 0.0, 0.0]], [[0.0, 0.0, 255.0]])
        pixels.append(torch.from_numpy(img).permute(2, 0, 1))
    short, long = min(h, w), max(h, w)
    other = int(IMAGE * long / short)
    size = (IMAGE, other) if h <= w else (other, IMAGE)
    x = torch.stack(pixels)
    x = torch.nn.functional.interpolate(x, (h, size[1]), mode="bicubic", antialias=True).round().clamp(0, 255)
    x = torch.nn.functional.interpolate(x, size, mode="bicubic", antialias=True).round().clamp(0, 255)
    top, left = (size[0] - IMAGE) // 2, (size[1] - IMAGE) // 2
    x = x[:, :, top:top + IMAGE, left:left + IMAGE] / 255
    mean, std = (torch.tensor(v, dtype=torch.float64).view(3, 1, 1) for v in (CLIP_MEAN, CLIP_STD))
    return [[h, w], (x - mean) / std]


def _exact_voxel(case, seed):
    ev = _events(case, seed)
    n, bins, h, w = case["events"], case["bins"], case["height"], case["width"]
    if case["by"] == "time":
        t = ev["t"].double()
        t0 = t.min()
        b = ((t - t0) / (t.max() - t0).clamp(min=1) * bins).long().clamp(0, bins - 1)
    else:
        b = torch.arange(n, device=DEV) * bins // n
    at = ((b * 2 + (ev["p"] != 0)) * h + ev["y"]) * w + ev["x"]
    hist = torch.bincount(at, minlength=bins * 2 * h * w).view(bins, 2, h, w)
    return [hist.int(), (hist[:, 1] - hist[:, 0]).double()]


def exact(case, seed):
    kind = case["kind"]
    if kind == "tune":
        return _exact_tune(case, seed)
    if kind == "adapter":
        return _exact_adapter(case, seed)
    with torch.no_grad():
        if kind == "events":
            return _exact_events(case, seed)
        if kind == "voxel":
            return _exact_voxel(case, seed)
        if kind == "vision":
            g = _gen(seed)
            w = _vision_weights(g)
            frames = torch.stack([_normal(g, 3, IMAGE, IMAGE) for _ in range(case["frames"])])
            return _exact_bridge({n: t.double() for n, t in w.items()}, _exact_tower(w, frames))
        if kind in ("chat", "prompt"):
            return _exact_chat(case, seed)
        return _exact_layered_case(case, seed)
