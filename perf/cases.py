"""The measured work of this package: twelve calls of its public entry points, the ranges they stand for, their inputs, the bytes
and operations none of them can do without, and what they return in 64-bit arithmetic.

    encode      frames -> visual tokens for the language model: VisionEncoder.encode_project (27-layer ViT of width 1152, projector
                to 3584), bf16. One image, a short clip, a clip that fills the token budget.
    preprocess  decoded uint8 frames -> pixel_values of the encoder: preprocess_videos_gpu.
    kmeans      a clip's visual tokens -> events: kmeans_with_time_min_max.
    prompt      Qwen2-7B, the prompt of one answer into an empty cache: Qwen2Engine.forward.
    token       Qwen2-7B, one generated token behind a prompt: embedding and Qwen2Engine.forward.
    latent / latent_token   Pabalix: a prompt; one token of every live sequence of a batch.
    delta / delta_trace     Lupanex: a prompt; requests of different lengths stepped as a batch from their prompts on.

Weights are random at the models' real sizes; the models of the last two lines have the sizes of bench.py."""
from __future__ import annotations

import math
import random

import torch

from cogstream_amd import kmeans, lupanex, pabalix
from cogstream_amd.llm import DecoderEngine, Qwen2Engine, Sequences
from cogstream_amd.preprocess_gpu import preprocess_videos_gpu
from cogstream_amd.vision import Projector, VisionEncoder
from cogstream_amd.weights import (LlmConfig, VisionConfig, random_decoder_state, random_llm_state, random_proj_state,
                                   random_vit_state)

BF16, F64 = torch.bfloat16, torch.float64
VIT, QWEN = VisionConfig(), LlmConfig()
VOCAB = 32768
# width: heads, query rank, feed-forward, layers; head parts 128 + 64 rotated, values 128, latents of 512
LATENT = {2048: (16, 768, 5632, 9), 3584: (28, 1536, 18944, 6), 4096: (32, 1536, 11008, 6)}
# width: heads, feed-forward, layers; heads of 128, every fourth layer attention, four residual streams
DELTA = {2048: (16, 8192, 8), 3584: (28, 28416, 4), 4096: (32, 16384, 8)}
FRAMES = ((360, 640), (480, 854), (720, 1280))


# ------------------------------------------------------------------------------------------------ the cases
def listed():
    return [
        # one still image of 224 x 224: the smallest request, bound by its launches
        {"name": "image_224", "kind": "encode", "frames": 1, "gh": 16, "gw": 16, "merge": 1},
        # a short clip, 8 frames of 224 x 224
        {"name": "clip_8x224", "kind": "encode", "frames": 8, "gh": 16, "gw": 16, "merge": 2},
        # 64 frames of 480p: the clip that fills the budget of 16 384 visual tokens; the headline throughput
        {"name": "clip_64x480p", "kind": "encode", "frames": 64, "gh": 22, "gw": 42, "merge": 2},
        # the same clip from decoded bytes
        {"name": "preprocess_64x480p", "kind": "preprocess", "frames": 64, "height": 480, "width": 854},
        # events of a 256-frame clip, 50 tokens a frame
        {"name": "events_256", "kind": "kmeans", "frames": 256, "tokens": 50},
        # the prompt of the short clip, a question about 8 small frames
        {"name": "prompt_621", "kind": "prompt", "rows": 621},
        # the prompt of the 64-frame clip: the longest a request has
        {"name": "prompt_15395", "kind": "prompt", "rows": 15395},
        # one answer token behind that prompt
        {"name": "token_15395", "kind": "token", "context": 15395},
        # a small decoder: one long prompt
        {"name": "latent_4096", "kind": "latent", "width": 2048, "rows": 4096},
        # serving it: sixteen live requests, contexts from 256 to 4096 tokens
        {"name": "latent_token_16", "kind": "latent_token", "width": 2048, "requests": 16, "context": 4096},
        # the recurrent decoder: one long prompt
        {"name": "delta_4096", "kind": "delta", "width": 2048, "rows": 4096},
        # serving it: eight requests with prompts of 64 to 512 tokens, then 24 tokens of each
        {"name": "delta_trace_8", "kind": "delta_trace", "width": 2048, "requests": 8, "prompt": 512, "steps": 24},
    ]


def _spread(rng, lo, hi):
    """whole numbers, even over the logarithm"""
    return min(hi, max(lo, round(math.exp(rng.uniform(math.log(lo), math.log(hi))))))


def draw(rng):
    kind = rng.choice(("encode", "encode", "preprocess", "kmeans", "prompt", "token", "latent", "latent_token", "delta", "delta_trace"))
    if kind == "encode":
        merge = rng.choice((1, 2, 2))
        gh, gw = merge * rng.randint(12 // merge, 44 // merge), merge * rng.randint(12 // merge, 44 // merge)
        most = min(64, 59136 // (gh * gw)) if merge == 2 else min(4, 16384 // (gh * gw))
        return {"kind": kind, "frames": _spread(rng, 1, most), "gh": gh, "gw": gw, "merge": merge}
    if kind == "preprocess":
        h, w = rng.choice(FRAMES)
        return {"kind": kind, "frames": _spread(rng, 1, 64), "height": h, "width": w}
    if kind == "kmeans":
        return {"kind": kind, "frames": rng.randint(136, 400), "tokens": rng.randint(24, 64)}
    if kind == "prompt":
        return {"kind": kind, "rows": _spread(rng, 40, 15395)}
    if kind == "token":
        return {"kind": kind, "context": _spread(rng, 40, 15395)}
    width = rng.choice((2048, 2048, 3584, 4096))
    if kind in ("latent", "delta"):
        return {"kind": kind, "width": width, "rows": _spread(rng, 100, 4096)}
    if kind == "latent_token":
        return {"kind": kind, "width": width, "requests": _spread(rng, 1, 32), "context": _spread(rng, 100, 4096)}
    return {"kind": kind, "width": width, "requests": _spread(rng, 1, 16), "prompt": _spread(rng, 24, 512), "steps": rng.randint(4, 24)}


# ------------------------------------------------------------------------------------------------ sizes and configurations
def _contexts(case):
    """cached tokens of every live request, from a sixteenth of the longest up"""
    n, most = case["requests"], case["context"]
    return [max(1, most * (i + 1) // n) for i in range(n)]


def _prompts(case):
    n, most = case["requests"], case["prompt"]
    return [max(1, most * (i + 1) // n) for i in range(n)]


def _latent_config(width):
    heads, q_rank, ff, layers = LATENT[width]
    kinds = ("latent_attention_3", "latent_attention", "latent_attention_2")
    out = []
    for i in range(layers):
        rot = dict(base=10000.0, dims=64)
        if kinds[i % 3] != "latent_attention_2":
            rot["scaling"] = dict(factor=4.0, original=4096, fast=32.0, slow=1.0)
        mix = dict(heads=heads, dim=128, rot_dim=64, vdim=128, q_rank=q_rank, kv_rank=512, scale=192 ** -0.5, rot=rot)
        if i % 6 == 5:
            mix["kv_from"] = i - 3
        out.append(dict(type=kinds[i % 3], mixer=mix, mlp=dict(kind="dense", ff=ff)))
    return dict(architecture="Pabalix", layers=out, norm=dict(eps=1e-6), vocab=VOCAB, width=width)


def _delta_config(width):
    heads, ff, layers = DELTA[width]
    out = []
    for i in range(layers):
        if i % 4 == 3:
            mix = dict(heads=heads, kv_heads=heads // 4, dim=128, vdim=128, scale=128 ** -0.5, bias_max=128, q_temp=dict(coef=0.1, every=2048))
        else:
            mix = dict(heads=heads, kv_heads=heads // 2, dim=128, vdim=128, conv=4)
        out.append(dict(type="attention" if i % 4 == 3 else "delta", mixer=mix, mlp=dict(kind="dense", ff=ff)))
    return dict(architecture="Lupanex", layers=out, norm=dict(eps=1e-6), vocab=VOCAB, width=width, streams=4,
                embedding=dict(scale=1.0), max_positions=4352)


def _decoder(case):
    """-> (config.json, the package's description)"""
    if case["kind"].startswith("latent"):
        c = _latent_config(case["width"])
        return c, pabalix.parse_config(c)
    c = _delta_config(case["width"])
    shapes = {f"l{i}.mix.rel": (32, lay["mixer"]["heads"]) for i, lay in enumerate(c["layers"]) if lay["type"] == "attention"}
    return c, lupanex.parse_config(c, shapes)


# ------------------------------------------------------------------------------------------------ inputs
def _generator(seed):
    return torch.Generator(device="cuda").manual_seed(seed * 1000003 + 17)


def _pixels(case, seed):
    n = case["frames"] * case["gh"] * case["gw"]
    b = torch.randint(0, 256, (n, VIT.patch_dim), generator=_generator(seed), device="cuda", dtype=torch.int16)
    return (b / 127.5 - 1).to(BF16)


def _bytes(case, seed):
    """frames of soft shapes under sensor noise"""
    g, t, h, w = _generator(seed), case["frames"], case["height"], case["width"]
    coarse = torch.rand(t, 3, 9, 16, generator=g, device="cuda") * 255
    out = torch.empty(t, h, w, 3, device="cuda", dtype=torch.uint8)
    for i in range(t):
        f = torch.nn.functional.interpolate(coarse[i:i + 1], size=(h, w), mode="bilinear")[0].permute(1, 2, 0)
        out[i] = (f + 12 * torch.randn(h, w, 3, generator=g, device="cuda")).clamp(0, 255).to(torch.uint8)
    return out


def _features(case, seed):
    """frames of some twenty scenes, each drifting along a direction of its own"""
    g, t, p = _generator(seed), case["frames"], case["tokens"]
    scenes = max(2, t // 12)
    centre = torch.randn(scenes, p, 3584, generator=g, device="cuda")
    drift = torch.randn(scenes, p, 3584, generator=g, device="cuda")
    at = torch.arange(t, device="cuda") * scenes // t
    return (centre[at] + 0.5 * torch.rand(t, 1, 1, generator=g, device="cuda") * drift[at]
            + 0.1 * torch.randn(t, p, 3584, generator=g, device="cuda")).to(BF16)


def _qwen_state(seed):
    return random_llm_state(QWEN, seed=seed + 2, device="cuda", dtype=BF16)


def _decoder_state(dc, seed):
    return random_decoder_state(dc, seed=seed + 3, device="cuda", dtype=BF16)


def _ids(n, vocab, seed):
    return torch.randint(0, vocab, (n,), generator=torch.Generator().manual_seed(seed + 5))


def _cached(shape, g):
    """rows that a prompt would have left: keys, values and normed latents are of deviation one"""
    return torch.randn(shape, generator=g, device="cuda").to(BF16)


def prepare(case, seed):
    kind = case["kind"]
    if kind == "encode":
        enc = VisionEncoder(random_vit_state(VIT, seed=seed, device="cuda", dtype=BF16), VIT)
        proj = Projector(random_proj_state(VIT.hidden_size, QWEN.hidden_size, seed=seed + 1, device="cuda", dtype=BF16))
        grid = torch.tensor([[case["frames"], case["gh"], case["gw"]]])
        return {"kind": kind, "encoder": enc, "projector": proj, "pixels": _pixels(case, seed), "grid": grid,
                "merge": torch.tensor([case["merge"]])}
    if kind == "preprocess":
        return {"kind": kind, "frames": _bytes(case, seed)}
    if kind == "kmeans":
        return {"kind": kind, "features": _features(case, seed), "clusters": -(-case["frames"] // 15), "seed": seed,
                "times": torch.arange(case["frames"], dtype=torch.float32)}
    if kind in ("prompt", "token"):
        engine = Qwen2Engine(_qwen_state(seed), QWEN)
        if kind == "prompt":
            return {"kind": kind, "engine": engine, "embeds": engine.embed_tokens(_ids(case["rows"], 150000, seed)),
                    "cache": engine.new_cache(case["rows"])}
        cache = engine.new_cache(case["context"] + 1)
        g = _generator(seed)
        for i in range(QWEN.num_hidden_layers):
            cache.k[i], cache.v[i] = _cached(cache.k.shape[1:], g), _cached(cache.v.shape[1:], g)
        return {"kind": kind, "engine": engine, "token": _ids(1, 150000, seed).cuda(), "cache": cache, "context": case["context"]}
    _, dc = _decoder(case)
    engine = DecoderEngine(_decoder_state(dc, seed), dc)
    if kind in ("latent", "delta"):
        return {"kind": kind, "engine": engine, "embeds": engine.embed_tokens(_ids(case["rows"], VOCAB, seed)),
                "cache": engine.new_cache(case["rows"])}
    if kind == "latent_token":
        g, caches = _generator(seed), []
        for n in _contexts(case):
            caches.append(engine.new_cache(n + 1))
            caches[-1].k.copy_(_cached(caches[-1].k.shape, g))
        return {"kind": kind, "engine": engine, "tokens": _ids(case["requests"], VOCAB, seed).cuda(), "caches": caches,
                "contexts": _contexts(case)}
    steps = [_ids(n + case["steps"], VOCAB, seed + 31 * i).tolist() for i, n in enumerate(_prompts(case))]
    return {"kind": kind, "engine": engine, "tokens": steps, "prompts": _prompts(case)}


# ------------------------------------------------------------------------------------------------ one pass
def run(state):
    kind = state["kind"]
    if kind == "encode":
        tokens, projected = state["encoder"].encode_project(state["pixels"], state["grid"], state["merge"], state["projector"])
        return {"tokens": tokens, "projected": projected}
    if kind == "preprocess":
        return preprocess_videos_gpu([state["frames"]])
    if kind == "kmeans":
        random.seed(state["seed"])
        torch.manual_seed(state["seed"])
        centres, times, assign = kmeans.kmeans_with_time_min_max(state["features"], state["times"], state["clusters"])
        return {"centres": centres, "times": times, "assign": assign}
    engine = state["engine"]
    if kind == "prompt":
        cache = state["cache"]
        cache.reset(0)
        return {"logits": engine.forward(state["embeds"], cache)["logits"], "k": cache.k, "v": cache.v}
    if kind == "token":
        cache, n = state["cache"], state["context"]
        cache.reset(n)
        return {"logits": engine.forward(engine.embed_tokens(state["token"]), cache)["logits"], "k": cache.k[:, n:], "v": cache.v[:, n:]}
    if kind in ("latent", "delta"):
        cache, n = state["cache"], state["embeds"].shape[0]
        cache.reset(0)
        out = {"logits": engine.forward_batch(state["embeds"], [n], [cache], [n - 1]), "rows": cache.k}
        if cache.state is not None:
            out["state"] = cache.state
        return out
    if kind == "latent_token":
        caches = state["caches"]
        for cache, n in zip(caches, state["contexts"]):
            cache.reset(n)
        B = len(caches)
        logits = engine.forward_batch(engine.embed_tokens(state["tokens"]), [1] * B, caches, list(range(B)))
        # the rows this step has appended (576 columns in each layer that caches)
        return {"logits": logits, "rows": [c.k.view(-1, c.max_len, 576)[:, n:] for c, n in zip(caches, state["contexts"])]}
    live = Sequences(engine)
    prompts, tokens = state["prompts"], state["tokens"]
    logits = [live.step([(i, t[:n], [n - 1]) for i, (t, n) in enumerate(zip(tokens, prompts))])]
    for s in range(len(tokens[0]) - prompts[0]):
        logits.append(live.step([(i, [t[n + s]], [0]) for i, (t, n) in enumerate(zip(tokens, prompts))]))
    return {"logits": logits, "states": [live.caches[i].state for i in range(len(tokens))]}


# ------------------------------------------------------------------------------------------------ what a pass cannot do without
def _target(case):
    """the processor's size rule: the budget of 16 384 tokens is shared by the frames"""
    h, w, most = case["height"], case["width"], 16384 * 784 // case["frames"]
    th, tw = round(h / 28) * 28, round(w / 28) * 28
    if th * tw > most:
        beta = math.sqrt(h * w / most)
        th, tw = math.floor(h / beta / 28) * 28, math.floor(w / beta / 28) * 28
    return th, tw


def _decoder_work(case, c, rows, contexts, wanted):
    """rows new tokens of each sequence behind contexts cached ones; wanted rows of logits. -> bytes, flops"""
    W, n = c["width"], sum(rows)
    pairs = sum(r * k + r * (r + 1) / 2 for r, k in zip(rows, contexts))       # visible (query, key) pairs
    weights, flops, cached = W * VOCAB, 2 * wanted * W * VOCAB, 0
    for lay in c["layers"]:
        m, ff = lay["mixer"], lay["mlp"]["ff"]
        H = m["heads"]
        if lay["type"].startswith("latent"):
            own = m.get("kv_from") is None
            mat = W * (m["q_rank"] + 576 * own) + m["q_rank"] * H * 192 + 512 * H * 256 + W * H * 128 + 3 * W * ff
            flops += 2 * pairs * H * (192 + 128)
            cached += (sum(contexts) + n * own) * 576 * 2
        elif lay["type"] == "attention":
            mat = W * 128 * (H + 2 * m["kv_heads"]) + W * H * 128 + 2 * W * ff
            flops += 2 * pairs * H * 256
            cached += (sum(contexts) + n) * m["kv_heads"] * 512
        else:
            mat = W * 128 * (2 * m["kv_heads"] + 2 * H) + 2 * W * H + W * H * 128 + 2 * W * ff
            flops += n * H * 6 * 128 * 128
            # the state is written once, and read too by a sequence that has one
            cached += sum(1 + (k > 0) for k in contexts) * (H * 128 * 128 + 4 * 128 * (2 * m["kv_heads"] + H)) * 4
        weights += mat
        flops += 2 * n * mat
    return weights * 2 + cached + n * W * 2 + wanted * VOCAB * 4, flops


def work(case):
    kind = case["kind"]
    if kind == "encode":
        f, p = case["frames"], case["gh"] * case["gw"]
        n, m, H, I, D = f * p, f * p // case["merge"] ** 2, VIT.hidden_size, VIT.intermediate_size, QWEN.hidden_size
        layer, ends = 4 * H * H + 2 * H * I, H * D + D * D
        flops = 27 * (2 * n * layer + 4 * n * p * H) + 2 * n * VIT.patch_dim * H + 2 * m * ends
        return {"bytes": 2 * (27 * layer + ends + VIT.patch_dim * H + n * VIT.patch_dim + m * (H + D)), "flops": flops}
    if kind == "preprocess":
        th, tw = _target(case)
        f, h, w = case["frames"], case["height"], case["width"]
        taps = lambda a, b: 4 * max(1.0, a / b)
        return {"bytes": f * (h * w * 3 + th * tw * 6), "flops": f * 6 * (h * tw * taps(w, tw) + th * tw * taps(h, th))}
    if kind == "kmeans":
        t, d = case["frames"], case["tokens"] * 3584
        K = -(-t // 15)
        # every feature against every centre once in the seeding and, at the least, in two Lloyd iterations with their means
        return {"bytes": t * d * 2 + K * d * 4, "flops": t * d * (3 * (K - 1) + 2 * (3 * K + 1))}
    if kind in ("prompt", "token"):
        rows, past = (case["rows"], 0) if kind == "prompt" else (1, case["context"])
        H, I, kv = QWEN.hidden_size, QWEN.intermediate_size, 512
        layer = 2 * H * H + 2 * H * kv + 3 * H * I
        pairs = rows * past + rows * (rows + 1) / 2
        return {"bytes": 2 * (28 * (layer + 2 * (rows + past) * kv) + H * QWEN.vocab_size + rows * H) + 4 * QWEN.vocab_size,
                "flops": 28 * (2 * rows * layer + 4 * pairs * H) + 2 * H * QWEN.vocab_size}
    c, _ = _decoder(case)
    if kind in ("latent", "delta"):
        b, f = _decoder_work(case, c, [case["rows"]], [0], 1)
    elif kind == "latent_token":
        b, f = _decoder_work(case, c, [1] * case["requests"], _contexts(case), case["requests"])
    else:
        lens = _prompts(case)
        b, f = _decoder_work(case, c, lens, [0] * len(lens), len(lens))
        for s in range(case["steps"]):
            db, df = _decoder_work(case, c, [1] * len(lens), [n + s for n in lens], len(lens))
            b, f = b + db, f + df
    return {"bytes": b, "flops": f}


def tolerance(case):
    """about four times the largest distance from `exact` that bf16 operands show over the ranges: 1.25e-2 behind the 27 layers of the
    encoder, 5.5e-2 behind the 28 of Qwen2, 9e-3 and 6e-3 behind the 4 to 9 of the small decoders; centres are 32-bit sums"""
    kind = case["kind"]
    if kind == "preprocess":
        return "exact"
    if kind == "kmeans":
        return {"rel": 1e-5, "differ": 0.0}
    return {"rel": {"encode": 0.05, "prompt": 0.2, "token": 0.2, "latent": 0.04, "latent_token": 0.04}.get(kind, 0.025)}


# ------------------------------------------------------------------------------------------------ the same in 64 bits
def _rms(x, eps=1e-6):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + eps)


def _mm(x, w, b=None):
    y = x @ w.to(F64).t()
    return y if b is None else y + b.to(F64)


def _softmax_rows(q, k, v, past, bias=None, sink=None, rows=2048):
    """causal attention of one head, `past` cached keys in front: blocks of queries against the keys they may see"""
    out = torch.empty(q.shape[0], v.shape[1], device=q.device, dtype=F64)
    for a in range(0, q.shape[0], rows):
        b = min(a + rows, q.shape[0])
        n = past + b
        s = q[a:b] @ k[:n].t()
        dist = torch.arange(past + a, past + b, device=q.device)[:, None] - torch.arange(n, device=q.device)[None]
        if bias is not None:
            s += bias[dist.clamp(0, bias.shape[0] - 1)]
        s.masked_fill_(dist < 0, -math.inf)
        top = s.amax(1, keepdim=True)
        if sink is not None:
            top = top.clamp_min(sink)
        e = torch.exp(s - top)
        z = e.sum(1, keepdim=True)
        if sink is not None:
            z = z + torch.exp(sink - top)
        out[a:b] = (e @ v[:n]) / z
    return out


def _turn(x, angle, mag=1.0, interleaved=False):
    """x [..., rows, dims] rotated by angle [rows, dims / 2] -> the pairs side by side, as the caches hold them"""
    h = x.shape[-1] // 2
    a, b = (x[..., 0::2], x[..., 1::2]) if interleaved else (x[..., :h], x[..., h:])
    c, s = torch.cos(angle) * mag, torch.sin(angle) * mag
    return torch.stack((a * c - b * s, b * c + a * s), -1).flatten(-2)


def _encode64(case, seed):
    w = random_vit_state(VIT, seed=seed, device="cuda", dtype=BF16)
    pw = random_proj_state(VIT.hidden_size, QWEN.hidden_size, seed=seed + 1, device="cuda", dtype=BF16)
    t, gh, gw, ms = case["frames"], case["gh"], case["gw"], case["merge"]
    H, p, heads, hd = VIT.hidden_size, gh * gw, 16, 72
    norm = lambda x, k: torch.nn.functional.layer_norm(x, (H,), w[k + ".weight"].to(F64), w[k + ".bias"].to(F64), VIT.layer_norm_eps)
    lin = lambda x, k: _mm(x, w[k + ".weight"].flatten(1), w[k + ".bias"])
    ids = torch.stack(torch.meshgrid(torch.arange(gh), torch.arange(gw), indexing="ij"), -1).view(gh // ms, ms, gw // ms, ms, 2)
    ids = ids.permute(0, 2, 1, 3, 4).reshape(p, 2).to("cuda", F64)
    inv = 10000.0 ** (-torch.arange(0, hd // 2, 2, device="cuda", dtype=F64) / (hd // 2))
    angle = (ids[:, :, None] * inv).flatten(1)
    x = lin(_pixels(case, seed).to(F64), "embeddings.patch_embedding")
    for i in range(VIT.num_hidden_layers):
        pre = f"encoder.layers.{i}."
        h = norm(x, pre + "layer_norm1")
        q, k, v = (lin(h, pre + f"self_attn.{n}_proj").view(t, p, heads, hd).transpose(1, 2) for n in "qkv")
        q, k = _turn(q, angle), _turn(k, angle)
        o = torch.empty_like(q)
        for f in range(t):
            o[f] = torch.softmax(q[f] @ k[f].transpose(1, 2).contiguous() * hd ** -0.5, -1) @ v[f].contiguous()
        x = x + lin(o.transpose(1, 2).reshape(t * p, H), pre + "self_attn.out_proj")
        h = lin(norm(x, pre + "layer_norm2"), pre + "mlp.fc1")
        x = x + lin(torch.nn.functional.gelu(h, approximate="tanh"), pre + "mlp.fc2")
    tokens = norm(x, "post_layernorm").view(-1, ms * ms, H).mean(1)
    hidden = torch.nn.functional.gelu(_mm(tokens, pw["readout.0.weight"], pw["readout.0.bias"]))
    return {"tokens": tokens, "projected": _mm(hidden, pw["readout.2.weight"], pw["readout.2.bias"])}


def _taps(n, m):
    """bicubic resampling of n samples to m as a matrix of weights in 22-bit fixed point"""
    scale = n / m
    wide = max(scale, 1.0)
    mat = torch.zeros(m, n, dtype=F64)
    for o in range(m):
        c = (o + 0.5) * scale
        a, b = max(0, int(c - 2 * wide + 0.5)), min(n, int(c + 2 * wide + 0.5))
        d = (torch.arange(a, b, dtype=F64) - c + 0.5).abs() / wide
        f = torch.where(d < 1, (1.5 * d - 2.5) * d * d + 1, torch.where(d < 2, -0.5 * (((d - 5) * d + 8) * d - 4), 0 * d))
        f = f / f.sum() * 2 ** 22
        mat[o, a:b] = torch.sign(f) * torch.floor(f.abs() + 0.5)
    return mat.cuda()


def _preprocess64(case, seed):
    t, h, w = case["frames"], case["height"], case["width"]
    th, tw = _target(case)
    byte = lambda x: torch.floor((x + 2.0 ** 21) / 2.0 ** 22).clamp(0, 255)
    across, down = _taps(w, tw), _taps(h, th)
    out = []
    for f in _bytes(case, seed):
        f = f.permute(2, 0, 1).to(F64)
        if tw != w:
            f = byte(f @ across.t())
        if th != h:
            f = byte(torch.stack([down @ c for c in f]))
        f = (f / 255 - 0.5) / 0.5
        f = f.view(3, th // 28, 2, 14, tw // 28, 2, 14).permute(1, 4, 2, 5, 0, 3, 6)
        out.append(f.reshape(-1, 588))
    return {"pixel_values": torch.cat(out), "grid_sizes": torch.tensor([[t, th // 14, tw // 14]]), "merge_sizes": torch.tensor([2])}


def _kmeans64(case, seed):
    x = _features(case, seed).to(F64).flatten(1)
    t, K = case["frames"], -(-case["frames"] // 15)
    ts = torch.arange(t, device="cuda", dtype=F64)
    random.seed(seed)
    torch.manual_seed(seed)
    d2 = lambda c: torch.stack([((x - r) ** 2).sum(1) for r in c], 1)
    idx = [random.randint(0, t - 1)]
    near = None
    for _ in range(K - 1):
        d = d2(x[idx[-1:]])[:, 0]
        near = d if near is None else torch.minimum(near, d)
        q = torch.empty(t, dtype=torch.float32).exponential_(1)        # what torch.multinomial draws for one sample
        idx.append(int((near / near.sum() / q.cuda().to(F64)).argmax()))
    c, ct = x[idx], ts[idx]
    for _ in range(30):
        df, dt = d2(c).sqrt(), (ts[:, None] - ct[None]).abs()
        unit = lambda d: (d - d.amin(1, keepdim=True)) / (d.amax(1, keepdim=True) - d.amin(1, keepdim=True))
        assign = torch.sqrt(unit(df) ** 2 + 2 * unit(dt) ** 2).argmin(1)
        nc, nt = torch.empty_like(c), torch.empty_like(ct)
        for k in range(K):
            rows = (assign == k).nonzero()[:, 0]
            if rows.numel() == 0:
                rows = torch.tensor([random.randint(0, t - 1)], device="cuda")
            nc[k], nt[k] = x[rows].mean(0), ts[rows].mean()
        shift = (nc - c).norm(dim=1).sum() + (nt - ct).norm()
        c, ct = nc, nt
        if shift <= 1e-4:
            break
    return {"centres": c.view(K, case["tokens"], 3584), "times": ct, "assign": assign}


def _qwen64(case, seed):
    rows, past = (case["rows"], 0) if case["kind"] == "prompt" else (1, case["context"])
    w = _qwen_state(seed)
    g = _generator(seed)
    ids = _ids(rows, 150000, seed).cuda()
    x = w["embed_tokens.weight"][ids].to(F64)
    inv = 1e6 ** (-torch.arange(0, 128, 2, device="cuda", dtype=F64) / 128)
    angle = torch.arange(past, past + rows, device="cuda", dtype=F64)[:, None] * inv
    keys, values = [], []
    for i in range(QWEN.num_hidden_layers):
        p, a = f"layers.{i}.", f"layers.{i}.self_attn."
        lin = lambda x, k: _mm(x, w[a + k + "_proj.weight"], w[a + k + "_proj.bias"])
        h = _rms(x) * w[p + "input_layernorm.weight"].to(F64)
        q = _turn(lin(h, "q").view(rows, 28, 128).transpose(0, 1), angle) * 128 ** -0.5
        k = _turn(lin(h, "k").view(rows, 4, 128).transpose(0, 1), angle)
        v = lin(h, "v").view(rows, 4, 128).transpose(0, 1)
        keys.append(k.transpose(0, 1).reshape(rows, 512))
        values.append(v.transpose(0, 1).reshape(rows, 512))
        if past:
            k, v = (torch.cat((_cached((past + 1, 512), g)[:past].to(F64).view(past, 4, 128).transpose(0, 1), n), 1) for n in (k, v))
        o = torch.stack([_softmax_rows(q[n], k[n // 7], v[n // 7], past) for n in range(28)], 1).flatten(1)
        x = x + _mm(o, w[a + "o_proj.weight"])
        h = _rms(x) * w[p + "post_attention_layernorm.weight"].to(F64)
        h = torch.nn.functional.silu(_mm(h, w[p + "mlp.gate_proj.weight"])) * _mm(h, w[p + "mlp.up_proj.weight"])
        x = x + _mm(h, w[p + "mlp.down_proj.weight"])
    h = _rms(x[-1:]) * w["norm.weight"].to(F64)
    return {"logits": _mm(h, w["lm_head.weight"])[0], "k": torch.stack(keys), "v": torch.stack(values)}


def _yarn(rot):
    n, base = rot["dims"], rot["base"]
    freq = [base ** (-2.0 * i / n) for i in range(n // 2)]
    s = rot.get("scaling")
    if s is None:
        return torch.tensor(freq, device="cuda", dtype=F64), 1.0
    place = lambda turns: n * math.log(s["original"] / (2 * math.pi * turns)) / (2 * math.log(base))
    lo, hi = max(math.floor(place(s["fast"])), 0), min(math.ceil(place(s["slow"])), n - 1)
    part = [min(max((i - lo) / max(hi - lo, 1e-3), 0.0), 1.0) for i in range(n // 2)]
    return (torch.tensor([f * (1 - r + r / s["factor"]) for f, r in zip(freq, part)], device="cuda", dtype=F64),
            1 + 0.1 * math.log(s["factor"]))


def _latent64(c, w, ids, cached):
    """one sequence: ids new tokens behind cached [layers that cache][past][576] -> (logits of the last row, new rows)"""
    x, n, new, held = w["embed"][ids].to(F64), len(ids), [], {}
    past = 0 if cached is None else cached.shape[1]
    pos = torch.arange(past, past + n, device="cuda", dtype=F64)[:, None]
    for i, lay in enumerate(c["layers"]):
        p, a, m = f"l{i}.", f"l{i}.mix.", lay["mixer"]
        pairs, H = lay["type"] == "latent_attention_2", m["heads"]
        freq, mag = _yarn(m["rot"])
        h = _rms(x) * w[p + "norm1"].to(F64)
        if m.get("kv_from") is None:
            d = _mm(h, w[a + "dkv"])
            row = torch.cat((_rms(d[:, :512]) * w[a + "dkv.norm"].to(F64), _turn(d[:, 512:], pos * freq, mag, pairs)), 1)
            held[i] = row if cached is None else torch.cat((cached[len(new)].to(F64), row))
            new.append(row)
        rows = held[i if m.get("kv_from") is None else m["kv_from"]]
        q = _mm(_rms(_mm(h, w[a + "dq"])) * w[a + "dq.norm"].to(F64), w[a + "uq"]).view(n, H, 192).transpose(0, 1)
        q = torch.cat((q[..., :128], _turn(q[..., 128:], pos * freq, mag, pairs)), -1) * m["scale"]
        uk, uv = (w[a + k].to(F64).view(H, 128, 512) for k in ("uk", "uv"))
        out = []
        for j in range(H):
            sink = w[a + "sink"][j].to(F64) if lay["type"] == "latent_attention_3" else None
            o = _softmax_rows(q[j], torch.cat((rows[:, :512] @ uk[j].t(), rows[:, 512:]), 1), rows[:, :512] @ uv[j].t(), past, sink=sink)
            out.append(o if sink is None else o * torch.sigmoid(_mm(h, w[a + "g"][j:j + 1])))
        x = x + _rms(_mm(torch.cat(out, 1), w[a + "o"])) * w[p + "norm1b"].to(F64)
        h = _rms(x) * w[p + "norm2"].to(F64)
        h = torch.nn.functional.silu(_mm(h, w[p + "mlp.gate"], w[p + "mlp.gate.b"])) * _mm(h, w[p + "mlp.up"], w[p + "mlp.up.b"])
        x = x + _rms(_mm(h, w[p + "mlp.down"], w[p + "mlp.down.b"])) * w[p + "norm2b"].to(F64)
    return _mm(_rms(x[-1:]) * w["final.norm"].to(F64), w["head"]), torch.stack(new)


def _bucket(n):
    """the bias row of distance n: 32 rows, far distances from 128 on"""
    return n if n < 16 else min(31, 16 + math.floor(math.log(n / 16) / math.log(8) * 16 + 1e-9))


def _delta64(c, w, ids, wanted):
    """one sequence from its start -> (logits of its last `wanted` rows, cached rows, state), laid out as the cache has them"""
    n, xs = len(ids), None
    x = w["embed"][ids].to(F64) + w["pos"][:n].to(F64)
    xs = x[None].repeat(4, 1, 1)
    rows, state = [], []

    def read(k):
        return (w[k + ".in"].to(F64)[:, None, None] * xs).sum(0)

    def write(k, y):
        return torch.einsum("st,snw->tnw", w[k + ".mix"].to(F64), xs) + w[k + ".out"].to(F64)[:, None, None] * y

    for i, lay in enumerate(c["layers"]):
        p, a, m = f"l{i}.", f"l{i}.mix.", lay["mixer"]
        H, G = m["heads"], m["kv_heads"]
        h = _rms(read(p + "hc1")) * w[p + "norm1"].to(F64)
        q, k, v = (_mm(h, w[a + s]) for s in "qkv")
        if lay["type"] == "attention":
            t = torch.tensor([1 + 0.1 * math.log((s + 1) // 2048 + 1) for s in range(n)], device="cuda", dtype=F64)
            q = _rms(q.view(n, H, 128)).transpose(0, 1) * t[:, None] * m["scale"]
            k, v = _rms(k.view(n, G, 128)).transpose(0, 1), v.view(n, G, 128).transpose(0, 1)
            bias = w[a + "rel"].to(F64)[[_bucket(s) for s in range(256)]]
            o = torch.cat([_softmax_rows(q[j], k[j * G // H], v[j * G // H], 0, bias=bias[:, j].contiguous()) for j in range(H)], 1)
            rows.append(torch.cat((k, v), -1).flatten())
        else:
            raw = torch.cat((q, k, v), 1)
            taps = torch.cat([w[a + s + ".conv"].to(F64) for s in "qkv"])
            ring = raw.new_zeros(4, raw.shape[1])
            for s in range(max(0, n - 4), n):
                ring[s % 4] = raw[s]
            back = torch.nn.functional.pad(raw, (0, 0, 3, 0))
            y = torch.nn.functional.silu(sum(taps[:, j] * back[j:j + n] for j in range(4)))
            q, k, v = y[:, :G * 128].view(n, G, 128), y[:, G * 128:2 * G * 128].view(n, G, 128), y[:, 2 * G * 128:].view(n, H, 128)
            unit = lambda z: z / torch.sqrt((z * z).sum(-1, keepdim=True) + 1e-6)
            q, k = (unit(z).repeat_interleave(H // G, 1) for z in (q, k))
            q = q * 128 ** -0.5
            beta = torch.sigmoid(_mm(h, w[a + "b"]))
            decay = torch.exp(-torch.exp(w[a + "A_log"].to(F64)) * torch.nn.functional.softplus(_mm(h, w[a + "a"]) + w[a + "dt_bias"].to(F64)))
            S = torch.zeros(H, 128, 128, device="cuda", dtype=F64)
            o = torch.empty(n, H, 128, device="cuda", dtype=F64)
            kt, qt, kc = k[:, :, None], q[:, :, None], k[:, :, :, None]
            for s in range(n):
                S *= decay[s, :, None, None]
                u = torch.baddbmm(v[s, :, None], kt[s], S, alpha=-1) * beta[s, :, None, None]
                S = torch.baddbmm(S, kc[s], u)
                o[s] = torch.bmm(qt[s], S)[:, 0]
            o = (_rms(o) * w[a + "norm"].to(F64)).flatten(1) * torch.nn.functional.silu(_mm(h, w[a + "g"]))
            state += [S.flatten(), ring.flatten()]
        xs = write(p + "hc1", _mm(o, w[a + "o"]))
        h = _rms(read(p + "hc2")) * w[p + "norm2"].to(F64)
        xs = write(p + "hc2", _mm(torch.nn.functional.gelu(_mm(h, w[p + "mlp.up"])), w[p + "mlp.down"]))
    last = _rms(xs.sum(0)[-wanted:]) * w["final.norm"].to(F64)
    return _mm(last, w["head"]), torch.cat(rows), torch.cat(state)


def exact(case, seed):
    kind = case["kind"]
    if kind == "encode":
        return _encode64(case, seed)
    if kind == "preprocess":
        return _preprocess64(case, seed)
    if kind == "kmeans":
        return _kmeans64(case, seed)
    if kind in ("prompt", "token"):
        return _qwen64(case, seed)
    c, dc = _decoder(case)
    w = _decoder_state(dc, seed)
    if kind == "latent":
        logits, rows = _latent64(c, w, _ids(case["rows"], VOCAB, seed).cuda(), None)
        return {"logits": logits, "rows": rows.flatten()}
    if kind == "delta":
        logits, rows, state = _delta64(c, w, _ids(case["rows"], VOCAB, seed).cuda(), 1)
        return {"logits": logits, "rows": rows, "state": state}
    if kind == "latent_token":
        g, ids = _generator(seed), _ids(case["requests"], VOCAB, seed).cuda()
        layers = sum(lay["mixer"].get("kv_from") is None for lay in c["layers"])
        outs = []
        for i, n in enumerate(_contexts(case)):
            held = _cached((layers * (n + 1) * 576,), g).view(layers, n + 1, 576)[:, :n]
            outs.append(_latent64(c, w, ids[i:i + 1], held))
        return {"logits": torch.cat([o[0] for o in outs]), "rows": [o[1] for o in outs]}
    lens, steps = _prompts(case), case["steps"]
    outs = [_delta64(c, w, _ids(n + steps, VOCAB, seed + 31 * i).cuda(), steps + 1) for i, n in enumerate(lens)]
    return {"logits": [torch.stack([o[0][s] for o in outs]) for s in range(steps + 1)], "states": [o[2] for o in outs]}
