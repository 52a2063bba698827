"""What users of this framework have it do, as calls that can be timed and checked: prompts and greedy decoding of every model family,
weight format and batch form, over the lengths they are used with.

A case is {"model", "format", "op", "batch", "tokens", "ragged", "grid", "steps"}:

    model    phi3 (Phi-3-Vision, 32 layers, full size) | pelalix | pudisun (8 layers of a Phi-3 decoder's sizes)
    format   bf16 | fp8 (e4m3 weights and prompt activations, int8 key / value cache) | q4 (4-bit group-64 weights)
    op       prefill: one model call on new prompts, up to the logits of the last position
             decode: `steps` steps of the captured greedy step behind `tokens` columns, the tokens given by the caller
    tokens   text tokens of the longest prompt; ragged: the other rows of the batch are shorter, left-padded
    grid     "HxW": 336-pixel tiles of one image in front of the text ("" none); a crop of the whole image comes on top

The program of a user loads one model and keeps it: so does this file (`_model`); what a seed makes is the requests.
"""
import gc
import math

import numpy as np
import torch

from phi_3_vision_mlx_amd.config import make_config, phi3v_config_dict
from phi_3_vision_mlx_amd.processor import collate_requests
from phi_3_vision_mlx_amd.registry import family
from phi_3_vision_mlx_amd.weights import Q4Weight, synth_weights, weight_specs

MAX_TOKENS = 128                                                 # answer length the caches are made for
DEV = "cuda:0"
EXACT_TOKENS = 12288                                             # beyond these 64 bits take too long


def _case(name, model="phi3", format="bf16", op="prefill", batch=1, tokens=128, ragged=False, grid="", steps=4):
    c = dict(model=model, format=format, op=op, batch=batch, tokens=tokens, ragged=ragged, grid=grid, steps=steps if op == "decode" else 0)
    return dict(c, name=name) if name else c


def listed():
    return [
        # a short question: the time to the first token of a chat turn
        _case("prefill_text_128"),
        # a question about one image: 16 tiles and the whole image, 2509 image tokens between 22 of text
        _case("prefill_image", tokens=22, grid="4x4"),
        # a long document, beyond the position range of the short rotation factors
        _case("prefill_long_32k", tokens=32768),
        # a prompt as long as an image's on 8-bit weights, activations quantised row by row
        _case("prefill_fp8", format="fp8", tokens=2531),
        # the smallest step: 4-bit weights, one sequence, a short context
        _case("decode_q4_128", format="q4", op="decode"),
        # the step behind an image question, the framework's headline
        _case("decode_2531", op="decode", tokens=2531),
        # the step behind a long document: the cache outweighs the weights
        _case("decode_long_32k", op="decode", tokens=32768),
        # the step on 8-bit weights and cache
        _case("decode_fp8", format="fp8", op="decode", tokens=2531),
        # a batch of prompts of different lengths, one decode step for all
        _case("decode_batch_15", op="decode", batch=15, tokens=509, ragged=True),
        # the layered families: prompts of each, and a decode batch
        _case("pelalix_prefill", model="pelalix", tokens=2048),
        _case("pudisun_prefill", model="pudisun", tokens=2048),
        _case("pudisun_decode_5", model="pudisun", op="decode", batch=5, tokens=1021, ragged=True),
    ]


def draw(rng):
    def length(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))
    kind = rng.choice(["prefill", "prefill", "image", "fp8", "decode", "decode_quant", "batch", "layered_prefill", "layered_decode"])
    if kind == "prefill":
        return _case(None, tokens=length(17, 16384))
    if kind == "image":
        h = rng.randint(1, 4)
        return _case(None, tokens=rng.randint(10, 300), grid=f"{h}x{rng.randint(1, 16 // h if h > 2 else 5)}")
    if kind == "fp8":
        return _case(None, format="fp8", tokens=length(128, 8192))
    if kind == "decode":
        return _case(None, op="decode", tokens=length(17, 32768))
    if kind == "decode_quant":
        return _case(None, format=rng.choice(["fp8", "q4"]), op="decode", tokens=length(17, 8192))
    if kind == "batch":
        return _case(None, op="decode", batch=rng.randint(2, 16), tokens=length(33, 1024), ragged=rng.random() < 0.7)
    model = rng.choice(["pelalix", "pudisun"])
    if kind == "layered_prefill":
        return _case(None, model=model, tokens=length(17, 8192))
    return _case(None, model=model, op="decode", batch=rng.randint(1, 8), tokens=length(17, 4096), ragged=rng.random() < 0.5)


# ---------------------------------------------------------------- models
def _config_dict(model):
    if model == "phi3":
        return phi3v_config_dict()
    mlp = {"kind": "dense", "ff": 8192}
    if model == "pelalix":
        layer = {"type": "attention", "mlp": mlp, "mixer": {"heads": 32, "kv_heads": 32, "dim": 96, "vdim": 96, "scale": 96 ** -0.5, "v_mix": True}}
        return {"architecture": "Pelalix", "width": 3072, "vocab": 32064, "norm": {"eps": 1e-5}, "embedding": {"scale": 1.0}, "layers": [layer] * 8}
    rot = {"base": 10000.0, "dims": 32, "scaling": {"factor": 4.0, "original": 4096, "fast": 32.0, "slow": 1.0}}
    latent = {"type": "latent_attention", "mlp": mlp,
              "mixer": {"heads": 32, "dim": 64, "rot_dim": 32, "vdim": 96, "kv_rank": 512, "rot": rot, "scale": 96 ** -0.5}}
    gla = {"type": "gla", "mlp": mlp, "mixer": {"heads": 32, "dim": 64, "vdim": 96, "tau": 16.0}}
    return {"architecture": "Pudisun", "width": 3072, "vocab": 32064, "norm": {"eps": 1e-5}, "residual_mult": 0.5, "logit_scale": 1.0,
            "layers": [latent, gla] * 4}


def _config(case):
    kw = dict(quantized_fp8=True, use_quantized_cache=True) if case["format"] == "fp8" else {}
    if case["model"] == "pudisun":
        kw["state_rows"] = 8                                     # a cache that can be rewound over a pass of decoding
    return make_config(_config_dict(case["model"]), **kw)


def _quantised(name):
    return name == "lm_head.weight" or (name.startswith("model.layers.") and name.endswith("_proj.weight"))


def _weights(case):
    """Random weights.  Phi-3's branches are scaled with the depth and its tokens' embeddings have length 1 per channel, so that, as in a
    trained stack, a layer adds to a stream larger than its branch; a 4-bit checkpoint's projections are drawn as codes."""
    cfg = _config(case)
    w = synth_weights(cfg, seed=0, device=DEV, residual_scale=True if case["model"] == "phi3" else None)
    if case["model"] == "phi3":
        w["model.embed_tokens.weight"] = w["model.embed_tokens.weight"] * 50
    if case["format"] == "q4":
        g = torch.Generator(DEV).manual_seed(1)
        for name, (n, k) in ((n, s) for n, s, _ in weight_specs(cfg) if _quantised(n)):
            std = 0.02 * ((2.0 * cfg.num_hidden_layers) ** -0.5 if name.endswith(("o_proj.weight", "down_proj.weight")) else 1.0)
            codes = torch.randint(-2 ** 31, 2 ** 31, (n, k // 8), dtype=torch.int32, device=DEV, generator=g)
            scale = std / 4.61 * (1 + 0.2 * torch.rand((n, k // 64), device=DEV, generator=g))
            w[name] = Q4Weight(codes, scale.to(torch.bfloat16), (-7.5 * scale).to(torch.bfloat16))
    return w


_held = {}


def _keep(kind, case, make):
    key = (kind, case["model"], case["format"])
    if key not in _held:
        _held.clear()                                            # one model at a time, as a program has
        gc.collect()
        torch.cuda.empty_cache()
        _held[key] = make()
    return _held[key]


def _model(case):
    def make():
        cfg = _config(case)
        return family(cfg).model_cls(cfg, _weights(case), device=DEV)
    return _keep("model", case, make)


# ---------------------------------------------------------------- requests
def _lengths(case):
    B, n = case["batch"], case["tokens"]
    return [n - (n - max(1, n // 4)) * i // B for i in range(B)] if case["ragged"] else [n] * B


def _grid(case):
    return tuple(int(v) for v in case["grid"].split("x")) if case["grid"] else (0, 0)


def _image_tokens(h, w):
    return (h * w + 1) * 144 + 1 + (h + 1) * 12 if h else 0


def _requests(case, seed):
    """Host token ids of every row; for an image its pixels, normalised as an image processor leaves them, on the GPU."""
    rng = np.random.default_rng(seed)
    rows = [np.concatenate([[1], rng.integers(3, 32000, n - 1)]).astype(np.int64) for n in _lengths(case)]
    forced = rng.integers(3, 32000, (case["steps"], case["batch"])).astype(np.int64)
    h, w = _grid(case)
    if not h:
        return [{"input_ids": r[None]} for r in rows], forced
    ids = np.concatenate([rows[0][:9], -np.ones(_image_tokens(h, w), dtype=np.int64), rows[0][9:]])[None]
    pix = torch.zeros((1, max(17, h * w + 1), 3, 336, 336), device=DEV)
    g = torch.Generator(DEV).manual_seed(seed)
    pix[:, :h * w + 1] = torch.rand((1, h * w + 1, 3, 336, 336), device=DEV, generator=g) * 3.9 - 1.8
    return [{"input_ids": ids, "pixel_values": pix, "image_sizes": np.array([[h * 336, w * 336]]), "positions": np.argwhere(ids < 0)}], forced


def prepare(case, seed):
    reqs, forced = _requests(case, seed)
    inputs = collate_requests(reqs) if case["batch"] > 1 else reqs[0]
    model = _model(case)
    if case["op"] == "prefill":
        return dict(model=model, inputs=inputs)
    _, cache = model(**inputs, max_tokens=MAX_TOKENS)
    return dict(model=model, cache=cache, past=cache[0].offset,
                tokens=[torch.tensor(t, dtype=torch.int32, device=DEV)[:, None] for t in forced])


def run(state):
    model = state["model"]
    if "inputs" in state:
        return model(**state["inputs"], max_tokens=MAX_TOKENS)[0]
    state["cache"][0].offset = state["past"]                     # (the same columns again)
    return [model.greedy_step(t, state["cache"])[0].clone() for t in state["tokens"]]


# ---------------------------------------------------------------- what a pass cannot do without
def _weight_numbers(case):
    """(weights of the projections every token meets, bytes of those, weights of the vocabulary head)."""
    cfg = _config(case)
    specs = [(n, math.prod(s)) for n, s, k in weight_specs(cfg) if k == "matrix" and "vision_embed_tokens" not in n]
    head = cfg.vocab_size * cfg.hidden_size
    body = sum(n for name, n in specs) - (head if any(name in ("lm_head.weight", "head") for name, _ in specs) else 0)
    return body, (body + head) * {"bf16": 2, "fp8": 1, "q4": 0.5625}[case["format"]], head


def _mixing(case):
    """(FLOP per visible (query, key) pair, FLOP per token, cache bytes per token, state bytes per sequence) over all layers."""
    if case["model"] == "phi3":
        return 32 * 4 * 3072, 0, 32 * 2 * 3072 * (1 if case["format"] == "fp8" else 2), 0
    if case["model"] == "pelalix":
        return 8 * (4 * 32 * 96 + 2 * 32 * 32), 0, 8 * 2 * 3072 * 2, 0
    return 4 * 2 * 32 * (96 + 96), 4 * 4 * 32 * 64 * 96, 4 * (512 + 32) * 2, 4 * 32 * 64 * 96 * 4


def work(case):
    body, wbytes, head = _weight_numbers(case)
    pair, token, cbytes, sbytes = _mixing(case)
    h, w = _grid(case)
    lens = [n + _image_tokens(h, w) for n in _lengths(case)]
    if case["op"] == "decode":
        flops = bytes_ = 0.0
        for i in range(case["steps"]):
            seen = sum(n + i for n in lens)
            flops += 2.0 * case["batch"] * (body + head) + pair * seen + token * case["batch"]
            bytes_ += wbytes + cbytes * seen + 2 * sbytes * case["batch"]
        return {"bytes": bytes_, "flops": flops}
    n = lens[0]
    flops, bytes_ = 2.0 * n * body + 2.0 * head + pair * n * n / 2 + token * n, wbytes + cbytes * n + sbytes
    if h:
        crops, D, F, T = h * w + 1, 1024, 4096, 577
        flops += crops * (23 * (2.0 * T * (4 * D * D + 2 * D * F) + 4.0 * T * T * D) + 2.0 * 576 * 588 * D) + 2.0 * _image_tokens(h, w) * (4096 * 3072 + 3072 * 3072)
        bytes_ += 2.0 * (23 * (4 * D * D + 2 * D * F) + 588 * D + 4096 * 3072 + 3072 * 3072) + crops * 3 * 336 * 336 * 4
    return {"bytes": bytes_, "flops": flops}


def tolerance(case):
    """Measured against 64 bits: 0.017 - 0.02 for the 32 layers in every format (one rounding of the stream to 16 bits a branch; 8-bit
    prompts 0.05), 0.014 - 0.018 for pudisun, 0.0026 for pelalix, whose stream is 32 bits wide."""
    return {"rel": 0.01 if case["model"] == "pelalix" else 0.03}


# ---------------------------------------------------------------- the same in 64 bits
def _rms(x, w, eps):
    return x * torch.rsqrt((x * x).mean(-1, keepdim=True) + eps) * w.double()


def _wide(case, w, name):
    """A projection's values as the format holds them, in 64 bits."""
    t = w[name]
    if isinstance(t, tuple):
        codes, scale, bias = t
        q = ((codes.long()[..., None] >> (torch.arange(8, device=DEV) * 4)) & 15).reshape(codes.shape[0], -1, 64)
        return (q * scale.double()[..., None] + bias.double()[..., None]).reshape(codes.shape[0], -1)
    if case["format"] == "fp8" and _quantised(name):
        s = t.float().abs().amax(1, keepdim=True) / 448.0
        return (t.float() / s).to(torch.float8_e4m3fn).double() * s.double()
    return t.double()


def _attend(q, k, v, scale, sink=None, talk=None):
    """Causal attention of q, k, v [T, heads, dim]; talk mixes the heads' scores, sink joins the denominator."""
    T, H = q.shape[:2]
    q, k, v = (t.transpose(0, 1).contiguous() for t in (q, k, v))
    out = torch.empty((T, H, v.shape[2]), dtype=torch.float64, device=DEV)
    kt, step = k.transpose(1, 2).contiguous(), max(1, min(T, (1 << 27) // (T * H)))
    for a in range(0, T, step):
        b = min(T, a + step)
        s = torch.matmul(q[:, a:b], kt[:, :, :b]) * scale
        if talk is not None:
            s = (talk @ s.reshape(H, -1)).reshape(s.shape)
        s.masked_fill_(torch.arange(b, device=DEV)[None] > torch.arange(a, b, device=DEV)[:, None], float("-inf"))
        if sink is not None:
            s = torch.cat([s, sink.double()[:, None, None].expand(H, b - a, 1)], dim=2)
        p = torch.softmax(s, dim=2)[:, :, :b]
        out[a:b] = torch.matmul(p, v[:, :b]).transpose(0, 1)
    return out


def _rotate(x, cos, sin):
    a, b = x.chunk(2, dim=-1)
    return torch.cat([a * cos - b * sin, b * cos + a * sin], dim=-1)


def _image_features(w, req, cfg):
    h, ww = (int(v) // 336 for v in req["image_sizes"][0])
    p, e = "model.vision_embed_tokens.img_processor.vision_model.", "model.vision_embed_tokens."
    pix = req["pixel_values"][0, :h * ww + 1].double()
    n, c = pix.shape[0], cfg.clip
    G, D = 24, c["hidden_size"]
    patches = pix.reshape(n, 3, G, 14, G, 14).permute(0, 2, 4, 1, 3, 5).reshape(n, G * G, 588)
    x = patches @ w[p + "embeddings.patch_embedding.weight"].double().reshape(D, 588).T
    x = torch.cat([w[p + "embeddings.class_embedding"].double().expand(n, 1, D), x], dim=1) + w[p + "embeddings.position_embedding.weight"].double()

    def ln(x, name):
        return torch.nn.functional.layer_norm(x, (D,), w[name + ".weight"].double(), w[name + ".bias"].double(), 1e-5)

    def lin(x, name):
        return x @ w[name + ".weight"].double().T + w[name + ".bias"].double()
    x = ln(x, p + "pre_layrnorm")
    for j in range(c["num_hidden_layers"] - 1):
        q = p + f"encoder.layers.{j}."
        y = ln(x, q + "layer_norm1")
        s = [lin(y, q + f"self_attn.{t}_proj").reshape(n, 577, 16, 64).transpose(1, 2).contiguous() for t in "qkv"]
        a = torch.softmax(torch.matmul(s[0], s[1].transpose(2, 3).contiguous()) / 8.0, dim=-1)
        x = x + lin(torch.matmul(a, s[2]).transpose(1, 2).reshape(n, 577, D), q + "self_attn.out_proj")
        y = lin(ln(x, q + "layer_norm2"), q + "mlp.fc1")
        x = x + lin(y * torch.sigmoid(1.702 * y), q + "mlp.fc2")
    x = x[:, 1:].reshape(n, 12, 2, 12, 2, D).permute(0, 1, 3, 2, 4, 5).reshape(n, 12, 12, 4 * D)
    tiles = x[1:].reshape(h * 12, ww * 12, 4 * D)                # (the reference lines the tiles up as they follow one another, phi.py:403-407)

    def lines(t):                                                # a separator behind every line
        return torch.cat([t, w[e + "sub_GN"].double().reshape(1, 1, -1).expand(t.shape[0], 1, -1)], dim=1).reshape(-1, 4 * D)
    x = torch.cat([lines(tiles), w[e + "glb_GN"].double().reshape(1, -1), lines(x[0])])
    return lin(torch.nn.functional.gelu(lin(x, e + "img_projection.0")), e + "img_projection.2")


def _phi3(case, w, cfg, ids, req):
    T, eps, nh, hd = len(ids), cfg.rms_norm_eps, cfg.num_attention_heads, 96
    x = w["model.embed_tokens.weight"][torch.as_tensor(np.maximum(ids, 0), device=DEV)].double()
    if (ids < 0).any():
        x[torch.as_tensor(ids < 0, device=DEV)] = _image_features(w, req, cfg)
    n_all = max(_lengths(case)) + _image_tokens(*_grid(case)) + MAX_TOKENS
    f = cfg.rope_scaling["long_factor" if n_all > cfg.original_max_position_embeddings else "short_factor"]
    inv = 1.0 / (torch.tensor(f, dtype=torch.float64, device=DEV) * cfg.rope_theta ** (torch.arange(0, hd, 2, dtype=torch.float64, device=DEV) / hd))
    m = math.sqrt(1 + math.log(cfg.max_position_embeddings / cfg.original_max_position_embeddings) / math.log(cfg.original_max_position_embeddings))
    ang = torch.arange(T, dtype=torch.float64, device=DEV)[:, None, None] * inv
    cos, sin = ang.cos() * m, ang.sin() * m
    for i in range(cfg.num_hidden_layers):
        p = f"model.layers.{i}."
        q, k, v = (_rms(x, w[p + "input_layernorm.weight"], eps) @ _wide(case, w, p + "self_attn.qkv_proj.weight").T).reshape(T, 3, nh, hd).unbind(1)
        o = _attend(_rotate(q, cos, sin), _rotate(k, cos, sin), v, hd ** -0.5)
        x = x + o.reshape(T, -1) @ _wide(case, w, p + "self_attn.o_proj.weight").T
        g, u = (_rms(x, w[p + "post_attention_layernorm.weight"], eps) @ _wide(case, w, p + "mlp.gate_up_proj.weight").T).chunk(2, dim=1)
        x = x + (torch.nn.functional.silu(g) * u) @ _wide(case, w, p + "mlp.down_proj.weight").T
    return _rms(x, w["model.norm.weight"], eps), _wide(case, w, "lm_head.weight")


def _pelalix(case, w, cfg, ids, req):
    def dyt(x, name):
        return torch.tanh(x * float(w[name + ".alpha"])) * w[name].double() + w[name + ".b"].double()
    x, v_first, T = w["embed"][torch.as_tensor(ids, device=DEV)].double() * cfg.embed_scale, None, len(ids)
    for i, s in enumerate(cfg.layers):
        p, m = f"l{i}.mix.", s.mixer
        h = dyt(x, f"l{i}.norm1")
        h = h + (torch.cat([torch.zeros_like(h[:1]), h[:-1]]) - h) * w[f"l{i}.shift"].double()
        q, k, v = (h @ w[p + t].double().T for t in "qkv")
        own = v
        if v_first is not None:
            lam = float(w[p + "vmix"])
            v = (1 - lam) * v + lam * v_first
        v_first = own if v_first is None else v_first
        o = _attend(_rms(q, w[p + "q.norm"], cfg.norm_eps).reshape(T, m.heads, m.dim), _rms(k, w[p + "k.norm"], cfg.norm_eps).reshape(T, m.kv_heads, m.dim),
                    v.reshape(T, m.kv_heads, m.vdim), m.scale, sink=w[p + "sink"], talk=w[p + "talk"].double())
        o = (o * torch.sigmoid(h @ w[p + "g"].double().T)[:, :, None]).reshape(T, -1)
        x = x + (o @ w[p + "o"].double().T) * w[f"l{i}.ls1"].double()
        h, p = dyt(x, f"l{i}.norm2"), f"l{i}.mlp."
        a = torch.nn.functional.silu(h @ w[p + "gate"].double().T) * (h @ w[p + "up"].double().T)
        x = x + (a @ w[p + "down"].double().T) * w[f"l{i}.ls2"].double()
    return dyt(x, "final.norm"), w["head"].double()


def _latent(h, w, p, m, eps):
    T, R = len(h), m.rank
    d = m.rot.dims
    factor, original, fast, slow = m.rot.yarn
    f = m.rot.base ** (-2.0 * np.arange(d // 2) / d)
    lo, hi = (d * math.log(original / (t * 2 * math.pi)) / (2 * math.log(m.rot.base)) for t in (fast, slow))
    lo, hi = max(math.floor(lo), 0), min(math.ceil(hi), d - 1)
    ramp = np.clip((np.arange(d // 2) - lo) / max(hi - lo, 0.001), 0, 1)
    ang = torch.arange(T, dtype=torch.float64, device=DEV)[:, None, None] * torch.tensor(f / factor * ramp + f * (1 - ramp), device=DEV)
    cos, sin = (t * (0.1 * math.log(factor) + 1.0) for t in (ang.cos(), ang.sin()))
    q = (h @ w[p + "q"].double().T).reshape(T, m.heads, m.dim + d)
    c = h @ w[p + "dkv"].double().T
    lat, kr = _rms(c[:, :R], w[p + "dkv.norm"], eps), _rotate(c[:, None, R:], cos, sin)
    k = torch.cat([(lat @ w[p + "uk"].double().T).reshape(T, m.heads, m.dim), kr.expand(T, m.heads, d)], dim=2)
    q = torch.cat([q[..., :m.dim], _rotate(q[..., m.dim:], cos, sin)], dim=2)
    o = _attend(q, k, (lat @ w[p + "uv"].double().T).reshape(T, m.heads, m.vdim), m.scale, sink=w[p + "sink"]).reshape(T, -1)
    return (o * torch.sigmoid(h @ w[p + "g"].double().T)) @ w[p + "o"].double().T


def _gla(h, w, p, m, eps):
    T = len(h)
    q = (h @ w[p + "q"].double().T).reshape(T, m.heads, 1, m.dim) * m.dim ** -0.5
    k, v = (h @ w[p + "k"].double().T).reshape(T, m.heads, m.dim, 1), (h @ w[p + "v"].double().T).reshape(T, m.heads, 1, m.vdim)
    z = (h @ w[p + "a1"].double().T) @ w[p + "a2"].double().T + w[p + "a2.b"].double()
    a = torch.exp(torch.nn.functional.logsigmoid(z) / m.tau).reshape(T, m.heads, m.dim, 1)
    s, o = torch.zeros((m.heads, m.dim, m.vdim), dtype=torch.float64, device=DEV), torch.empty((T, m.heads, 1, m.vdim), dtype=torch.float64, device=DEV)
    for t in range(T):
        s = torch.addcmul(a[t] * s, k[t], v[t])
        torch.matmul(q[t], s, out=o[t])
    o = _rms(o.squeeze(2), w[p + "norm"], eps).reshape(T, -1)
    return (o * torch.nn.functional.silu(h @ w[p + "g"].double().T)) @ w[p + "o"].double().T


def _pudisun(case, w, cfg, ids, req):
    x, eps = w["embed"][torch.as_tensor(ids, device=DEV)].double(), cfg.norm_eps
    for i, s in enumerate(cfg.layers):
        mix = _latent if hasattr(s.mixer, "rot") else _gla
        x = x + cfg.residual_mult * mix(_rms(x, w[f"l{i}.norm1"], eps), w, f"l{i}.mix.", s.mixer, eps)
        h, p = _rms(x, w[f"l{i}.norm2"], eps), f"l{i}.mlp."
        a = torch.nn.functional.gelu(h @ w[p + "gate"].double().T, approximate="tanh") * (h @ w[p + "up"].double().T)
        x = x + cfg.residual_mult * (a @ w[p + "down"].double().T)
    return _rms(x, w["final.norm"], eps) * cfg.logit_scale, w["embed"].double()


def exact(case, seed):
    if case["tokens"] * case["batch"] > EXACT_TOKENS:
        return None
    reqs, forced = _requests(case, seed)
    w, cfg = _keep("weights", case, lambda: _weights(case)), _config(case)
    rows = []
    for b, req in enumerate(reqs):
        ids = np.concatenate([req["input_ids"][0], forced[:, b]])
        x, head = {"phi3": _phi3, "pelalix": _pelalix, "pudisun": _pudisun}[case["model"]](case, w, cfg, ids, req)
        rows.append(x[-max(1, case["steps"]):] @ head.T)
    rows = torch.stack(rows)                                     # [batch, steps, vocabulary]
    return [rows[:, i:i + 1] for i in range(case["steps"])] if case["steps"] else rows
