"""What the encoder's users run, as timed cases over the library's public entry points.

Weights have the distributions of the synthetic models (linear weights uniform
with the variance that keeps activations at unit scale, norm weights around
one), token ids are uniform over the vocabulary, images are uint8 noise, clips
are sines in noise, search embeddings are normal. `exact` restates each path in
float64 with torch; the rotary and sinusoidal angles are taken in float32
first, as the model defines them.
"""
import math
import os
import random
import sys

import numpy as np
import torch

_ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
for _p in (os.path.join(os.getcwd(), "seldon-vault-lite-rust_amd"),
           os.path.join(_ROOT, "seldon-vault-lite-rust_amd")):
    if os.path.isdir(_p):
        if _p not in sys.path:
            sys.path.insert(0, _p)
        break

import svl_amd  # noqa: E402
import svl_audio  # noqa: E402
import svl_search  # noqa: E402
import svl_synth  # noqa: E402
import svl_vision  # noqa: E402

DEV = "cuda:0"
# Rows of the embedding table: enough that a batch's rows are spread over
# memory, few enough that making the model stays quick.
VOCAB = 32768
DIMS = [768, 512, 256, 128]
# The projections of the synthetic text, vision and audio models (in, out).
PROJECTIONS = [(768, 1280), (768, 768), (768, 2304), (1152, 768), (768, 256), (256, 768),
               (512, 2048), (2048, 512), (512, 4096), (768, 6144), (3072, 768), (1024, 4096),
               (4096, 1024), (1024, 2048), (1024, 1536), (1536, 768)]
# Heads, KV heads, head dim and window of the models' attention layers.
ATTENTIONS = [(3, 1, 256, 512), (3, 1, 256, None), (4, 2, 256, 512), (4, 1, 512, None),
              (12, 12, 64, None)]


def listed():
    return [
        # A search query: one short row, ids on the host, the embedding back on the host.
        {"name": "embed_query_17", "kind": "embed_ids", "shape": "a", "tokens": 17, "dim": 768},
        # One document chunk embedded alone (latency of an interactive indexer).
        {"name": "text_1x128", "kind": "text", "shape": "a", "rows": 1, "lo": 128, "hi": 128},
        # A small request of the server: a few ragged chunks through the manifest's shape, every
        # token's projected state and the pooled embeddings back on the host.
        {"name": "forward_9_ragged", "kind": "forward", "shape": "b", "rows": 9, "lo": 19,
         "hi": 331},
        # Bulk indexing: the benchmark's batch.
        {"name": "text_64x512", "kind": "text", "shape": "a", "rows": 64, "lo": 64, "hi": 512},
        # Long documents: sliding-window and global layers at 2048 tokens.
        {"name": "text_8x2048", "kind": "text", "shape": "a", "rows": 8, "lo": 2048, "hi": 2048},
        # Images indexed from the host: four 768 x 768 pictures to embeddings.
        {"name": "image_4x768", "kind": "image", "images": 4, "gw": 48, "gh": 48},
        # Audio indexed from samples: four 30 s clips to embeddings.
        {"name": "audio_4x30s", "kind": "audio", "clips": 4, "samples": 480000},
        # One projection of the audio tower alone.
        {"name": "linear_3001x1024x4096", "kind": "linear", "rows": 3001, "in": 1024, "out": 4096},
        # One attention layer alone, an odd length beyond the window.
        {"name": "attention_1111", "kind": "attention", "seq": 1111, "heads": 3, "kv": 1,
         "hd": 256, "window": 512},
        # One norm over a bulk batch's tokens.
        {"name": "norm_18688x768", "kind": "norm", "rows": 18688, "width": 768},
        # Search of a personal vault: one query, and a batch of queries.
        {"name": "search_1", "kind": "search", "queries": 1, "chunks": 200003, "dim": 768,
         "limit": 10},
        {"name": "search_64", "kind": "search", "queries": 64, "chunks": 200003, "dim": 768,
         "limit": 10},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["embed_ids", "forward", "text", "text", "tower", "image", "audio", "linear",
                       "linear", "attention", "norm", "search", "search"])
    if kind == "embed_ids":
        return {"kind": kind, "shape": rng.choice("ab"), "tokens": _log(rng, 3, 700),
                "dim": rng.choice(DIMS)}
    if kind in ("text", "forward"):
        hi = _log(rng, 16, 2048)
        rows = _log(rng, 1, max(1, min(24 if kind == "forward" else 96, 18000 // hi)))
        return {"kind": kind, "shape": rng.choice("aab"), "rows": rows,
                "lo": max(1, int(hi * rng.uniform(0.1, 1.0))), "hi": hi}
    if kind in ("tower", "image"):
        return {"kind": kind, "images": rng.randint(1, 4), "gw": 3 * rng.randint(3, 16),
                "gh": 3 * rng.randint(3, 16)}
    if kind == "audio":
        return {"kind": kind, "clips": rng.randint(1, 4), "samples": _log(rng, 6000, 480000)}
    if kind == "linear":
        i, o = rng.choice(PROJECTIONS + [(4 * rng.randint(8, 500), rng.randint(3, 2000))])
        return {"kind": kind, "rows": _log(rng, 1, 18688), "in": i, "out": o}
    if kind == "attention":
        nh, nkv, hd, win = rng.choice(ATTENTIONS)
        return {"kind": kind, "seq": _log(rng, 5, 4096), "heads": nh, "kv": nkv, "hd": hd,
                "window": win}
    if kind == "norm":
        return {"kind": kind, "rows": _log(rng, 1, 40000),
                "width": rng.choice([256, 512, 768, 1024, 1536, 4 * rng.randint(16, 400)])}
    return {"kind": "search", "queries": _log(rng, 1, 64), "chunks": _log(rng, 3000, 200000),
            "dim": rng.choice(DIMS), "limit": _log(rng, 1, 100)}


# ---- inputs, from the seed alone -------------------------------------------------


def _gen(seed, salt=0):
    g = torch.Generator(device=DEV)
    g.manual_seed(1000003 * (int(seed) + 1) + salt)
    return g


def _uniform(g, shape, lo, hi):
    return torch.rand(shape, generator=g, device=DEV, dtype=torch.float32) * (hi - lo) + lo


def _weights(shapes, seed, salt):
    """name -> float32 CUDA tensor; one draw per tensor in the inventory's order."""
    g, out = _gen(seed, salt), {}
    for name, shape in shapes:
        if name.endswith(("input_min", "output_min")):
            t = -_uniform(g, (1,), 2.5, 4.0)
        elif name.endswith(("input_max", "output_max")):
            t = _uniform(g, (1,), 2.5, 4.0)
        elif name.endswith("layer_scalar"):
            t = _uniform(g, shape, 0.5, 1.0)
        elif name.endswith(("q_norm.weight", "k_norm.weight")):
            lo = 0.3 if name.startswith("vision") else 0.2
            t = _uniform(g, shape, lo, lo + 0.1)
        elif name.endswith(("per_dim_scale", "position_embedding_table")):
            t = _uniform(g, shape, -0.5, 0.5)
        elif name.endswith("output_proj.bias"):
            t = _uniform(g, shape, -0.1, 0.1)
        elif len(shape) == 1:
            t = _uniform(g, shape, 0.9, 1.1)
        else:
            b = math.sqrt(3.0 / float(np.prod(shape[1:])))
            t = _uniform(g, shape, -b, b)
        out[name] = t.reshape(shape)
    return out


def _host(weights):
    return {k: v.cpu().numpy() for k, v in weights.items()}


def _text_config(shape):
    return (svl_synth.config_a if shape == "a" else svl_synth.config_b)(24, VOCAB)


def _text_weights(shape, seed):
    cfg = svl_amd.TextConfig.from_json_value(_text_config(shape))
    return cfg, _weights(cfg.tensor_shapes(), seed, 1)


def _text_model(shape, seed):
    cfg, w = _text_weights(shape, seed)
    return svl_amd.TextModel(cfg, _host(w))


def _lengths(case):
    """Row lengths of a text case, spread over [lo, hi], in a mixed order."""
    if case["kind"] == "embed_ids":
        return np.array([case["tokens"]], np.int64)
    n, span = case["rows"], case["hi"] - case["lo"] + 1
    lengths = [case["lo"] + span * (2 * i + 1) // (2 * n) for i in range(n)]
    random.Random(n).shuffle(lengths)
    return np.array(lengths, np.int64)


def _rows(case, seed):
    """Row lengths of a text case and its packed ids (a CUDA int32 tensor)."""
    g = torch.Generator().manual_seed(int(seed) + 17)
    lengths = _lengths(case)
    ids = torch.randint(0, VOCAB, (int(lengths.sum()),), generator=g, dtype=torch.int32)
    return lengths, ids.to(DEV)


def _offsets(lengths):
    o = np.zeros(len(lengths) + 1, np.int64)
    o[1:] = np.cumsum(lengths)
    return o


def _pixels(case, seed):
    n = case["images"] * case["gw"] * case["gh"]
    u8 = torch.randint(0, 256, (n, 768), generator=_gen(seed, 5), device=DEV, dtype=torch.int32)
    return (u8.to(torch.float32) * np.float32(1.0 / 255.0)).contiguous()


def _image_tokens():
    return svl_vision.ImageSpecialTokens(boi=VOCAB - 6, image=VOCAB - 5, eoi=VOCAB - 4)


def _audio_tokens():
    return svl_audio.AudioSpecialTokens(boa=VOCAB - 3, audio=VOCAB - 2, eoa=VOCAB - 1)


def _vision(seed):
    c = svl_synth.config_v(16, text=_text_config("a"))
    vc = svl_vision.VisionConfig.from_json_value(c)
    return vc, _weights(vc.tensor_shapes(768), seed, 2)


def _audio(seed):
    c = svl_synth.config_au(12, text=_text_config("a"))
    ac = svl_audio.AudioConfig.from_json_value(c)
    return ac, _weights(ac.tensor_shapes(768), seed, 3)


def _clips(case, seed):
    g = _gen(seed, 7)
    t = torch.arange(case["samples"], device=DEV, dtype=torch.float64) / 16000.0
    out = []
    for _ in range(case["clips"]):
        f = torch.rand(3, generator=g, device=DEV, dtype=torch.float64) * 3900.0 + 100.0
        x = 0.3 * torch.sin(2 * math.pi * f[:, None] * t[None, :]).sum(0)
        x = x + 0.05 * torch.randn(t.numel(), generator=g, device=DEV, dtype=torch.float64)
        out.append(x.to(torch.float32))
    return torch.cat(out)


def _embeddings(case, seed):
    e = torch.randn((case["chunks"], case["dim"]), generator=_gen(seed, 8), device=DEV)
    q = torch.randn((case["queries"], case["dim"]), generator=_gen(seed, 9), device=DEV)
    return e / e.norm(dim=1, keepdim=True), q / q.norm(dim=1, keepdim=True)


def _linear_inputs(case, seed):
    g = _gen(seed, 10)
    b = math.sqrt(3.0 / case["in"])
    return (torch.randn((case["rows"], case["in"]), generator=g, device=DEV),
            _uniform(g, (case["out"], case["in"]), -b, b))


def _attention_inputs(case, seed):
    g, s, hd = _gen(seed, 11), case["seq"], case["hd"]
    q = torch.randn((s, case["heads"], hd), generator=g, device=DEV)
    k = torch.randn((s, case["kv"], hd), generator=g, device=DEV)
    v = torch.randn((s, case["kv"], hd), generator=g, device=DEV)
    # normed queries and keys: scores of about unit spread at scale 1
    f = hd ** -0.25
    return q * f, k * f, v


def _norm_inputs(case, seed):
    g = _gen(seed, 12)
    return (torch.randn((case["rows"], case["width"]), generator=g, device=DEV) * 3.0,
            _uniform(g, (case["width"],), 0.9, 1.1))


def prepare(case, seed):
    kind, s = case["kind"], {"case": case}
    if kind == "embed_ids":
        _, ids = _rows(case, seed)
        s["ids"] = ids.cpu().numpy().astype(np.uint32)
        s["model"] = _text_model(case["shape"], seed)
    elif kind == "forward":
        lengths, ids = _rows(case, seed)
        s["rows"] = np.split(ids.cpu().numpy(), _offsets(lengths)[1:-1])
        s["model"] = _text_model(case["shape"], seed)
    elif kind == "text":
        lengths, s["ids"] = _rows(case, seed)
        s["offsets"] = _offsets(lengths)
        s["out"] = torch.zeros((case["rows"], sum(_dims(case))), device=DEV)
        s["stream"] = torch.cuda.Stream()
        s["model"] = _text_model(case["shape"], seed)
    elif kind in ("tower", "image"):
        vc, w = _vision(seed)
        vision = svl_vision.VisionModel(vc, _host(w), 768)
        pixels = _pixels(case, seed)
        per = pixels.reshape(case["images"], -1, 768).cpu().numpy()
        s["patches"] = [svl_vision.ImagePatches.from_grid(p, case["gw"], case["gh"]) for p in per]
        if kind == "tower":
            s["vision"], s["source"] = vision, pixels
            s["pixels"] = torch.empty_like(pixels)
            s["out"] = torch.zeros((sum(p.soft_tokens for p in s["patches"]), 768), device=DEV)
            s["stream"] = torch.cuda.Stream()
        else:
            s["embedder"] = svl_vision.ImageEmbedder(_text_model("a", seed), vision,
                                                     _image_tokens())
    elif kind == "audio":
        ac, w = _audio(seed)
        audio = svl_audio.AudioModel(ac, _host(w), 768)
        s["embedder"] = svl_audio.AudioEmbedder(_text_model("a", seed), audio, _audio_tokens())
        s["samples"] = _clips(case, seed)
        s["lengths"] = np.full(case["clips"], case["samples"], np.int64)
    elif kind == "linear":
        s["x"], s["w"] = _linear_inputs(case, seed)
        s["out"] = torch.empty((case["rows"], case["out"]), device=DEV)
    elif kind == "attention":
        s["q"], s["k"], s["v"] = _attention_inputs(case, seed)
        s["out"] = torch.empty_like(s["q"])
    elif kind == "norm":
        s["x"], s["w"] = _norm_inputs(case, seed)
        s["out"] = torch.empty_like(s["x"])
    else:
        e, s["queries"] = _embeddings(case, seed)
        ids = np.arange(case["chunks"], dtype=np.uint64)
        s["index"] = svl_search.VectorIndex(e.cpu().numpy(), ids)
    torch.cuda.synchronize()
    return s


def _dims(case):
    return DIMS if case["shape"] == "a" else [768, 256]


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "embed_ids":
        return state["model"].embed_ids(state["ids"], case["dim"])
    if kind == "forward":
        rows = state["model"].forward_batch(state["rows"])
        return {"projected": [r.projected() for r in rows],
                "normalized": [r.normalized() for r in rows]}
    if kind == "text":
        state["model"].forward_device(state["ids"].data_ptr(), state["offsets"], _dims(case),
                                      state["out"].data_ptr(), state["stream"].cuda_stream)
        return state["out"]
    if kind == "tower":
        # the tower rescales its input in place
        with torch.cuda.stream(state["stream"]):
            state["pixels"].copy_(state["source"])
        state["vision"].forward_device(state["pixels"].data_ptr(), state["patches"],
                                       state["out"].data_ptr(), state["stream"].cuda_stream)
        return state["out"]
    if kind == "image":
        return state["embedder"].embed_batch(state["patches"], 768)
    if kind == "audio":
        return state["embedder"].embed_samples_device(state["samples"].data_ptr(),
                                                      state["lengths"], 768)
    if kind == "linear":
        svl_amd.linear(state["x"], state["w"], case["rows"], case["in"], case["out"],
                       state["out"])
        return state["out"]
    if kind == "attention":
        svl_amd.bidirectional_attention(state["q"], state["k"], state["v"], case["seq"],
                                        case["heads"], case["kv"], case["hd"], case["window"],
                                        1.0, state["out"])
        return state["out"]
    if kind == "norm":
        svl_amd.rms_norm_rows(state["x"], state["w"], case["rows"], case["width"], 1e-6,
                              state["out"])
        return state["out"]
    found = state["index"].rank_device(state["queries"].data_ptr(), case["queries"], case["dim"],
                                       limit=case["limit"])
    return {"index": np.stack([i for i, _ in found]), "score": np.stack([s for _, s in found])}


# ---- work and tolerance ----------------------------------------------------------


def _keys(n, window):
    """Query-key pairs of one row under a symmetric inclusive window."""
    if window is None or window >= n:
        return n * n
    return n * n - (n - 1 - window) * (n - window)


def _text_work(shape, lengths, projected=False):
    cfg = svl_amd.TextConfig.from_json_value(_text_config(shape))
    H, I, P, L = (cfg.hidden_size, cfg.intermediate_size, cfg.hidden_size_per_layer_input,
                  cfg.num_hidden_layers)
    T = sum(lengths)
    per_token, weights, attn = 2 * H * L * P + 2 * H * cfg.embedding_dim, 0, 0
    weights += H * L * P + H * cfg.embedding_dim
    for l in range(L):
        qd, kd = cfg.num_attention_heads * cfg.head_dim[l], cfg.num_kv_heads[l] * cfg.head_dim[l]
        m = H * (qd + 2 * kd) + qd * H + 3 * H * I + 2 * H * P
        per_token += 2 * m
        weights += m
        win = None if cfg.layer_type[l] == 1 else cfg.sliding_window
        attn += sum(4 * qd * _keys(n, win) for n in lengths)
    out = len(lengths) + (T if projected else 0)
    return {"bytes": 4 * weights + 4 * T * H + 4 * T + 4 * out * cfg.embedding_dim,
            "flops": T * per_token + attn}


def _add(*works):
    return {k: sum(w[k] for w in works) for k in ("bytes", "flops")}


def _vision_work(images, patches):
    H, I, L = 768, 3072, 16
    T, m = images * patches, 4 * 768 * 768 + 3 * 768 * 3072
    soft = images * (patches // 9)
    return {"bytes": 4 * (L * m + 2 * 768 * 768 + T * 768 + soft * 768),
            "flops": 2 * T * (L * m + 768 * 768) + 2 * soft * 768 * 768
            + L * images * 4 * H * patches * patches}


def _audio_rows(samples):
    frames = svl_audio.log_mel_layout(samples)[0]
    return frames, ((frames + 1) // 2 + 1) // 2


def _audio_work(clips, samples):
    frames, rows = _audio_rows(samples)
    H, I, L = 1024, 4096, 12
    m = 4 * H * I + 4 * H * H + 3 * H * H
    T, f1 = clips * rows, clips * ((frames + 1) // 2)
    conv = 2 * f1 * 64 * 128 * 9 + 2 * T * 32 * 32 * 1152
    return {"bytes": 4 * (L * m + H * H + H * 1536 + 1536 * 768 + clips * samples),
            "flops": 2 * T * (L * m + H * H + H * 1536 + 1536 * 768) + conv
            + L * T * 8 * 24 * 128 * 6}


def work(case):
    kind = case["kind"]
    if kind in ("embed_ids", "text", "forward"):
        lengths = [int(n) for n in _lengths(case)]
        return _text_work(case["shape"], lengths, kind == "forward")
    if kind in ("tower", "image"):
        n = case["gw"] * case["gh"]
        tower = _vision_work(case["images"], n)
        return tower if kind == "tower" else _add(
            tower, _text_work("a", [n // 9 + 4] * case["images"]))
    if kind == "audio":
        _, rows = _audio_rows(case["samples"])
        return _add(_audio_work(case["clips"], case["samples"]),
                    _text_work("a", [rows + 4] * case["clips"]))
    if kind == "linear":
        r, i, o = case["rows"], case["in"], case["out"]
        return {"bytes": 4 * (r * i + i * o + r * o), "flops": 2 * r * i * o}
    if kind == "attention":
        s, hd = case["seq"], case["hd"]
        return {"bytes": 4 * s * hd * (2 * case["heads"] + 2 * case["kv"]),
                "flops": 4 * case["heads"] * hd * _keys(s, case["window"])}
    if kind == "norm":
        return {"bytes": 8 * case["rows"] * case["width"], "flops": 4 * case["rows"] * case["width"]}
    q, n, d = case["queries"], case["chunks"], case["dim"]
    return {"bytes": 4 * d * (n + q) + 16 * q * case["limit"], "flops": 2 * q * n * d}


def tolerance(case):
    kind = case["kind"]
    if kind == "search":
        # f64 sums in the reference's order: indices and scores are defined to the bit
        return "exact"
    if kind in ("embed_ids", "text", "forward", "tower", "image", "audio"):
        # 24 layers of 32-bit sums: 2e-6 to 7e-6 against 64 bits
        return {"rel": 3e-5}
    # single sums: 5e-8 (norm) to 1.2e-6 (4096 terms) against 64 bits
    return {"rel": 1e-5}


# ---- the same results in 64 bits -------------------------------------------------


def _rms(x, w=None, eps=1e-6):
    y = x * torch.rsqrt((x * x).mean(-1, keepdim=True) + eps)
    return y if w is None else y * w


def _gelu(x):
    return 0.5 * x * (1.0 + torch.tanh(0.7978846 * (x + 0.044715 * x ** 3)))


def _angles(pos, hd_pairs, dim, theta):
    """float32 angles pos * theta^(-2i / dim), the model's definition."""
    inv = np.array([1.0 / float(np.float32(theta)) ** (2.0 * i / dim) for i in range(hd_pairs)])
    inv = torch.from_numpy(inv.astype(np.float32)).to(DEV)
    return (pos.to(torch.float32)[:, None] * inv[None, :]).to(torch.float64)


def _rotate(x, ang):
    """x [seq, heads, 2n]: element i pairs with i + n."""
    n = x.shape[-1] // 2
    c, s = ang.cos()[:, None, :], ang.sin()[:, None, :]
    a, b = x[..., :n], x[..., n:]
    return torch.cat([a * c - b * s, b * c + a * s], -1)


def _attend(q, k, v, window=None):
    """q [seq, heads, hd], k and v [seq, kv, hd], scale 1."""
    s, nh, hd = q.shape
    rep = nh // k.shape[1]
    out = torch.empty_like(q)
    i = torch.arange(s, device=DEV)
    far = None if window is None else (i[:, None] - i[None, :]).abs() > window
    for h in range(nh):
        sc = q[:, h] @ k[:, h // rep].t().contiguous()
        if far is not None:
            sc.masked_fill_(far, -math.inf)
        out[:, h] = torch.softmax(sc, -1) @ v[:, h // rep].contiguous()
    return out


def _text64(shape, seed, ids, lengths, features=None):
    """Projected states [tokens, 768] and normalized embeddings [rows, 768]; features: one
    [tokens, H] per row, put at position 2."""
    cfg, w32 = _text_weights(shape, seed)
    pick = ids.to(torch.int64)
    h = w32["language_model.embed_tokens.weight"][pick].double()
    w = {k: v.double() for k, v in w32.items() if not k.endswith("embed_tokens.weight")}
    H, P, L = cfg.hidden_size, cfg.hidden_size_per_layer_input, cfg.num_hidden_layers
    eps = float(np.float32(cfg.rms_norm_eps))
    h = h * float(np.sqrt(np.float32(H)))
    off = _offsets(lengths)
    if features is not None:
        for r, f in enumerate(features):
            h[off[r] + 2: off[r] + 2 + f.shape[0]] = f
    pos = torch.cat([torch.arange(int(n), device=DEV) for n in lengths])
    T = h.shape[0]
    ple = (h @ w["language_model.ple.per_layer_model_projection.weight"].t()) / math.sqrt(H)
    ple = _rms(ple.reshape(T, L, P), w["language_model.ple.per_layer_projection_norm.weight"], eps)
    for l in range(L):
        p = f"language_model.layers.{l}."
        hd, nkv, nh = cfg.head_dim[l], cfg.num_kv_heads[l], cfg.num_attention_heads
        full = cfg.layer_type[l] == 1
        ang = _angles(pos, hd // 2, hd, cfg.full_rope_theta if full else cfg.sliding_rope_theta)
        n = _rms(h, w[p + "input_layernorm.weight"], eps)
        q = (n @ w[p + "self_attn.q_proj.weight"].t()).reshape(T, nh, hd)
        k = (n @ w[p + "self_attn.k_proj.weight"].t()).reshape(T, nkv, hd)
        v = (n @ w[p + "self_attn.v_proj.weight"].t()).reshape(T, nkv, hd)
        q = _rotate(_rms(q, w[p + "self_attn.q_norm.weight"], eps), ang)
        k = _rotate(_rms(k, w[p + "self_attn.k_norm.weight"], eps), ang)
        v = _rms(v, None, eps)
        a = torch.cat([_attend(q[x:y], k[x:y], v[x:y], None if full else cfg.sliding_window)
                       for x, y in zip(off[:-1], off[1:])])
        a = a.reshape(T, nh * hd) @ w[p + "self_attn.o_proj.weight"].t()
        h = h + _rms(a, w[p + "post_attention_layernorm.weight"], eps)
        n = _rms(h, w[p + "pre_feedforward_layernorm.weight"], eps)
        a = _gelu(n @ w[p + "mlp.gate_proj.weight"].t()) * (n @ w[p + "mlp.up_proj.weight"].t())
        a = a @ w[p + "mlp.down_proj.weight"].t()
        h = h + _rms(a, w[p + "post_feedforward_layernorm.weight"], eps)
        a = _gelu(h @ w[p + "ple_block.per_layer_input_gate.weight"].t()) * ple[:, l]
        a = a @ w[p + "ple_block.per_layer_projection.weight"].t()
        h = (h + _rms(a, w[p + "ple_block.post_per_layer_input_norm.weight"], eps)) \
            * w[p + "layer_scalar"]
    n = _rms(h, w["language_model.norm.weight"], eps)
    proj = n @ w["language_model.embedding_projection.weight"].t()
    pooled = torch.stack([proj[x:y].mean(0) for x, y in zip(off[:-1], off[1:])])
    return proj, pooled / pooled.norm(dim=1, keepdim=True)


def _matryoshka(e, dims):
    return torch.cat([e[:, :d] / e[:, :d].norm(dim=1, keepdim=True) for d in dims], 1)


def _vision64(case, seed):
    """Soft tokens of every image, one [soft, 768] each."""
    vc, w32 = _vision(seed)
    w = {k: v.double() for k, v in w32.items()}
    x = _pixels(case, seed).double()
    n_img, gw, gh = case["images"], case["gw"], case["gh"]
    per = gw * gh
    i = torch.arange(per, device=DEV)
    px, py = (i % gw).repeat(n_img), (i // gw).repeat(n_img)
    table = w["vision_tower.patch_embedder.position_embedding_table"]
    h = (2.0 * (x - 0.5)) @ w["vision_tower.patch_embedder.input_proj.weight"].t()
    h = h + table[0][px] + table[1][py]
    nh, hd, eps = vc.num_attention_heads, vc.head_dim, vc.rms_norm_eps
    ang = [_angles(p, hd // 4, hd // 2, vc.rope_theta) for p in (px, py)]
    T, half = h.shape[0], hd // 2

    def axial(y):
        return torch.cat([_rotate(y[..., :half], ang[0]), _rotate(y[..., half:], ang[1])], -1)

    for l in range(vc.num_hidden_layers):
        p = f"vision_tower.encoder.layers.{l}."
        n = _rms(h, w[p + "input_layernorm.weight"], eps)
        q, k, v = ((n @ w[p + f"self_attn.{c}_proj.linear.weight"].t()).reshape(T, nh, hd)
                   for c in "qkv")
        q = axial(_rms(q, w[p + "self_attn.q_norm.weight"], eps))
        k = axial(_rms(k, w[p + "self_attn.k_norm.weight"], eps))
        v = _rms(v, None, eps)
        a = torch.cat([_attend(q[o:o + per], k[o:o + per], v[o:o + per])
                       for o in range(0, T, per)])
        a = a.reshape(T, nh * hd) @ w[p + "self_attn.o_proj.linear.weight"].t()
        h = h + _rms(a, w[p + "post_attention_layernorm.weight"], eps)
        n = _rms(h, w[p + "pre_feedforward_layernorm.weight"], eps)
        a = _gelu(n @ w[p + "mlp.gate_proj.linear.weight"].t()) \
            * (n @ w[p + "mlp.up_proj.linear.weight"].t())
        a = a @ w[p + "mlp.down_proj.linear.weight"].t()
        h = h + _rms(a, w[p + "post_feedforward_layernorm.weight"], eps)
    h = h.reshape(n_img, gh // 3, 3, gw // 3, 3, 768).sum((2, 4)).reshape(n_img, -1, 768)
    h = _rms(h / 9.0 * math.sqrt(768.0), None, eps)
    return list(h @ w["embed_vision.embedding_projection.weight"].t())


def _mel64(x):
    """Log-mel frames [frames, 128] of one clip and the frame mask."""
    samples = x.numel()
    padded = -(-samples // 128) * 128
    frames = (padded + 160 - 321) // 160 + 1
    buf = torch.zeros(160 + max(padded, frames * 160 + 512), device=DEV, dtype=torch.float64)
    buf[160:160 + samples] = x.double()
    win = 0.5 - 0.5 * torch.cos(2 * math.pi * torch.arange(320, device=DEV,
                                                           dtype=torch.float64) / 320)
    seg = buf.unfold(0, 320, 160)[:frames] * win.float().double()
    mag = torch.fft.rfft(seg, 512).abs()
    mel = lambda f: 2595.0 * math.log10(1.0 + f / 700.0)
    pts = np.linspace(mel(0.0), mel(8000.0), 130)
    freqs = 700.0 * (10.0 ** (pts / 2595.0) - 1.0)
    f = np.linspace(0.0, 8000.0, 257)[:, None]
    down = (f - freqs[None, :-2]) / (freqs[1:-1] - freqs[:-2])[None]
    up = (freqs[None, 2:] - f) / (freqs[2:] - freqs[1:-1])[None]
    bank = torch.from_numpy(np.maximum(0.0, np.minimum(down, up))).to(DEV)
    t = torch.arange(frames, device=DEV) * 160 + 160 < samples
    return torch.where(t[:, None], torch.log(mag @ bank + 1e-3), 0.0), t


def _conv64(x, mask, w, ln):
    """Masked 3 x 3 stride-2 convolution, LayerNorm over channels, ReLU:
    x [rows, freqs, channels] -> [rows', freqs', channels'] and the next mask."""
    x = (x * mask[:, None, None]).permute(2, 0, 1)[None]
    y = torch.nn.functional.conv2d(x, w, stride=2, padding=1)[0].permute(1, 2, 0)
    y = y - y.mean(-1, keepdim=True)
    y = y * torch.rsqrt((y * y).mean(-1, keepdim=True) + 1e-6) * ln
    return y.relu(), mask[::2]


def _audio64(case, seed):
    """Soft tokens of every clip, one [tokens, 768] each."""
    ac, w32 = _audio(seed)
    w = {k: v.double() for k, v in w32.items()}
    H, nh = ac.hidden_size, ac.num_attention_heads
    hd, chunk, left = H // nh, 12, 13
    context = chunk + left - 1
    positions = context // 2 + 1
    inc = math.log(10000.0) / (H // 2 - 1)
    inv = torch.tensor([math.exp(-i * inc) for i in range(H // 2)], dtype=torch.float64).float()
    rel = (torch.arange(positions - 1, -1, -1, dtype=torch.float32)[:, None] * inv[None]).double()
    posemb = torch.cat([rel.sin(), rel.cos()], 1).to(DEV)
    q_scale = float(np.float32(hd ** -0.5 / math.log(2.0)))
    k_scale = float(np.float32(math.log(1.0 + math.e) / math.log(2.0)))

    def clipped(x, name):
        b = {k: float(w32[f"{name}.{k}"]) for k in ("input_min", "input_max", "output_min",
                                                   "output_max")}
        y = x.clamp(b["input_min"], b["input_max"]) @ w[name + ".linear.weight"].t()
        return y.clamp(b["output_min"], b["output_max"])

    def feed(x, q):
        n = _rms(x, w[q + ".pre_layer_norm.weight"])
        n = torch.nn.functional.silu(clipped(n, q + ".ffw_layer_1"))
        return x + 0.5 * _rms(clipped(n, q + ".ffw_layer_2"), w[q + ".post_layer_norm.weight"])

    out = []
    for clip in _clips(case, seed).reshape(case["clips"], -1):
        x, mask = _mel64(clip)
        sub = "audio_tower.subsample_conv_projection."
        x, mask = _conv64(x[:, :, None], mask, w[sub + "layer0.conv.weight"],
                          w[sub + "layer0.norm.weight"])
        x, mask = _conv64(x, mask, w[sub + "layer1.conv.weight"], w[sub + "layer1.norm.weight"])
        h = x.reshape(x.shape[0], -1) @ w[sub + "input_proj_linear.weight"].t()
        rows = h.shape[0]
        qi = torch.arange(rows, device=DEV)
        d = qi[:, None] - qi[None, :]                      # query minus key
        ok = (d >= 0) & (d < left - 1) & mask[None, :] & mask[:, None]
        # context slot of the key within its query's block, minus the query's offset
        slot = (left - 1) - d
        for l in range(ac.num_hidden_layers):
            p = f"audio_tower.layers.{l}."
            h = feed(h, p + "feed_forward1")
            n = _rms(h, w[p + "norm_pre_attn.weight"])
            q, k, v = (clipped(n, p + f"self_attn.{c}_proj").reshape(rows, nh, hd)
                       for c in "qkv")
            q = q * (q_scale * torch.nn.functional.softplus(w[p + "self_attn.per_dim_scale"]))
            k = k * k_scale
            relk = (posemb @ w[p + "self_attn.relative_k_proj.weight"].t()).reshape(
                positions, nh, hd)
            att = torch.zeros_like(q)
            for j in range(nh):
                s = q[:, j] @ k[:, j].t().contiguous()
                r = q[:, j] @ relk[:, j].t().contiguous()
                inside = (slot >= 0) & (slot < positions)
                s = s + torch.where(inside, r.gather(1, slot.clamp(0, positions - 1)), 0.0)
                s = torch.tanh(s / 50.0) * 50.0
                s = s.masked_fill(~ok, -math.inf)
                a = torch.softmax(s, -1).nan_to_num(0.0)
                att[:, j] = a @ v[:, j].contiguous()
            a = clipped(att.reshape(rows, H), p + "self_attn.post")
            h = h + _rms(a, w[p + "norm_post_attn.weight"])
            n = clipped(_rms(h, w[p + "lconv1d.pre_layer_norm.weight"]),
                        p + "lconv1d.linear_start")
            n = n[:, :H] * torch.sigmoid(n[:, H:])
            taps = w[p + "lconv1d.depthwise_conv1d.weight"]
            K = taps.shape[-1]
            n = torch.nn.functional.pad(n.t()[None], (K - 1, 0))
            n = torch.nn.functional.conv1d(n, taps, groups=H)[0].t()
            n = torch.nn.functional.silu(_rms(n, w[p + "lconv1d.conv_norm.weight"]))
            h = h + clipped(n, p + "lconv1d.linear_end")
            h = _rms(feed(h, p + "feed_forward2"), w[p + "norm_out.weight"])
        y = h @ w["audio_tower.output_proj.weight"].t() + w["audio_tower.output_proj.bias"]
        y = _rms(y) @ w["embed_audio.embedding_projection.weight"].t()
        out.append(y[mask])
    return out


def _prompt64(seed, features, first, token, last):
    """The multimodal prompt of every item through the text encoder."""
    rows = [[2, first] + [token] * f.shape[0] + [last, 1] for f in features]
    ids = torch.tensor([t for r in rows for t in r], dtype=torch.int32, device=DEV)
    return _text64("a", seed, ids, np.array([len(r) for r in rows], np.int64), features)[1]


def exact(case, seed):
    kind = case["kind"]
    with torch.no_grad():
        if kind == "embed_ids":
            lengths, ids = _rows(case, seed)
            e = _text64(case["shape"], seed, ids, lengths)[1]
            return _matryoshka(e, [case["dim"]])[0].cpu().numpy()
        if kind == "forward":
            lengths, ids = _rows(case, seed)
            proj, e = _text64(case["shape"], seed, ids, lengths)
            return {"projected": np.split(proj.cpu().numpy(), _offsets(lengths)[1:-1]),
                    "normalized": list(e.cpu().numpy())}
        if kind == "text":
            lengths, ids = _rows(case, seed)
            return _matryoshka(_text64(case["shape"], seed, ids, lengths)[1], _dims(case))
        if kind == "tower":
            return torch.cat(_vision64(case, seed))
        if kind == "image":
            t = _image_tokens()
            return _prompt64(seed, _vision64(case, seed), t.boi, t.image, t.eoi).cpu().numpy()
        if kind == "audio":
            t = _audio_tokens()
            return _prompt64(seed, _audio64(case, seed), t.boa, t.audio, t.eoa).cpu().numpy()
        if kind == "linear":
            x, w = _linear_inputs(case, seed)
            return x.double() @ w.double().t()
        if kind == "attention":
            return _attend(*(t.double() for t in _attention_inputs(case, seed)), case["window"])
        if kind == "norm":
            x, w = _norm_inputs(case, seed)
            return _rms(x.double(), w.double(), float(np.float32(1e-6)))
        e, q = (t.double() for t in _embeddings(case, seed))
        s = (q @ e.t()) / (q.norm(dim=1)[:, None] * e.norm(dim=1)[None, :])
        score, index = torch.topk(s, min(case["limit"], case["chunks"]), dim=1)
        return {"index": index.cpu().numpy(), "score": score.cpu().numpy()}
