"""The work whose speed is followed: products with block-quantized weights, attention over the paged cache and the three
decoders, each through the package's public entry points and each beside a plain 64-bit computation of the same thing.

A case is a dict of plain values; "kind" says what it calls:
  matvec     Context.matvec_q       y = W x, W block-quantized [n, k], one activation row
  gemm       Context.gemm_q         C = A W^T for m rows of bf16 activations
  attention  KVCache.attn_decode    one query per sequence and head over everything cached, a serving step of a batch
  llama, nusilix, lebelix   DecoderModel.generate, logits: a prompt, then greedy tokens; the logits behind the last one
"""
import math

import numpy as np
import torch

from skainet_amd import lebelix, llama, nusilix, runtime

DEVICE = "cuda"
TYPES = {"q4_k": runtime.Q4_K, "q5_k": runtime.Q5_K, "q6_k": runtime.Q6_K, "q8_0": runtime.Q8_0, "q4_0": runtime.Q4_0}
BLOCK = {"q4_k": (256, 144), "q5_k": (256, 176), "q6_k": (256, 210), "q8_0": (32, 34), "q4_0": (32, 18)}  # elements, bytes


# ---- cases ---------------------------------------------------------------------------------------------------------------

def listed():
    return [
        # a projection of one token at width 4096: the smallest call, its launch and its latency
        {"name": "matvec q4_k 4096x4096", "kind": "matvec", "format": "q4_k", "n": 4096, "k": 4096},
        # the feed-forward's down projection of a 7B-shaped model, one token (bench.py's headline)
        {"name": "matvec q4_k 4096x11008", "kind": "matvec", "format": "q4_k", "n": 4096, "k": 11008},
        # the output head of the same model: the largest matrix of a step
        {"name": "matvec q6_k 32000x4096", "kind": "matvec", "format": "q6_k", "n": 32000, "k": 4096},
        # a feed-forward projection of a prompt of 512 tokens
        {"name": "gemm q4_k 512x14336x4096", "kind": "gemm", "format": "q4_k", "m": 512, "n": 14336, "k": 4096},
        # a short prompt's rows, ragged, against the format that mixed files give their down projections
        {"name": "gemm q6_k 41x4096x11008", "kind": "gemm", "format": "q6_k", "m": 41, "n": 4096, "k": 11008},
        # a format without a GEMM of its own, ragged rows
        {"name": "gemm q8_0 333x4096x4096", "kind": "gemm", "format": "q8_0", "m": 333, "n": 4096, "k": 4096},
        # one step of eight sequences with 4096 cached tokens each
        {"name": "attention 8x32x4096x128", "kind": "attention", "seqs": 8, "heads": 32, "dim": 128, "tokens": 4096, "ragged": False},
        # a prompt of 512 tokens of the 7B shape, up to its first answer token
        {"name": "llama 7B prompt 512", "kind": "llama", "hidden": 4096, "ffn": 11008, "layers": 32, "heads": 32, "kv_heads": 32, "vocab": 32000,
         "format": "q4_k", "mix": "", "prompt": 512, "new": 1},
        # a chat turn of the 7B shape in the usual mixed quantization: a short question, 64 answer tokens
        {"name": "llama 7B chat 120+64", "kind": "llama", "hidden": 4096, "ffn": 11008, "layers": 32, "heads": 32, "kv_heads": 32, "vocab": 32000,
         "format": "q4_k", "mix": "q6_k", "prompt": 120, "new": 64},
        # a long document in front of a small model with grouped keys, a short answer
        {"name": "llama 2048 prompt 2000+8", "kind": "llama", "hidden": 2048, "ffn": 8192, "layers": 8, "heads": 32, "kv_heads": 8, "vocab": 32000,
         "format": "q4_k", "mix": "", "prompt": 2000, "new": 8},
        # attention over a shared cache and the delta rule in turn, dense bf16 weights: a prompt and an answer
        {"name": "nusilix 2048 1000+32", "kind": "nusilix", "width": 2048, "ffn": 8192, "layers": 8, "heads": 32, "kv_heads": 8, "dim": 64,
         "delta_heads": 32, "delta_dim": 64, "rank": 64, "groups": 4, "vocab": 32000, "prompt": 1000, "new": 32},
        # ranged attention, latent attention and the gated delta rule in turn: a longer prompt and an answer
        {"name": "lebelix 2048 2048+32", "kind": "lebelix", "width": 2048, "ffn": 8192, "layers": 6, "heads": 32, "kv_heads": 8, "dim": 64,
         "latent_heads": 16, "latent_rank": 512, "delta_heads": 16, "delta_dim": 128, "rank": 128, "side": 256, "chunk": 8192, "window": 4096,
         "vocab": 32000, "prompt": 2048, "new": 32},
    ]


def _log(rng, lo, hi):
    """A whole number, its logarithm uniform."""
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["matvec", "matvec", "gemm", "gemm", "attention", "llama", "llama", "nusilix", "lebelix"])
    if kind == "matvec":
        return {"kind": kind, "format": rng.choice(sorted(TYPES)), "n": _log(rng, 500, 32000), "k": 256 * _log(rng, 2, 56)}
    if kind == "gemm":
        return {"kind": kind, "format": rng.choice(sorted(TYPES)), "m": _log(rng, 2, 1024), "n": _log(rng, 500, 14336), "k": 256 * _log(rng, 2, 56)}
    if kind == "attention":
        return {"kind": kind, "seqs": rng.randint(1, 8), "heads": _log(rng, 4, 32), "dim": rng.choice([64, 128]), "tokens": _log(rng, 50, 4096),
                "ragged": rng.random() < 0.7}
    if kind == "llama":
        hidden, dim = 256 * rng.randint(2, 16), rng.choice([64, 128])
        heads = hidden // dim
        kv = rng.choice([heads // g for g in (1, 2, 4, 8) if heads % g == 0])
        return {"kind": kind, "hidden": hidden, "ffn": 256 * _log(rng, 4, 48), "layers": rng.randint(2, 12), "heads": heads, "kv_heads": kv,
                "vocab": _log(rng, 2000, 32000), "format": rng.choice(["q4_k", "q4_k", "q4_k", "q5_k", "q8_0", "q6_k"]),
                "mix": rng.choice(["", "q6_k"]), "prompt": _log(rng, 1, 2000), "new": _log(rng, 1, 64)}
    heads, dim = rng.choice([8, 12, 16, 24, 32]), rng.choice([64, 128])
    both = {"width": 64 * rng.randint(8, 40), "ffn": _log(rng, 1000, 8192), "layers": rng.randint(2, 6), "heads": heads, "kv_heads": rng.choice([heads, heads // 2, heads // 4]),
            "dim": dim, "rank": rng.choice([32, 64, 128]), "vocab": _log(rng, 2000, 32000), "prompt": _log(rng, 1, 2000), "new": _log(rng, 1, 32)}
    if kind == "nusilix":
        return {"kind": kind, **both, "delta_heads": rng.choice([8, 16, 24, 32]), "delta_dim": rng.choice([32, 64, 128]), "groups": rng.choice([1, 2, 4, 8])}
    return {"kind": kind, **both, "latent_heads": rng.choice([4, 8, 16]), "latent_rank": rng.choice([128, 256, 512]), "delta_heads": rng.choice([4, 8, 16]),
            "delta_dim": rng.choice([64, 128]), "side": rng.choice([32, 100, 256]), "chunk": _log(rng, 200, 4096), "window": _log(rng, 100, 4096)}


# ---- block-quantized weights -----------------------------------------------------------------------------------------------

def _generator(seed):
    return torch.Generator(device=DEVICE).manual_seed(seed)


def _bytes(g, *shape):
    return torch.randint(0, 256, shape, dtype=torch.uint8, device=DEVICE, generator=g)


def _f16_field(values):
    return values.to(torch.float16).contiguous().view(torch.uint8).reshape(-1, 2)


# rms of scale * (quant - centre) of the blocks below, for the scale of a whole matrix
_SPREAD = {"q4_k": 4.61 * 43.4, "q5_k": 9.233 * 43.4, "q6_k": 18.475 * 43.4, "q8_0": 73.3, "q4_0": 4.638}


def _blocks(g, fmt, n, k, gain=1.0):
    """Raw blocks of an [n, k] weight: quants over their whole range, values centred on zero (the minimum of a sub-block is half
    its range), scaled so that a row times a vector of unit rms has an rms of about `gain`."""
    be, bb = BLOCK[fmt]
    nb = n * (k // be)
    b = _bytes(g, nb, bb)
    d = (gain / (math.sqrt(k) * _SPREAD[fmt])) * (0.75 + 0.5 * torch.rand(nb, device=DEVICE, generator=g))
    if fmt in ("q4_k", "q5_k"):
        b[:, 0:2] = _f16_field(d)
        b[:, 2:4] = _f16_field((7.5 if fmt == "q4_k" else 15.5) * d)
        sc = torch.randint(20, 64, (nb, 8), dtype=torch.uint8, device=DEVICE, generator=g)  # scales and minima alike
        b[:, 4:8] = (sc[:, :4] & 63) | ((sc[:, 4:] >> 4) << 6)
        b[:, 8:12] = b[:, 4:8]
        b[:, 12:16] = (sc[:, 4:] & 15) | ((sc[:, 4:] & 15) << 4)
    elif fmt == "q6_k":
        sc = torch.randint(20, 64, (nb, 16), dtype=torch.int8, device=DEVICE, generator=g)
        b[:, 192:208] = torch.where(b[:, 192:208] > 127, -sc, sc).view(torch.uint8)
        b[:, 208:210] = _f16_field(d)
    else:
        b[:, 0:2] = _f16_field(d)
    return b.reshape(-1)


def _dequantized(raw, fmt, n, k):
    """[n, k] in float64 by the formulas of the block formats."""
    be, bb = BLOCK[fmt]
    b = raw.reshape(-1, bb)
    nb = b.shape[0]

    def half(at):
        return b[:, at:at + 2].contiguous().view(torch.float16).double()

    d = half(208 if fmt == "q6_k" else 0)
    if fmt in ("q4_k", "q5_k"):
        s = b[:, 4:16]
        sc = torch.cat([s[:, 0:4] & 63, (s[:, 8:12] & 15) | ((s[:, 0:4] >> 6) << 4)], 1).double()
        mn = torch.cat([s[:, 4:8] & 63, (s[:, 8:12] >> 4) | ((s[:, 4:8] >> 6) << 4)], 1).double()
        q = b[:, bb - 128:].reshape(nb, 4, 32)
        q = torch.stack([q & 15, q >> 4], 2).reshape(nb, 8, 32)
        if fmt == "q5_k":
            bit = torch.arange(8, dtype=torch.uint8, device=b.device).reshape(1, 8, 1)
            q = q | (((b[:, 16:48].reshape(nb, 1, 32) >> bit) & 1) << 4)
        w = (d * sc)[:, :, None] * q - (half(2) * mn)[:, :, None]
    elif fmt == "q6_k":
        ql, qh = b[:, :128].reshape(nb, 2, 2, 32), b[:, 128:192].reshape(nb, 2, 32)
        lo = torch.stack([ql[:, :, 0] & 15, ql[:, :, 1] & 15, ql[:, :, 0] >> 4, ql[:, :, 1] >> 4], 2)
        hi = torch.stack([(qh >> (2 * r)) & 3 for r in range(4)], 2)
        q = (lo | (hi << 4)).reshape(nb, 16, 16).double() - 32
        w = (d * b[:, 192:208].contiguous().view(torch.int8).double())[:, :, None] * q
    elif fmt == "q8_0":
        w = d * b[:, 2:].contiguous().view(torch.int8).double()
    else:
        w = d * (torch.cat([b[:, 2:] & 15, b[:, 2:] >> 4], 1).double() - 8)
    return w.reshape(n, k)


def _weight_bytes(fmt, n, k):
    be, bb = BLOCK[fmt]
    return n * (k // be) * bb


# ---- the entry points ------------------------------------------------------------------------------------------------------

_CONTEXT = []


def _context():
    """One context for the whole program, as a program has one."""
    if not _CONTEXT:
        torch.zeros(1, device=DEVICE)
        _CONTEXT.append(runtime.Context(0))
    return _CONTEXT[0]


class _Model:
    """A decoder and its prompt; gives its device memory back when it is dropped."""

    def __init__(self, model, prompt, new):
        self.model, self.prompt, self.new = model, prompt, new

    def __del__(self):
        self.model.free()


class _Cache:
    def __init__(self, kv, lengths, q, scale):
        self.kv, self.lengths, self.q, self.scale, self.out = kv, lengths, q, scale, torch.empty_like(q)


def _lengths(case):
    t, s = case["tokens"], case["seqs"]
    return [max(1, t * (i + 1) // s) for i in range(s)] if case["ragged"] else [t] * s


def _product_inputs(case, seed):
    g = _generator(seed)
    raw = _blocks(g, case["format"], case["n"], case["k"])
    x = torch.randn(case.get("m", 1), case["k"], device=DEVICE, generator=g)
    return raw, x if case["kind"] == "matvec" else x.to(torch.bfloat16)


def _attention_inputs(case, seed):
    """K and V of each sequence as the cache holds them (fp16), one query per sequence and head."""
    g = _generator(seed)
    h, d = case["heads"], case["dim"]
    kv = [torch.randn(2, n, h, d, device=DEVICE, generator=g).to(torch.float16) for n in _lengths(case)]
    return kv, torch.randn(case["seqs"], h, d, device=DEVICE, generator=g)


def prepare(case, seed):
    ctx = _context()
    kind = case["kind"]
    if kind in ("matvec", "gemm"):
        raw, x = _product_inputs(case, seed)
        y = torch.empty(x.shape[0], case["n"], device=DEVICE)
        torch.cuda.synchronize()
        return {"case": case, "w": raw, "x": x, "y": y}
    if kind == "attention":
        rows, q = _attention_inputs(case, seed)
        torch.cuda.synchronize()
        page = 256
        kv = ctx.kv_cache(case["seqs"], case["heads"], case["dim"], page, -(-case["tokens"] // page) * page)
        for s, r in enumerate(rows):
            kv.append_run(s, r[0].data_ptr(), r[1].data_ptr(), r.shape[1])
        ctx.sync()
        return {"case": case, "cache": _Cache(kv, _lengths(case), q, case["dim"] ** -0.5)}
    if kind == "llama":
        model = _llama_model(ctx, case, seed)
    elif kind == "nusilix":
        tensors = _hybrid_tensors(case, seed)
        model = nusilix.NusilixModel(ctx, _nusilix_config(case), lambda name: _to_host(tensors[name]))
    else:
        tensors = _hybrid_tensors(case, seed)
        model = lebelix.LebelixModel(ctx, _lebelix_config(case), lambda name: _to_host(tensors[name]))
    return {"case": case, "model": _Model(model, _prompt(case, seed), case["new"])}


def run(state):
    case, ctx = state["case"], _context()
    kind = case["kind"]
    if kind == "matvec":
        ctx.matvec_q(TYPES[case["format"]], state["w"].data_ptr(), case["n"], case["k"], state["x"].data_ptr(), state["y"].data_ptr())
        return state["y"]
    if kind == "gemm":
        ctx.gemm_q(TYPES[case["format"]], state["w"].data_ptr(), case["n"], case["k"], state["x"].data_ptr(), case["m"], state["y"].data_ptr())
        return state["y"]
    if kind == "attention":
        c = state["cache"]
        c.kv.attn_decode(c.q.data_ptr(), c.out.data_ptr(), c.scale)
        return c.out
    m = state["model"]
    tokens = m.model.generate(m.prompt, m.new)
    return {"tokens": np.asarray(tokens, dtype=np.int64), "logits": m.model.logits()}


# ---- what a pass cannot do without -------------------------------------------------------------------------------------------

def work(case):
    kind = case["kind"]
    if kind in ("matvec", "gemm"):
        m, n, k = case.get("m", 1), case["n"], case["k"]
        return {"bytes": _weight_bytes(case["format"], n, k) + m * k * (4 if kind == "matvec" else 2) + 4 * m * n, "flops": 2 * m * n * k}
    if kind == "attention":
        rows, h, d = sum(_lengths(case)), case["heads"], case["dim"]
        return {"bytes": 4 * rows * h * d + 8 * case["seqs"] * h * d, "flops": 4 * rows * h * d}
    p, steps = case["prompt"], case["new"] - 1
    # the weights once for the prompt and once for every token after it (they are more than the chip holds on it), the cached
    # rows that a token looks at, the recurrent states in and out; the head once for the prompt's last row and once a step
    if kind == "llama":
        layer_bytes = layer_weights = 0
        kvd = case["kv_heads"] * case["hidden"] // case["heads"]
        for l in range(case["layers"]):
            for name, (rows, cols) in _llama_shapes(case).items():
                layer_bytes += _weight_bytes(_llama_format(case, l, name), rows, cols)
                layer_weights += rows * cols
        head_bytes, head = _weight_bytes(_head_format(case), case["vocab"], case["hidden"]), case["vocab"] * case["hidden"]
        seen = sum(p + i + 1 for i in range(steps))
        kv_bytes = case["layers"] * 4 * kvd * (p + steps + seen)
        scores = case["layers"] * 4 * case["hidden"] * (p * (p + 1) // 2 + seen)
        return {"bytes": (1 + steps) * (layer_bytes + head_bytes) + kv_bytes + 4 * case["vocab"],
                "flops": 2 * layer_weights * (p + steps) + 2 * head * (1 + steps) + scores}
    layer_weights = sum(s[0] * s[1] for name, s in _hybrid_shapes(case).items() if len(s) == 2 and "embed" not in name and "conv" not in name and name != "head")
    head = case["vocab"] * case["width"]
    cfg = _nusilix_config(case) if kind == "nusilix" else _lebelix_config(case)
    kv_bytes = flops = 0
    for layer in cfg.layers:
        if layer.mixer in ("attention", "latent_attention"):
            size = getattr(layer, "mask_size", 0) or p + steps
            if layer.mixer == "latent_attention":
                row, per_key = 2 * (layer.kv_rank + layer.rot_dims), 2 * layer.heads * (layer.dim + layer.rot_dims + layer.vdim)
                seen = [min(i + 1, size) for i in range(p + steps)]
            elif kind == "lebelix":
                row, per_key = 2 * layer.kv_heads * (layer.dim + layer.vdim), 2 * layer.heads * (layer.dim + layer.vdim)
                seen = [i % size + 1 for i in range(p + steps)]
            else:
                row, per_key = 2 * layer.kv_heads * layer.dim, 4 * layer.heads * layer.dim
                seen = [i + 1 for i in range(p + steps)]
            kv_bytes += row * (p + steps + sum(seen[p:]))
            flops += per_key * sum(seen)
        else:
            d, v = layer.dim, getattr(layer, "vdim", layer.dim)
            kv_bytes += 8 * layer.heads * d * v * (1 + steps)
            flops += 6 * layer.heads * d * v * (p + steps)
    return {"bytes": (1 + steps) * 2 * (layer_weights + head) + kv_bytes + 4 * case["vocab"],
            "flops": 2 * layer_weights * (p + steps) + 2 * head * (1 + steps) + flops}


def tolerance(case):
    """About four times what the largest difference from exact() is on the listed cases and a few drawn ones."""
    kind = case["kind"]
    if kind == "matvec":
        return {"rel": 1e-6, "max": 2e-5}  # fp32 sums
    if kind == "gemm":
        return {"rel": 1.6e-6, "max": 3e-5}  # exact operands, fp32 sums in the matrix cores
    if kind == "attention":
        return {"rel": 1.5e-6, "max": 3e-5}
    if kind == "llama":
        return {"rel": 1.5e-2, "max": 2e-1}  # prompt rows rounded to bf16, cached rows to fp16
    return {"rel": 1e-2, "max": 1e-1}  # bf16 weights and rows


# ---- the decoders ------------------------------------------------------------------------------------------------------------
# The embedding is a large part of the residual stream at the end, and the head is the embedding in another order, so the
# likeliest token stands well clear of the others, as in a trained model (with independent draws the two best of 32000 logits
# often lie closer together than the rounding of a cached key); every logit still depends on every layer and position.

def _prompt(case, seed):
    return np.random.default_rng(seed).integers(0, case["vocab"], case["prompt"]).tolist()


def _order(case, seed):
    """The token that follows each token."""
    if case["kind"] == "lebelix":  # (the head is the embedding itself)
        return np.arange(case["vocab"])
    return np.random.default_rng(seed + 1).permutation(case["vocab"])


def _room(case):
    return -(-(case["prompt"] + case["new"]) // 256) * 256


def _to_host(t):
    a = t.cpu()
    return a.view(torch.int16).numpy().view(np.uint16) if t.dtype == torch.bfloat16 else a.numpy()


_LLAMA_GAIN = {"wo": 1.5}


def _llama_shapes(case):
    h, f, kvd = case["hidden"], case["ffn"], case["kv_heads"] * case["hidden"] // case["heads"]
    return {"wq": (h, h), "wk": (kvd, h), "wv": (kvd, h), "wo": (h, h), "w_gate": (f, h), "w_up": (f, h), "w_down": (h, f)}


def _llama_format(case, layer, name):
    """Mixed files give more bits to the values and the down projection of every second layer."""
    return case["mix"] if case["mix"] and layer % 2 == 0 and name in ("wv", "w_down") else case["format"]


def _head_format(case):
    return "q8_0" if case["format"] == "q8_0" else "q6_k"


def _llama_layer(g, case, layer):
    out = {name: _blocks(g, _llama_format(case, layer, name), rows, cols, _LLAMA_GAIN.get(name, 1.0)) for name, (rows, cols) in _llama_shapes(case).items()}
    for name in ("attn_norm", "ffn_norm"):
        out[name] = 1.0 + 0.1 * torch.randn(case["hidden"], device=DEVICE, generator=g)
    return out


def _llama_ends(case, seed):
    """The embedding's blocks, the head's and the last norm."""
    g = _generator(seed)
    fmt, h = _head_format(case), case["hidden"]
    table = _blocks(g, fmt, case["vocab"], h, gain=2.0 * math.sqrt(h))
    follows = torch.from_numpy(_order(case, seed)).to(DEVICE)
    head = torch.empty_like(table).reshape(case["vocab"], -1)
    head[follows] = table.reshape(case["vocab"], -1)
    return table, head.reshape(-1), 1.0 + 0.1 * torch.randn(h, device=DEVICE, generator=g)


def _llama_model(ctx, case, seed):
    types = {}
    for l in range(case["layers"]):
        for name in _llama_shapes(case):
            types[f"l{l}.{name}"] = TYPES[_llama_format(case, l, name)]
    end = TYPES[_head_format(case)]
    cfg = llama.Config(n_layer=case["layers"], hidden=case["hidden"], ffn=case["ffn"], n_head=case["heads"], head_dim=case["hidden"] // case["heads"],
                       vocab=case["vocab"], max_tokens=_room(case), n_kv_head=case["kv_heads"], type_embd=end, type_head=end, matrix_types=types)
    table, head, norm = _llama_ends(case, seed)
    w = {"tok_embd": (end, _to_host(table)), "out_head": (end, _to_host(head)), "out_norm": (None, _to_host(norm))}
    for l in range(case["layers"]):
        for name, t in _llama_layer(_generator(seed + 1000 * (l + 1)), case, l).items():
            w[f"l{l}.{name}"] = (types.get(f"l{l}.{name}"), _to_host(t))
    model = llama.LlamaModel(ctx, cfg, weights=w)
    model.host_weights = None
    return model


def _nusilix_config(case):
    attn = nusilix.Layer("attention", heads=case["heads"], dim=case["dim"], kv_heads=case["kv_heads"], scale=case["dim"] ** -0.5, temp_coef=0.1,
                         temp_every=1024, ff=case["ffn"])
    delta = nusilix.Layer("general_delta", heads=case["delta_heads"], dim=case["delta_dim"], ff=case["ffn"])
    return nusilix.Config(width=case["width"], vocab=case["vocab"], norm_groups=case["groups"], norm_eps=1e-6, residual_mult=0.5,
                          layers=[(attn, delta)[i % 2] for i in range(case["layers"])], max_tokens=_room(case))


def _lebelix_config(case):
    d, dd, ff = case["dim"], case["delta_dim"], case["ffn"]
    attn = lebelix.Layer("attention", case["heads"], d, d, kv_heads=case["kv_heads"], mask_size=case["chunk"], scale=d ** -0.5, softcap=30.0, rot_dims=d // 2, ff=ff)
    latent = lebelix.Layer("latent_attention", case["latent_heads"], 64, 128, mask_size=case["window"], scale=128 ** -0.5, rot_dims=64,
                           kv_rank=case["latent_rank"], ff=ff)
    delta = lebelix.Layer("channel_delta", case["delta_heads"], dd, dd, kv_heads=case["delta_heads"], taps=4, ff=ff)
    return lebelix.Config(width=case["width"], vocab=case["vocab"], norm_eps=1e-6, embed_scale=1.0, side_dim=case["side"],
                          layers=[(attn, latent, delta)[i % 3] for i in range(case["layers"])], max_tokens=_room(case))


def _hybrid_shapes(case):
    if case["kind"] == "nusilix":
        return nusilix.tensor_shapes(_nusilix_config(case), case["rank"])
    return lebelix.tensor_shapes(_lebelix_config(case), case["rank"], case["rank"])


def _hybrid_tensors(case, seed):
    """name -> tensor: matrices and tables in bf16, vectors in fp32; decays from nearly nothing to nearly one."""
    g = _generator(seed)
    out = {}
    for name, shape in _hybrid_shapes(case).items():
        last = name.rsplit(".", 1)[-1]
        a = torch.randn(shape, device=DEVICE, generator=g)
        if last in ("norm1", "norm2") or name == "final.norm":
            a = 0.1 * a + (1.0 if case["kind"] == "nusilix" else 0.0)
        elif last == "norm":
            a = 1.0 + 0.1 * a
        elif last == "A_log":
            a = torch.rand(shape, device=DEVICE, generator=g) * 6 - 4
        elif last == "dt_bias":
            a = 2.0 * a - 1.0
        elif last == "w0":
            a = 2.0 * a
        elif len(shape) == 1 and last != "act":
            a = 0.3 * a
        elif name == "embed":
            a = 2.0 * a
        elif len(shape) == 2 and name != "side.embed":
            a = a * shape[1] ** -0.5
        out[name] = a if len(shape) == 1 else a.to(torch.bfloat16)
    if "head" in out:
        out["head"] = torch.empty_like(out["embed"])
        out["head"][torch.from_numpy(_order(case, seed)).to(DEVICE)] = (out["embed"].float() * case["width"] ** -0.5).to(torch.bfloat16)
    return out


# ---- the same in 64 bits -------------------------------------------------------------------------------------------------------

def exact(case, seed):
    kind = case["kind"]
    if kind in ("matvec", "gemm"):
        raw, x = _product_inputs(case, seed)
        return x.double() @ _dequantized(raw, case["format"], case["n"], case["k"]).T
    if kind == "attention":
        rows, q = _attention_inputs(case, seed)
        out = []
        for s, r in enumerate(rows):
            k, v = (r[i].double().transpose(0, 1) for i in (0, 1))  # [heads, tokens, dim]
            p = torch.softmax(torch.matmul(k, q[s].double()[:, :, None])[:, :, 0] * case["dim"] ** -0.5, -1)
            out.append(torch.matmul(p[:, None, :], v)[:, 0])
        return torch.stack(out)
    prompt, follows = _prompt(case, seed), _order(case, seed)
    tokens = [int(follows[prompt[-1]])]  # (what the model will answer; the forward pass below has the last word)
    while len(tokens) < case["new"]:
        tokens.append(int(follows[tokens[-1]]))
    ids = torch.tensor(prompt + tokens[:-1], device=DEVICE)
    forward = {"llama": _llama_forward, "nusilix": _nusilix_forward, "lebelix": _lebelix_forward}[kind]
    logits = forward(case, seed, ids, case["new"])
    return {"tokens": logits.argmax(-1).cpu().numpy(), "logits": logits[-1].cpu().numpy()}


def _rms_norm(x, w, eps):
    return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + eps) * w


def _attend(q, k, v, score):
    """q [T, H, D], k [T, G, D], v [T, G, V] -> [T, H * V]; score(h, raw products [T, T]) -> probabilities."""
    group = q.shape[1] // k.shape[1]
    return torch.cat([score(h, q[:, h] @ k[:, h // group].T) @ v[:, h // group] for h in range(q.shape[1])], -1)


def _behind(T):
    i = torch.arange(T, device=DEVICE)
    return i[:, None] - i[None, :]


def _llama_forward(case, seed, ids, last):
    h, heads = case["hidden"], case["heads"]
    d, T, eps = h // heads, len(ids), 1e-5
    table, head, norm = _llama_ends(case, seed)
    row = table.numel() // case["vocab"]
    x = _dequantized(table.reshape(case["vocab"], row)[ids].reshape(-1), _head_format(case), T, h)
    freq = 10000.0 ** (-2.0 * torch.arange(d // 2, device=DEVICE, dtype=torch.float64) / d)
    angle = torch.arange(T, device=DEVICE, dtype=torch.float64)[:, None] * freq
    cos, sin = angle.cos()[:, None], angle.sin()[:, None]

    def rope(z):  # pairs of neighbours
        z = z.reshape(T, -1, d // 2, 2)
        a, b = z[..., 0], z[..., 1]
        return torch.stack([a * cos - b * sin, a * sin + b * cos], -1).reshape(T, -1, d)

    ahead = _behind(T) < 0
    for l in range(case["layers"]):
        raw = _llama_layer(_generator(seed + 1000 * (l + 1)), case, l)
        w = {name: _dequantized(raw[name], _llama_format(case, l, name), *shape) for name, shape in _llama_shapes(case).items()}
        n = _rms_norm(x, raw["attn_norm"].double(), eps)
        q, k, v = rope(n @ w["wq"].T), rope(n @ w["wk"].T), (n @ w["wv"].T).reshape(T, -1, d)
        x = x + _attend(q, k, v, lambda _, s: torch.softmax((s * d ** -0.5).masked_fill(ahead, -math.inf), -1)) @ w["wo"].T
        n = _rms_norm(x, raw["ffn_norm"].double(), eps)
        x = x + (torch.nn.functional.silu(n @ w["w_gate"].T) * (n @ w["w_up"].T)) @ w["w_down"].T
    return _rms_norm(x[-last:], norm.double(), eps) @ _dequantized(head, _head_format(case), case["vocab"], h).T


def _nusilix_forward(case, seed, ids, last):
    cfg, w, T, eps, W = _nusilix_config(case), _hybrid_tensors(case, seed), len(ids), 1e-6, case["width"]
    m = lambda name: w[name].double()  # noqa: E731
    pos = torch.arange(T, device=DEVICE, dtype=torch.float64)
    col = torch.arange(W, device=DEVICE)
    angle = pos[:, None] * 10000.0 ** (-(col // 2 * 2).double() / W)

    def grouped(z, name):
        z = z.reshape(len(z), case["groups"], -1)
        return (z * torch.rsqrt(z.square().mean(-1, keepdim=True) + eps)).reshape(len(z), W) * m(name)

    x = w["embed"][ids].double() + torch.where(col % 2 == 0, angle.sin(), angle.cos())
    dist = _behind(T)
    for i, layer in enumerate(cfg.layers):
        p, n = f"l{i}.mix.", grouped(x, f"l{i}.norm1")
        if layer.mixer == "attention":
            k = n @ m(p + "k").T + m(p + "k.b")
            q = _rms_norm(n @ m(p + "q").T + m(p + "q.b"), m(p + "q.norm"), eps)
            q = q * (1.0 + layer.temp_coef * torch.log(torch.floor((pos + 1.0) / layer.temp_every) + 1.0))[:, None]
            v = k.reshape(T, -1, layer.dim)

            def score(h, s):
                s = s * layer.scale - 2.0 ** (-8.0 * (h + 1.0) / layer.heads) * dist
                return torch.softmax(s.masked_fill(dist < 0, -math.inf), -1)

            y = _attend(q.reshape(T, -1, layer.dim), _rms_norm(k, m(p + "k.norm"), eps).reshape(T, -1, layer.dim), v, score) @ m(p + "o").T + m(p + "o.b")
        else:
            r, k, v = ((n @ m(p + c).T).reshape(T, layer.heads, layer.dim) for c in ("r", "k", "v"))
            z = torch.tanh(n @ m(p + "w1").T) @ m(p + "w2").T + m(p + "w0")
            decay = torch.exp(-math.exp(-0.5) * torch.sigmoid(z)).reshape(r.shape)
            rate = torch.sigmoid(n @ m(p + "a").T + m(p + "a.b")).reshape(r.shape)
            u = k * torch.rsqrt(k.square().sum(-1, keepdim=True) + 1e-6)
            S = torch.zeros(layer.heads, layer.dim, layer.dim, device=DEVICE, dtype=torch.float64)
            o = torch.empty_like(r)
            for t in range(T):
                S = decay[t][:, :, None] * S - (rate[t] * u[t])[:, :, None] * (u[t][:, :, None] * S).sum(1)[:, None] + k[t][:, :, None] * v[t][:, None]
                o[t] = (S * r[t][:, :, None]).sum(1)
            o = o * torch.rsqrt(o.square().mean(-1, keepdim=True) + eps)
            y = (o.reshape(T, -1) * m(p + "norm") * torch.sigmoid(n @ m(p + "g").T)) @ m(p + "o").T
        act = torch.nn.functional.softplus(m(f"l{i}.mlp.act"))
        z = n @ m(f"l{i}.mlp.up").T
        neg = z.clamp(max=0.0)
        y = y + (torch.where(z > 0, act[0] * z * z, (0.5 + act[1]) * (torch.expm1(neg) - neg)) + 0.5 * z) @ m(f"l{i}.mlp.down").T
        x = x + cfg.residual_mult * y
    return grouped(x[-last:], "final.norm") @ m("head").T


def _lebelix_forward(case, seed, ids, last):
    cfg, w, T, eps, S = _lebelix_config(case), _hybrid_tensors(case, seed), len(ids), 1e-6, case["side"]
    m = lambda name: w[name].double()  # noqa: E731
    F = torch.nn.functional
    pos = torch.arange(T, device=DEVICE, dtype=torch.float64)
    dist, place = _behind(T), torch.arange(T, device=DEVICE)

    def gelu(z):
        return F.gelu(z, approximate="tanh")

    def rotated(z, base, dims):
        angle = pos[:, None, None] * float(base) ** (-2.0 * torch.arange(dims // 2, device=DEVICE, dtype=torch.float64) / dims)
        a, b = z[..., :dims // 2], z[..., dims // 2:dims]
        return torch.cat([a * angle.cos() - b * angle.sin(), b * angle.cos() + a * angle.sin(), z[..., dims:]], -1)

    x = w["embed"][ids].double()
    for i, layer in enumerate(cfg.layers):
        p, n, H, D, V = f"l{i}.mix.", _rms_norm(x, 1.0 + m(f"l{i}.norm1"), eps), layer.heads, layer.dim, layer.vdim
        if layer.mixer == "attention":
            q, k, v = ((n @ m(p + c).T + m(p + c + ".b")).reshape(T, -1, D) for c in ("q", "k", "v"))
            q, k = (rotated(_rms_norm(z, m(p + c + ".norm"), eps), layer.rot_base, layer.rot_dims) for z, c in ((q, "q"), (k, "k")))
            block = (dist < 0) | (place[:, None] // layer.mask_size != place[None, :] // layer.mask_size)

            def score(_, s):  # a sink of score 0 takes its share
                s = (layer.softcap * torch.tanh(s * layer.scale / layer.softcap)).masked_fill(block, -math.inf)
                return torch.softmax(torch.cat([s, torch.zeros_like(s[:, :1])], 1), -1)[:, :-1]

            y = (_attend(q, k, v, score) * torch.sigmoid(n @ m(p + "g").T)) @ m(p + "o").T
        elif layer.mixer == "latent_attention":
            R = layer.rot_dims
            q = (n @ m(p + "q").T).reshape(T, H, D + R)
            d = n @ m(p + "dkv").T
            c = _rms_norm(d[:, :layer.kv_rank], m(p + "dkv.norm"), eps)
            k_rot = rotated(d[:, None, layer.kv_rank:], layer.rot_base, R).expand(T, H, R)
            q = torch.cat([q[..., :D], rotated(q[..., D:], layer.rot_base, R)], -1)
            k = torch.cat([(c @ m(p + "uk").T).reshape(T, H, D), k_rot], -1)
            block = (dist < 0) | (dist >= layer.mask_size)
            y = _attend(q, k, (c @ m(p + "uv").T).reshape(T, H, V), lambda _, s: torch.softmax((s * layer.scale).masked_fill(block, -math.inf), -1)) @ m(p + "o").T
        else:
            def conv(c):
                z, taps = n @ m(p + c).T, m(p + c + ".conv")
                z = F.pad(z, (0, 0, layer.taps - 1, 0))
                return F.silu(sum(z[j:j + T] * taps[:, j] for j in range(layer.taps)))

            unit = lambda z: z * torch.rsqrt(z.square().sum(-1, keepdim=True) + 1e-6)  # noqa: E731
            of_head = torch.arange(H, device=DEVICE) // (H // layer.kv_heads)
            q, k = (unit(conv(c).reshape(T, layer.kv_heads, D))[:, of_head] for c in ("q", "k"))
            q, v = q * D ** -0.5, conv("v").reshape(T, H, V)
            rate = torch.sigmoid(n @ m(p + "b").T)
            z = ((n @ m(p + "a1").T) @ m(p + "a2").T + m(p + "dt_bias")).reshape(T, H, D)
            decay = torch.exp(-torch.exp(m(p + "A_log"))[:, None] * F.softplus(z))
            st = torch.zeros(H, D, V, device=DEVICE, dtype=torch.float64)
            o = torch.empty(T, H, V, device=DEVICE, dtype=torch.float64)
            for t in range(T):
                st = decay[t][:, :, None] * st
                u = rate[t][:, None] * (v[t] - (st * k[t][:, :, None]).sum(1))
                st = st + k[t][:, :, None] * u[:, None]
                o[t] = (st * q[t][:, :, None]).sum(1)
            o = _rms_norm(o, m(p + "norm"), eps).reshape(T, -1)
            y = (o * torch.sigmoid((n @ m(p + "g1").T) @ m(p + "g2").T)) @ m(p + "o").T
        x = x + y
        x = x + gelu(_rms_norm(x, 1.0 + m(f"l{i}.norm2"), eps) @ m(f"l{i}.mlp.up").T) @ m(f"l{i}.mlp.down").T
        e = w["side.embed"][ids, i * S:(i + 1) * S].double()
        x = x + _rms_norm((gelu(x @ m(f"l{i}.side.gate").T) * e) @ m(f"l{i}.side.proj").T, m(f"l{i}.side.norm"), eps)
    return _rms_norm(x[-last:], 1.0 + m("final.norm"), eps) @ m("embed").T
