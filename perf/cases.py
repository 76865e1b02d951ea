"""What a user of this framework has it do, as cases that can be timed.

Each case is a dict of plain values; its "kind" names the part of the model
it stands for. prepare() makes a case's inputs from a seed (torch only, so
that exact() can restate them in float64) and wraps them in the layers and
caches that a program keeps; run() is one pass through the public entry
points. Sizes are those of the benchmark's decoder layer (hidden 2560, FFN
9728, QKV 3584, lm_head 131072), of the W8 out_proj (2560 x 4096) and of the
attention geometries served (32/8 heads of 128, 16/4 heads of 256, 20/4 heads
of 128).
"""

import math
import os
import sys

import torch

_ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
for _p in (_ROOT, os.path.join(_ROOT, "spark-mlx-llm_amd")):
    if _p not in sys.path:
        sys.path.insert(0, _p)

_DEV = "cuda"
_TYPES = {"bf16": torch.bfloat16, "f16": torch.float16, "f32": torch.float32}
_PROJ = {"qkv": (3584, 2560), "gate_up": (19456, 2560), "down": (2560, 9728),
         "out": (2560, 4096), "square": (2560, 2560)}
_HEADS = {"32x8x128": (32, 8, 128), "16x4x256": (16, 4, 256), "20x4x128": (20, 4, 128),
          "12x4x96": (12, 4, 96)}


def listed():
    return [
        # one decoded token through a layer's attention: QKV + RoPE, quantized
        # append, attention over 4096 cached tokens, gated W8 output projection
        {"name": "attention_block_1", "kind": "attention_block", "n": 4095, "heads": "16x4x256",
         "group": 32, "bits": 8, "dtype": "bf16"},
        # the same token through the layer's FFN block
        {"name": "ffn_1", "kind": "ffn", "m": 1, "k": 2560, "i": 9728, "group": 64,
         "dtype": "bf16"},
        # speculative verification of 8 drafted tokens: the projections of 12
        # layers, replayed as a HIP graph as the decode benchmark does
        {"name": "verify_sweep_8", "kind": "sweep", "m": 8, "layers": 12, "group": 64,
         "dtype": "bf16"},
        # a prompt of odd length through the FFN block
        {"name": "ffn_1000", "kind": "ffn", "m": 1000, "k": 2560, "i": 9728, "group": 64,
         "dtype": "bf16"},
        # a long prompt chunk through the largest W4 projection
        {"name": "w4_prefill_2048", "kind": "w4", "m": 2048, "n": 19456, "k": 2560, "group": 64,
         "dtype": "bf16"},
        # a short odd prompt through a float16 checkpoint's longest rows
        {"name": "w4_f16_333", "kind": "w4", "m": 333, "n": 2560, "k": 9728, "group": 128,
         "dtype": "f16"},
        # prefill of the W8A8 output projection
        {"name": "w8a8_512", "kind": "w8a8", "m": 512, "n": 2560, "k": 4096, "dtype": "bf16"},
        # prefill of a groupwise W8 checkpoint (or of a W8 layer's fallback)
        {"name": "w8_affine_512", "kind": "w8_affine", "m": 512, "n": 3584, "k": 2560,
         "group": 64, "dtype": "bf16", "scales": "bf16"},
        # the W8 lm_head of one decoded token
        {"name": "w8_head_1", "kind": "w8_head", "m": 1, "n": 131072, "k": 2560,
         "dtype": "bf16"},
        # a batch of 8 long contexts, one new token each
        {"name": "kv_decode_8x32768", "kind": "kv_decode", "b": 8, "n": 32768,
         "heads": "32x8x128", "format": "s8", "group": 32, "dtype": "bf16"},
        # a prompt into an empty 8-bit cache: append and fused attention
        {"name": "kv_prefill_2048", "kind": "kv_prefill", "l": 2048, "n": 2048,
         "heads": "16x4x256", "group": 32, "bits": 8, "fused": True, "mask": "causal",
         "dtype": "bf16"},
        # a prompt chunk over a 4-bit cache under the default configuration
        {"name": "kv_prefill_4bit_512", "kind": "kv_prefill", "l": 512, "n": 4096,
         "heads": "32x8x128", "group": 64, "bits": 4, "fused": False, "mask": "causal",
         "dtype": "bf16"},
    ]


def _log(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["attention_block", "ffn", "ffn", "sweep", "w4", "w4", "w4", "w8a8",
                       "w8a8", "w8_affine", "w8_head", "kv_decode", "kv_decode", "kv_prefill",
                       "kv_prefill", "kv_prefill"])
    dtype = rng.choice(["bf16", "bf16", "f16"])
    group = rng.choice([32, 64, 64, 128])
    if kind == "attention_block":
        return {"kind": kind, "n": _log(rng, 1, 16384), "heads": rng.choice(["16x4x256", "32x8x128"]),
                "group": rng.choice([32, 64]), "bits": rng.choice([8, 8, 4]), "dtype": dtype}
    if kind == "ffn":
        return {"kind": kind, "m": _log(rng, 1, 1200), "k": 2560,
                "i": rng.choice([9728, 9728, 128 * rng.randint(16, 76)]), "group": group,
                "dtype": dtype}
    if kind == "sweep":
        return {"kind": kind, "m": rng.randint(1, 16), "layers": rng.randint(3, 12),
                "group": group, "dtype": dtype}
    if kind in ("w4", "w8a8", "w8_affine"):
        n, k = _PROJ[rng.choice(sorted(_PROJ))]
        if rng.random() < 0.3:  # a narrower model or a rank's odd share of the rows
            n = _log(rng, 200, n)
        c = {"kind": kind, "m": _log(rng, 1, 2048 if kind != "w8_affine" else 700), "n": n, "k": k}
        if kind != "w8a8":
            c["group"] = group
        c["dtype"] = dtype
        if kind == "w8_affine":
            c["scales"] = rng.choice([dtype, dtype, "f32"])
        return c
    if kind == "w8_head":
        return {"kind": kind, "m": rng.choice([1, 1, 2, 4]), "n": _log(rng, 8000, 131072),
                "k": 2560, "dtype": dtype}
    if kind == "kv_decode":
        fmt = rng.choice(["s8", "u8", "u8", "u4"])
        return {"kind": kind, "b": rng.randint(1, 8), "n": _log(rng, 60, 32768),
                "heads": rng.choice(["32x8x128", "16x4x256"]), "format": fmt,
                "group": 32 if fmt == "s8" else rng.choice([32, 64]), "dtype": dtype}
    fused = rng.random() < 0.35
    n = _log(rng, 40, 4096)
    length = min(n, _log(rng, 2, 2048 if fused else 512))
    heads = rng.choice(["32x8x128", "16x4x256"] if fused
                       else ["32x8x128", "16x4x256", "20x4x128", "12x4x96"])
    return {"kind": kind, "l": length, "n": n, "heads": heads,
            "group": 32 if heads == "12x4x96" else rng.choice([32, 64]),
            "bits": 8 if fused else rng.choice([8, 8, 4, 4, 2]), "fused": fused,
            "mask": "causal" if fused else rng.choice(["causal", "causal", "none", "bool"]),
            "dtype": dtype}


# ---------------------------------------------------------------------------
# inputs, made with torch alone
# ---------------------------------------------------------------------------

def _gen(seed):
    return torch.Generator(device=_DEV).manual_seed(int(seed))


def _randn(gen, *shape, std=1.0, dtype=torch.float32):
    return torch.randn(shape, generator=gen, device=_DEV).mul_(std).to(dtype)


def _pack(codes, bits):
    """Codes (uint8 values) [..., D] -> int32 words, code j at bits bits*j."""
    per = 32 // bits
    c = codes.to(torch.int64).reshape(*codes.shape[:-1], codes.shape[-1] // per, per)
    word = (c << (bits * torch.arange(per, device=c.device))).sum(-1)
    return torch.where(word >= 1 << 31, word - (1 << 32), word).to(torch.int32)


def _affine(w, bits, group, dtype):
    """Groupwise affine quantization over the last axis: codes (uint8),
    scales and biases in dtype, value = code * scale + bias."""
    g = w.to(torch.float32).reshape(*w.shape[:-1], w.shape[-1] // group, group)
    lo, hi = g.amin(-1), g.amax(-1)
    s = ((hi - lo) / (2 ** bits - 1)).to(dtype)
    b = lo.to(dtype)
    codes = ((g - b.float()[..., None]) / s.float()[..., None]).round_().clamp_(0, 2 ** bits - 1)
    return codes.to(torch.uint8).reshape(w.shape), s, b


def _value(codes, s, b):
    """float64 values of an affine tuple."""
    group = codes.shape[-1] // s.shape[-1]
    c = codes.double().reshape(*s.shape, group)
    return c.mul_(s.double()[..., None]).add_(b.double()[..., None]).reshape(codes.shape)


def _w4_raw(gen, n, k, group, dtype):
    return _affine(_randn(gen, n, k, std=0.02, dtype=dtype), 4, group, dtype)


def _w8_raw(gen, n, k):
    """Per-channel symmetric int8 rows of N(0, 0.02) weights."""
    w = _randn(gen, n, k, std=0.02)
    s = w.abs().amax(1) / 127
    return w.div_(s[:, None]).round_().clamp_(-127, 127).to(torch.int8), s


def _kv_raw(gen, c, b, hkv, n, d):
    """One K or V cache: (codes, scales, biases), or (codes, fp16 scales)."""
    dtype = _TYPES[c["dtype"]]
    x = _randn(gen, b, hkv, n, d, dtype=dtype)
    if c.get("format") == "s8":
        x = x.float()
        s = (x.abs().amax(-1) / 127).to(torch.float16)
        return x.div_(s.float()[..., None]).round_().clamp_(-127, 127).to(torch.int8), s
    return _affine(x, _bits(c), c["group"], dtype)


def _bits(c):
    return {"u8": 8, "u4": 4}[c["format"]] if "format" in c else c["bits"]


def _inputs(c, seed):
    gen = _gen(seed)
    dtype = _TYPES[c["dtype"]]
    kind = c["kind"]
    if kind == "attention_block":
        h, hkv, d = _HEADS[c["heads"]]
        return {"x": _randn(gen, 1, 1, 2560, dtype=dtype),
                "qkv": _w4_raw(gen, (h + 2 * hkv) * d, 2560, c["group"], dtype),
                "k": _kv_raw(gen, c, 1, hkv, c["n"], d), "v": _kv_raw(gen, c, 1, hkv, c["n"], d),
                "g": _randn(gen, h, 2560, std=0.02, dtype=dtype), "out": _w8_raw(gen, 2560, h * d)}
    if kind == "ffn":
        m, k, i, g = c["m"], c["k"], c["i"], c["group"]
        return {"x": _randn(gen, m, k, dtype=dtype), "a": _randn(gen, m, k, std=0.5, dtype=dtype),
                "norm": (1 + _randn(gen, k, std=0.1)).to(dtype),
                "gate": _w4_raw(gen, i, k, g, dtype), "up": _w4_raw(gen, i, k, g, dtype),
                "down": _w4_raw(gen, k, i, g, dtype)}
    if kind == "sweep":
        return {"x": {k: _randn(gen, c["m"], k, dtype=dtype) for k in (2560, 9728)},
                "w": [{p: _w4_raw(gen, *_PROJ[p], c["group"], dtype)
                       for p in ("qkv", "gate_up", "down")} for _ in range(c["layers"])]}
    if kind == "w4":
        return {"x": _randn(gen, 1, c["m"], c["k"], dtype=dtype),
                "w": _w4_raw(gen, c["n"], c["k"], c["group"], dtype)}
    if kind in ("w8a8", "w8_head"):
        return {"x": _randn(gen, 1, c["m"], c["k"], dtype=dtype), "w": _w8_raw(gen, c["n"], c["k"])}
    if kind == "w8_affine":
        return {"x": _randn(gen, 1, c["m"], c["k"], dtype=dtype),
                "w": _affine(_randn(gen, c["n"], c["k"], std=0.02), 8, c["group"],
                             _TYPES[c["scales"]])}
    h, hkv, d = _HEADS[c["heads"]]
    if kind == "kv_decode":
        return {"q": _randn(gen, c["b"], h, 1, d, dtype=dtype),
                "k": _kv_raw(gen, c, c["b"], hkv, c["n"], d),
                "v": _kv_raw(gen, c, c["b"], hkv, c["n"], d)}
    # kv_prefill: n - l tokens are cached, l are new
    r = {"q": _randn(gen, 1, h, c["l"], d, dtype=dtype),
         "k_new": _randn(gen, 1, hkv, c["l"], d, dtype=dtype),
         "v_new": _randn(gen, 1, hkv, c["l"], d, dtype=dtype)}
    if c["n"] > c["l"]:
        r["k"] = _kv_raw(gen, c, 1, hkv, c["n"] - c["l"], d)
        r["v"] = _kv_raw(gen, c, 1, hkv, c["n"] - c["l"], d)
    if c["mask"] == "bool":  # causal, with earlier tokens hidden here and there
        seen = torch.ones((c["l"], c["n"]), dtype=torch.bool, device=_DEV).tril(c["n"] - c["l"])
        hide = torch.rand((c["l"], c["n"]), generator=gen, device=_DEV) < 0.1
        hide[:, 0] = False
        r["mask"] = seen & ~hide
    return r


# ---------------------------------------------------------------------------
# the program's layers and caches
# ---------------------------------------------------------------------------

def _linear4(raw, group):
    from sparkq.ops import QuantizedLinear

    return QuantizedLinear(_pack(raw[0], 4), raw[1], raw[2], group_size=group, bits=4)


def _cache(c, raw_k, raw_v, hkv, d, n):
    """A quantized cache with room for n tokens that holds the raw ones."""
    from sparkq import QuantizedKVCache

    bits, group = c["bits"], c["group"]
    dtype = _TYPES[c["dtype"]]
    cache = QuantizedKVCache(group_size=group, bits=bits)
    room = -(-n // cache.step) * cache.step

    def store(raw):
        t = (torch.zeros((1, hkv, room, d * bits // 32), dtype=torch.int32, device=_DEV),
             torch.zeros((1, hkv, room, d // group), dtype=dtype, device=_DEV),
             torch.zeros((1, hkv, room, d // group), dtype=dtype, device=_DEV))
        if raw is not None:
            for dst, src in zip(t, (_pack(raw[0], bits), raw[1], raw[2])):
                dst[:, :, : src.shape[2]] = src
        return t

    cache.keys, cache.values = store(raw_k), store(raw_v)
    return cache


class _MLP(torch.nn.Module):
    def __init__(self, gate, up, down):
        super().__init__()
        self.gate_proj, self.up_proj, self.down_proj = gate, up, down


def prepare(case, seed):
    import sparkq
    from sparkq import ops

    c, t = case, _inputs(case, seed)
    kind = c["kind"]
    s = {"case": c}
    if kind == "attention_block":
        h, hkv, d = _HEADS[c["heads"]]
        w8, ws = t["out"]
        packed = (w8.view(torch.int32) ^ -2139062144).contiguous()
        affine = ops.QuantizedLinear(packed, ws[:, None].repeat(1, h * d // 64),
                                     (-128 * ws)[:, None].repeat(1, h * d // 64), group_size=64,
                                     bits=8)
        gate = torch.nn.Linear(2560, h, bias=False, device=_DEV, dtype=t["x"].dtype)
        gate.weight.requires_grad_(False).copy_(t["g"])
        s.update(x=t["x"], qkv=_linear4(t["qkv"], c["group"]),
                 rope=ops.RoPE(d, base=500000.0), gate=gate,
                 out=ops.W8A16PerChannelLinear(affine, w8, ws),
                 cache=_cache(c, t["k"], t["v"], hkv, d, c["n"] + 1), config=ops.SDPAConfig())
    elif kind == "ffn":
        s.update(x=t["x"], a=t["a"], norm=ops.RMSNorm(c["k"], 1e-6, weight=t["norm"]),
                 mlp=_MLP(*(_linear4(t[p], c["group"]) for p in ("gate", "up", "down"))))
    elif kind == "sweep":
        out = {p: torch.empty((c["layers"], c["m"], _PROJ[p][0]), dtype=_TYPES[c["dtype"]],
                              device=_DEV) for p in ("qkv", "gate_up", "down")}
        layers = [{p: (_pack(w[p][0], 4), w[p][1], w[p][2]) for p in w} for w in t["w"]]

        def step():
            for i, layer in enumerate(layers):
                for p in ("qkv", "gate_up", "down"):
                    sparkq.affine_quantized_matmul(t["x"][_PROJ[p][1]], *layer[p],
                                                   group_size=c["group"], out=out[p][i])

        side = torch.cuda.Stream()
        side.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(side):
            step()
        torch.cuda.current_stream().wait_stream(side)
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=side):
            step()
        s.update(graph=graph, out=out, keep=(t["x"], layers, side))
    elif kind == "w4":
        layer = _linear4(t["w"], c["group"])
        ops.prepare_w4_layers(layer)
        s.update(x=t["x"], layer=layer)
    elif kind == "w8a8":
        s.update(x=t["x"], layer=sparkq.W8A8Linear(*t["w"]))
    elif kind == "w8_head":
        s.update(x=t["x"], w=t["w"])
    elif kind == "w8_affine":
        s.update(x=t["x"], layer=ops.QuantizedLinear(_pack(t["w"][0], 8), t["w"][1], t["w"][2],
                                                     group_size=c["group"], bits=8))
    elif kind == "kv_decode":
        if c["format"] == "s8":
            k, v = t["k"], t["v"]
        else:
            k, v = ((_pack(r[0], _bits(c)), r[1], r[2]) for r in (t["k"], t["v"]))
        s.update(q=t["q"], k=k, v=v)
    else:
        h, hkv, d = _HEADS[c["heads"]]
        s.update(q=t["q"], k_new=t["k_new"], v_new=t["v_new"],
                 cache=_cache(c, t.get("k"), t.get("v"), hkv, d, c["n"]),
                 mask={"causal": "causal", "none": None}.get(c["mask"], t.get("mask")),
                 config=ops.SDPAConfig(fused_quantized_sdpa_prefill=c["fused"]))
    return s


def run(state):
    import sparkq
    from sparkq import ops

    c = state["case"]
    kind = c["kind"]
    if kind == "attention_block":
        h, hkv, d = _HEADS[c["heads"]]
        cache = state["cache"]
        cache.offset = c["n"]  # the position that this token takes
        q, k, v = ops.dispatch_qkv(state["x"], state["qkv"], state["rope"], q_size=h * d,
                                   kv_size=hkv * d, n_heads=h, n_kv_heads=hkv, head_dim=d,
                                   offset=cache.offset)
        keys, values = cache.update_and_fetch(k, v)
        y = ops.dispatch_sdpa(q, keys, values, cache=cache, scale=d ** -0.5, mask=None,
                              config=state["config"])
        y = ops.dispatch_attention_output(state["x"], y, state["gate"], state["out"])
        return {"y": y, "keys": keys, "values": values}
    if kind == "ffn":
        return ops.dispatch_ffn(state["x"], state["a"], state["norm"], state["mlp"],
                                mlp_type=_MLP)
    if kind == "sweep":
        state["graph"].replay()
        return state["out"]
    if kind == "w4":
        return ops.dispatch_linear(state["x"], state["layer"])
    if kind in ("w8a8", "w8_affine"):
        return state["layer"](state["x"])
    if kind == "w8_head":
        return sparkq.w8a16_per_channel(state["x"], *state["w"])
    if kind == "kv_decode":
        d = _HEADS[c["heads"]][2]
        return sparkq.int8_quantized_sdpa(state["q"], state["k"], state["v"], scale=d ** -0.5,
                                          group_size=c["group"],
                                          bits=8 if c["format"] == "s8" else _bits(c))
    d = _HEADS[c["heads"]][2]
    cache = state["cache"]
    cache.offset = c["n"] - c["l"]
    keys, values = cache.update_and_fetch(state["k_new"], state["v_new"])
    y = ops.dispatch_sdpa(state["q"], keys, values, cache=cache, scale=d ** -0.5,
                          mask=state["mask"], config=state["config"])
    return {"y": y, "keys": keys, "values": values}


# ---------------------------------------------------------------------------
# what a pass cannot do without
# ---------------------------------------------------------------------------

def _w4_bytes(n, k, group):
    return n * k // 2 + 4 * n * k // group


def work(case):
    c = case
    kind = c["kind"]
    e = 2
    if kind == "attention_block":
        h, hkv, d = _HEADS[c["heads"]]
        rows = (h + 2 * hkv) * d
        cached = 2 * hkv * (c["n"] + 1) * (d * c["bits"] // 8 + 4 * d // c["group"])
        return {"bytes": _w4_bytes(rows, 2560, c["group"]) + cached + e * h * 2560
                + 2560 * h * d + 4 * 2560 + 2 * e * 2560,
                "flops": 2 * rows * 2560 + 4 * h * d * (c["n"] + 1) + 2 * h * 2560
                + 2 * 2560 * h * d}
    if kind == "ffn":
        m, k, i = c["m"], c["k"], c["i"]
        return {"bytes": 3 * _w4_bytes(i, k, c["group"]) + 3 * m * k * e + k * e,
                "flops": 6 * m * k * i}
    if kind == "sweep":
        m = c["m"]
        one = [_PROJ[p] for p in ("qkv", "gate_up", "down")]
        return {"bytes": c["layers"] * sum(_w4_bytes(n, k, c["group"]) + e * m * n for n, k in one)
                + e * m * (2560 + 9728),
                "flops": c["layers"] * sum(2 * m * n * k for n, k in one)}
    if kind in ("w4", "w8a8", "w8_head", "w8_affine"):
        m, n, k = c["m"], c["n"], c["k"]
        eo = e
        if kind == "w4":
            w = _w4_bytes(n, k, c["group"])
        elif kind == "w8_affine":
            es = 4 if c["scales"] == "f32" else 2
            w, eo = n * k + 2 * es * n * k // c["group"], es
        else:
            w = n * k + 4 * n
        return {"bytes": w + e * m * k + eo * m * n, "flops": 2 * m * n * k}
    h, hkv, d = _HEADS[c["heads"]]
    if kind == "kv_decode":
        token = d + 2 if c["format"] == "s8" else d * _bits(c) // 8 + 4 * d // c["group"]
        return {"bytes": 2 * c["b"] * hkv * c["n"] * token + 2 * e * c["b"] * h * d,
                "flops": 4 * c["b"] * h * d * c["n"]}
    n, length = c["n"], c["l"]
    token = d * c["bits"] // 8 + 4 * d // c["group"]
    pairs = length * n - (length * (length - 1) // 2 if c["mask"] != "none" else 0)
    return {"bytes": 2 * hkv * n * token + 2 * hkv * length * (token + e * d) + 2 * e * h * length * d,
            "flops": 4 * h * d * pairs}


def tolerance(case):
    """16-bit results: two roundings of the same value differ by at most one
    unit in the last place; blocks of several roundings add up."""
    half = 8 if case["dtype"] == "bf16" else 1
    kind = case["kind"]
    if kind == "w8_affine" and case["scales"] == "f32":
        return {"rel": 1e-5}
    if kind == "attention_block":
        return {"rel": 2e-3 * half, "max": 0.3, "differ": 1e-3}
    if kind == "ffn":
        return {"rel": 1.2e-3 * half}
    if kind == "kv_prefill":
        return {"rel": 1e-3 * half, "differ": 1e-6}
    return {"rel": 8e-4 * half}


# ---------------------------------------------------------------------------
# the same in float64, without this repository's code
# ---------------------------------------------------------------------------

def _mm(x, raw):
    return x.double().reshape(-1, x.shape[-1]) @ _value(*raw).T


def _rope(x, base, pos):
    d = x.shape[-1]
    i = torch.arange(d // 2, device=x.device, dtype=torch.float64)
    a = pos * base ** (-2 * i / d)
    u, v = x[..., : d // 2], x[..., d // 2:]
    return torch.cat([u * a.cos() - v * a.sin(), u * a.sin() + v * a.cos()], -1)


def _attend(q, k, v, scale, mask=None):
    """q [B,H,L,D] over k, v [B,Hkv,N,D], one KV head at a time."""
    b, h, length, d = q.shape
    hkv = k.shape[1]
    y = torch.empty((b, h, length, v.shape[-1]), dtype=torch.float64, device=q.device)
    r = h // hkv
    for i in range(b):
        for j in range(hkv):
            qq = q[i, j * r:(j + 1) * r].double().reshape(r * length, d)
            s = (qq @ k[i, j].T).mul_(scale).reshape(r, length, -1)
            if mask is not None:
                s.masked_fill_(~mask, -math.inf)
            p = s.softmax(-1).reshape(r * length, -1)
            y[i, j * r:(j + 1) * r] = (p @ v[i, j]).reshape(r, length, -1)
    return y


def exact(case, seed):
    c, t = case, _inputs(case, seed)
    kind = c["kind"]
    if kind == "attention_block":
        h, hkv, d = _HEADS[c["heads"]]
        x = t["x"].double().reshape(2560)
        qkv = _value(*t["qkv"]) @ x
        q, k, v = qkv.split([h * d, hkv * d, hkv * d])
        q = _rope(q.reshape(1, h, 1, d), 500000.0, c["n"])
        k = _rope(k.reshape(1, hkv, 1, d), 500000.0, c["n"])
        new = [_value(*_affine(u.to(_TYPES[c["dtype"]]), c["bits"], c["group"],
                               _TYPES[c["dtype"]])) for u in (k, v.reshape(1, hkv, 1, d))]
        keys = torch.cat([_value(*t["k"]), new[0]], 2)
        values = torch.cat([_value(*t["v"]), new[1]], 2)
        y = _attend(q, keys, values, d ** -0.5).reshape(h, d)
        y = (y * torch.sigmoid(t["g"].double() @ x)[:, None]).reshape(h * d)
        w, s = t["out"]
        return {"y": (w.double() @ y * s.double()).reshape(1, 1, 2560),
                "keys": (None, None, None), "values": (None, None, None)}
    if kind == "ffn":
        hid = t["x"].double() + t["a"].double()
        nrm = hid * (hid.square().mean(-1, keepdim=True) + 1e-6).rsqrt() * t["norm"].double()
        gate = nrm @ _value(*t["gate"]).T
        act = gate * (1 + torch.erf(gate / math.sqrt(2))) / 2 * (nrm @ _value(*t["up"]).T)
        return hid + act @ _value(*t["down"]).T
    if kind == "sweep":
        return {p: torch.stack([_mm(t["x"][_PROJ[p][1]], w[p]) for w in t["w"]])
                for p in ("qkv", "gate_up", "down")}
    if kind in ("w4", "w8_affine"):
        return _mm(t["x"], t["w"]).reshape(1, c["m"], c["n"])
    if kind == "w8a8":
        x = t["x"].double().reshape(c["m"], c["k"])
        sa = (t["x"].float().abs().amax(-1) / 127).double().reshape(c["m"], 1)
        qa = (x / sa).round_().clamp_(-127, 127)
        return ((qa @ t["w"][0].double().T) * sa * t["w"][1].double()).reshape(1, c["m"], c["n"])
    if kind == "w8_head":
        x = t["x"].double().reshape(c["m"], c["k"])
        y = torch.cat([x @ part.double().T for part in t["w"][0].split(16384)], 1)
        return (y * t["w"][1].double()).reshape(1, c["m"], c["n"])
    h, hkv, d = _HEADS[c["heads"]]
    if kind == "kv_decode":
        if c["format"] == "s8":
            k, v = (r[0].double() * r[1].double()[..., None] for r in (t["k"], t["v"]))
        else:
            k, v = _value(*t["k"]), _value(*t["v"])
        return _attend(t["q"], k, v, d ** -0.5)
    new = [_value(*_affine(t[p], c["bits"], c["group"], _TYPES[c["dtype"]]))
           for p in ("k_new", "v_new")]
    keys = torch.cat([_value(*t["k"]), new[0]], 2) if "k" in t else new[0]
    values = torch.cat([_value(*t["v"]), new[1]], 2) if "v" in t else new[1]
    mask = t.get("mask")
    if c["mask"] == "causal":
        mask = torch.ones((c["l"], c["n"]), dtype=torch.bool, device=_DEV).tril(c["n"] - c["l"])
    return {"y": _attend(t["q"], keys, values, d ** -0.5, mask),
            "keys": (None, None, None), "values": (None, None, None)}
