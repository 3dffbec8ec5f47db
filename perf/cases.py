"""The work that programs give this framework, as cases whose time is measured.

A case is a dict of plain values; its "kind" says which part of a program it stands for:

  decode_layer   one transformer layer of a token-by-token generation step: norms, projections, KV-cache append,
                 attention against the cache, gated MLP.  A few rows of activations against all the layer's weights.
  prefill_layer  the same layer over a whole prompt (causal attention), which also fills the cache.
  prefill        causal attention over a prompt.
  chunk          a prompt chunk (or several new tokens) against a paged KV cache, aligned with the end of the keys.
  decode         one query token per sequence against long KV caches.
  padded         attention of an encoder batch padded to one length, with a key-padding or an additive mask.
  attn_train     attention forward and backward.
  linear_train   a linear layer's forward and backward with its bias gradient.
  loss           logSoftmax over a vocabulary and its backward.

Sizes of attention are those of bench.py's workloads and of the tests, and the ranges between them; a layer has 128 (or
64) columns per head and an MLP of about 2.7 to 3.5 times its width.
"""
import math

import torch

import tinytorch_amd as tt

_TYPES = {"f32": torch.float32, "f16": torch.float16, "bf16": torch.bfloat16}
_BYTES = {"f32": 4, "f16": 2, "bf16": 2}


def listed():
    return [
        # A chat with one user: a layer 4096 wide, 32 query and 8 KV heads; bound by its weights and by the launches.
        {"name": "decode_layer_1", "kind": "decode_layer", "dtype": "bf16", "B": 1, "width": 4096, "ffn": 14336,
         "Hq": 32, "Hkv": 8, "D": 128, "kv": 1500, "cache": 2048},
        # A server's step: 24 users with histories of different lengths on a layer of half the width.
        {"name": "decode_layer_24", "kind": "decode_layer", "dtype": "f16", "B": 24, "width": 2048, "ffn": 5632,
         "Hq": 16, "Hkv": 4, "D": 128, "kv": 3000, "cache": 4096},
        # A prompt of odd length through a whole layer.
        {"name": "prefill_layer_1999", "kind": "prefill_layer", "dtype": "bf16", "B": 1, "width": 4096, "ffn": 14336,
         "Hq": 32, "Hkv": 8, "D": 128, "L": 1999},
        # The attention of two prompts of 4096 tokens: bench.py's headline shape.
        {"name": "prefill_2x4096", "kind": "prefill", "dtype": "bf16", "B": 2, "Hq": 32, "Hkv": 8, "L": 4096, "D": 128},
        # Chunked prefill: the next 500 tokens of three conversations in a paged cache.
        {"name": "chunk_500_paged", "kind": "chunk", "dtype": "bf16", "B": 3, "Hq": 32, "Hkv": 8, "L": 500, "kv": 6000,
         "D": 128, "page": 64},
        # Batched generation with a long context: bench.py's decode shape, the most bytes that a call streams.
        {"name": "decode_64x8192", "kind": "decode", "dtype": "bf16", "B": 64, "Hq": 32, "Hkv": 8, "kv": 8192,
         "ragged": False, "D": 128, "page": 0},
        # An encoder's batch of sentences, padded: head_dim 64, as many KV as query heads, odd length.
        {"name": "padded_16x197", "kind": "padded", "dtype": "f16", "B": 16, "H": 12, "L": 197, "D": 64, "mask": "keys"},
        # One layer's attention in training at the headline shape.
        {"name": "attn_train_2x4096", "kind": "attn_train", "dtype": "bf16", "B": 2, "Hq": 32, "Hkv": 8, "L": 4096,
         "D": 128, "causal": True},
        # The smallest attention of bench.py, forward and backward in the default type: bound by latency.
        {"name": "attn_train_f32_128", "kind": "attn_train", "dtype": "f32", "B": 1, "Hq": 4, "Hkv": 4, "L": 128, "D": 64,
         "causal": True},
        # The QKV projection in training.
        {"name": "linear_train_8192", "kind": "linear_train", "dtype": "bf16", "M": 8192, "K": 4096, "N": 6144},
        # A small classifier's first layer in the default type; sizes that no tile divides.
        {"name": "linear_train_f32_64", "kind": "linear_train", "dtype": "f32", "M": 64, "K": 784, "N": 500},
        # The loss of a training step of 4096 tokens over a vocabulary of 32000.
        {"name": "loss_4096x32000", "kind": "loss", "dtype": "bf16", "rows": 4096, "cols": 32000},
    ]


# ---- drawn cases ---------------------------------------------------------------------------------------------------

#: What a drawn case may cost (work() priced at the rates below): the dearest listed case's figure, rounded down.
_MOST_SECONDS = 7e-4


def _seconds(case):
    w = work(case)
    return max(w["bytes"] / 6e12, w["flops"] / (1.2e14 if case["dtype"] == "f32" else 1.5e15))


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _layer(rng, dtype):
    width = rng.choice([1024, 1536, 2048, 3072] if dtype == "f32" else [1024, 1536, 2048, 3072, 4096, 5120])
    D = rng.choice([64, 128, 128])
    heads = width // D
    group = rng.choice([g for g in (1, 2, 4, 7, 8) if heads % g == 0])
    return {"width": width, "ffn": int(width * rng.uniform(2.6, 3.5)) // 64 * 64, "Hq": heads, "Hkv": heads // group, "D": D}


def _heads(rng):
    Hkv = rng.choice([1, 2, 4, 8, 8])
    return Hkv * rng.choice([1, 2, 4, 4, 7, 8]), Hkv


def _drawn(rng):
    kind = rng.choice(["decode_layer", "decode_layer", "prefill_layer", "prefill", "chunk", "decode", "padded", "attn_train",
                       "attn_train", "linear_train", "linear_train", "loss"])
    c = {"kind": kind, "dtype": rng.choice(["bf16", "bf16", "bf16", "f16", "f16", "f32"])}
    if kind == "decode_layer":
        c["B"] = _log(rng, 1, 64)
        c.update(_layer(rng, c["dtype"]))
        c["kv"] = _log(rng, 128, 8192)
        c["cache"] = -(-c["kv"] // 1024) * 1024
    elif kind == "prefill_layer":
        c["B"] = rng.choice([1, 1, 2, 4])
        c.update(_layer(rng, c["dtype"]))
        c["L"] = _log(rng, 64, 4096)
    elif kind == "prefill":
        c["B"] = rng.choice([1, 2, 4])
        c["Hq"], c["Hkv"] = _heads(rng)
        c["L"] = _log(rng, 128, 16384)
        c["D"] = rng.choice([64, 80, 128, 128])
    elif kind == "chunk":
        c["B"] = _log(rng, 1, 16)
        c["Hq"], c["Hkv"] = _heads(rng)
        c["L"] = _log(rng, 2, 1024)
        c["kv"] = max(c["L"], _log(rng, 256, 16384))
        c["D"] = rng.choice([64, 128, 128])
        c["page"] = rng.choice([64, 128, 256])
    elif kind == "decode":
        c["B"] = _log(rng, 1, 64)
        c["Hq"], c["Hkv"] = _heads(rng)
        c["kv"] = _log(rng, 128, 65536)
        c["ragged"] = rng.random() < 0.5
        c["D"] = rng.choice([64, 128, 128])
        c["page"] = rng.choice([0, 0, 64, 256])
    elif kind == "padded":
        c["B"] = _log(rng, 1, 64)
        c["H"] = rng.choice([4, 8, 12, 16])
        c["L"] = _log(rng, 16, 1024)
        c["D"] = rng.choice([32, 64, 64, 80, 128])
        c["mask"] = rng.choice(["keys", "keys", "add"])
    elif kind == "attn_train":
        c["B"] = rng.choice([1, 2, 4, 8])
        c["Hq"], c["Hkv"] = _heads(rng)
        c["L"] = _log(rng, 64, 4096)
        c["D"] = rng.choice([64, 64, 128, 128])
        c["causal"] = rng.random() < 0.75
    elif kind == "linear_train":
        c["M"] = _log(rng, 16, 8192)
        step = rng.choice([1, 8, 64, 64])  # sizes of a real layer are mostly multiples of 64; some are not
        c["K"] = max(step, _log(rng, 64, 8192) // step * step)
        c["N"] = max(step, _log(rng, 16, 8192) // step * step)
    else:
        c["rows"] = _log(rng, 8, 8192)
        c["cols"] = _log(rng, 500, 130000)
    return c


def draw(rng):
    while True:
        c = _drawn(rng)
        if _seconds(c) <= _MOST_SECONDS:
            return c


# ---- inputs --------------------------------------------------------------------------------------------------------

class _Maker:
    """Device tensors of one case, from the seed alone."""

    def __init__(self, case, seed):
        self.dtype = _TYPES[case["dtype"]]
        self.gen = torch.Generator(device="cuda").manual_seed(seed)

    def normal(self, *shape, mul=1.0):
        out = torch.empty(shape, dtype=self.dtype, device="cuda")
        flat = out.view(-1)
        for lo in range(0, flat.numel(), 1 << 27):
            part = flat[lo:lo + (1 << 27)]
            part.copy_(torch.randn(part.numel(), generator=self.gen, device="cuda").mul_(mul))
        return out

    def weight(self, n, k):
        return self.normal(n, k, mul=1.0 / math.sqrt(k))

    def gain(self, n):
        return (1.0 + 0.1 * torch.randn(n, generator=self.gen, device="cuda")).to(self.dtype)

    def lengths(self, B, lo, hi):
        """B lengths from lo to hi, the longest being hi."""
        n = torch.randint(lo, hi + 1, (B,), generator=self.gen, device="cuda", dtype=torch.int32)
        n[0] = hi
        return n

    def pages(self, B, per_entry):
        """A block table whose pages lie scattered over the pool, as after a while of serving."""
        return torch.randperm(B * per_entry, generator=self.gen, device="cuda").to(torch.int32).view(B, per_entry)


def _layer_weights(make, c):
    width, cols = c["width"], (c["Hq"] + 2 * c["Hkv"]) * c["D"]
    return {"attn_norm": make.gain(width), "qkv": make.weight(cols, width), "o": make.weight(width, c["Hq"] * c["D"]),
            "mlp_norm": make.gain(width), "gate_up": make.weight(2 * c["ffn"], width), "down": make.weight(width, c["ffn"])}


def prepare(case, seed):
    c, make = case, _Maker(case, seed)
    s = {"case": case}
    kind = c["kind"]
    if kind == "decode_layer":
        s["w"] = _layer_weights(make, c)
        s["x"] = make.normal(c["B"], c["width"])
        s["kc"] = make.normal(c["B"], c["Hkv"], c["cache"], c["D"])
        s["vc"] = make.normal(c["B"], c["Hkv"], c["cache"], c["D"])
        s["lens"] = make.lengths(c["B"], max(1, c["kv"] // 3), c["kv"])  # keys of each sequence with the new one
        s["at"] = s["lens"] - 1
    elif kind == "prefill_layer":
        s["w"] = _layer_weights(make, c)
        s["x"] = make.normal(c["B"] * c["L"], c["width"])
        s["kc"] = torch.zeros(c["B"], c["Hkv"], -(-c["L"] // 256) * 256, c["D"], dtype=make.dtype, device="cuda")
        s["vc"] = torch.zeros_like(s["kc"])
    elif kind == "prefill":
        s["q"] = make.normal(c["B"], c["Hq"], c["L"], c["D"])
        s["k"], s["v"] = (make.normal(c["B"], c["Hkv"], c["L"], c["D"]) for _ in "kv")
    elif kind in ("chunk", "decode"):
        rows = c.get("L", 1)
        s["q"] = make.normal(c["B"], c["Hq"], rows, c["D"])
        if c["page"]:
            per = -(-c["kv"] // c["page"])
            s["table"] = make.pages(c["B"], per)
            s["k"], s["v"] = (make.normal(c["B"] * per, c["Hkv"], c["page"], c["D"]) for _ in "kv")
        else:
            s["table"] = None
            s["k"], s["v"] = (make.normal(c["B"], c["Hkv"], c["kv"], c["D"]) for _ in "kv")
        whole = kind == "decode" and not c["ragged"]
        s["lens"] = None if whole and not c["page"] else make.lengths(c["B"], c["kv"] if whole else max(rows, c["kv"] // 3), c["kv"])
    elif kind == "padded":
        s["q"], s["k"], s["v"] = (make.normal(c["B"], c["H"], c["L"], c["D"]) for _ in "qkv")
        if c["mask"] == "keys":
            n = make.lengths(c["B"], max(1, c["L"] // 4), c["L"])
            s["mask"] = (torch.arange(c["L"], device="cuda")[None, :] < n[:, None]).view(c["B"], 1, 1, c["L"])
        else:
            s["mask"] = make.normal(c["H"], c["L"], c["L"])
    elif kind == "attn_train":
        s["q"] = make.normal(c["B"], c["Hq"], c["L"], c["D"])
        s["k"], s["v"] = (make.normal(c["B"], c["Hkv"], c["L"], c["D"]) for _ in "kv")
        s["grad"] = make.normal(c["B"], c["Hq"], c["L"], c["D"])
    elif kind == "linear_train":
        s["x"], s["w"], s["b"] = make.normal(c["M"], c["K"]), make.weight(c["N"], c["K"]), make.normal(c["N"])
        s["grad"] = make.normal(c["M"], c["N"])
    else:
        s["x"] = make.normal(c["rows"], c["cols"], mul=2.0)
        s["grad"] = make.normal(c["rows"], c["cols"], mul=1.0 / c["rows"])
    return s


# ---- one pass ------------------------------------------------------------------------------------------------------

def _layer_pass(s, B, L):
    """One transformer layer over B x L tokens; returns its two streams (the MLP's output and the residual)."""
    c, w = s["case"], s["w"]
    Hq, Hkv, D = c["Hq"], c["Hkv"], c["D"]
    residual = s["x"].clone()  # the layer adds to its residual stream in place
    h = tt.rmsNorm(residual, [c["width"]], w["attn_norm"], 1e-5)
    qkv = tt.linear(h, w["qkv"]).view(B, L, Hq + 2 * Hkv, D).transpose(1, 2)
    q, k, v = qkv[:, :Hq], qkv[:, Hq:Hq + Hkv], qkv[:, Hq + Hkv:]
    if c["kind"] == "decode_layer":
        tt.kvCacheAppend(s["kc"], s["vc"], k, v, s["at"])
        a = tt.sdpAttention(q, s["kc"], s["vc"], kvLens=s["lens"])
    else:
        tt.kvCacheAppend(s["kc"], s["vc"], k, v, 0)
        a = tt.sdpAttention(q, k, v, isCausal=True)
    h = tt.linear(a.transpose(1, 2).reshape(B * L, Hq * D), w["o"])
    tt.fusedAddRmsNorm(h, residual, w["mlp_norm"], 1e-5)
    return tt.linear(tt.siluMul(tt.linear(h, w["gate_up"])), w["down"]), residual


def run(state):
    s = state
    c = s["case"]
    kind = c["kind"]
    if kind in ("decode_layer", "prefill_layer"):
        h, residual = _layer_pass(s, c["B"], c.get("L", 1))
        return h, residual, s["kc"], s["vc"]
    if kind == "prefill":
        return tt.sdpAttention(s["q"], s["k"], s["v"], isCausal=True)
    if kind == "chunk":
        return tt.sdpAttention(s["q"], s["k"], s["v"], isCausal=True, kvLens=s["lens"], causalAlign="bottom-right",
                               blockTable=s["table"])
    if kind == "decode":
        return tt.sdpAttention(s["q"], s["k"], s["v"], kvLens=s["lens"], blockTable=s["table"])
    if kind == "padded":
        return tt.sdpAttention(s["q"], s["k"], s["v"], attnMask=s["mask"])
    if kind == "attn_train":
        out = tt.sdpAttention(s["q"], s["k"], s["v"], isCausal=c["causal"])
        return (out,) + tuple(tt.sdpAttentionBackward(s["grad"], s["q"], s["k"], s["v"], out, isCausal=c["causal"]))
    if kind == "linear_train":
        return (tt.linear(s["x"], s["w"], s["b"]),) + tuple(tt.linearBackward(s["grad"], s["x"], s["w"]))
    y = tt.logSoftmax(s["x"], -1)
    return y, tt.logSoftmaxBackward(s["grad"], y, -1)


# ---- what a pass cannot do without, and how exact it is --------------------------------------------------------------

def _causal_pairs(L):
    return L * (L + 1) / 2


def work(case):
    c, e = case, _BYTES[case["dtype"]]
    kind = c["kind"]
    if kind in ("decode_layer", "prefill_layer"):
        T = c["B"] * c.get("L", 1)
        weights = c["width"] * ((2 * c["Hq"] + 2 * c["Hkv"]) * c["D"] + 3 * c["ffn"])
        # keys in the cache: a third of the range is the shortest history, so two thirds of it on average
        keys = c["B"] * c["kv"] * 2 / 3 if kind == "decode_layer" else c["B"] * _causal_pairs(c["L"])
        rows = c["B"] * c["kv"] * 2 / 3 if kind == "decode_layer" else c["B"] * c["L"]
        return {"bytes": e * (weights + 3 * T * c["width"] + 2 * rows * c["Hkv"] * c["D"]),
                "flops": 2 * T * weights + 4 * keys * c["Hq"] * c["D"]}
    if kind == "prefill":
        n = c["B"] * c["L"] * c["D"]
        return {"bytes": e * n * 2 * (c["Hq"] + c["Hkv"]), "flops": 4 * c["B"] * c["Hq"] * c["D"] * _causal_pairs(c["L"])}
    if kind in ("chunk", "decode"):
        L = c.get("L", 1)
        kv = c["kv"] if kind == "decode" and not c["ragged"] else (max(L, c["kv"] // 3) + c["kv"]) / 2
        pairs = L * (kv - (L - 1) / 2)
        return {"bytes": e * c["B"] * c["D"] * (2 * L * c["Hq"] + 2 * kv * c["Hkv"]), "flops": 4 * c["B"] * c["Hq"] * c["D"] * pairs}
    if kind == "padded":
        n = c["B"] * c["H"] * c["L"]
        mask = c["B"] * c["L"] if c["mask"] == "keys" else e * c["H"] * c["L"] ** 2
        return {"bytes": 4 * e * n * c["D"] + mask, "flops": 4 * n * c["L"] * c["D"]}
    if kind == "attn_train":
        pairs = _causal_pairs(c["L"]) if c["causal"] else c["L"] ** 2
        n = c["B"] * c["L"] * c["D"]
        # two products forward and five backward; q, k, v, grad in, out and three gradients out
        return {"bytes": e * n * (4 * c["Hq"] + 4 * c["Hkv"]), "flops": 14 * c["B"] * c["Hq"] * c["D"] * pairs}
    if kind == "linear_train":
        M, K, N = c["M"], c["K"], c["N"]
        return {"bytes": e * (2 * M * K + 2 * N * K + 2 * M * N + 2 * N), "flops": 6 * M * K * N}
    n = c["rows"] * c["cols"]
    return {"bytes": e * 4 * n, "flops": 8 * n}


def tolerance(case):
    # the rounding of the element type, through the few roundings that a chain of these calls has
    return {"rel": {"f32": 2e-5, "f16": 3e-3, "bf16": 1e-2}[case["dtype"]]}
