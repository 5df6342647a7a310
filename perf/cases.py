"""The work that programs using hexmi give it, as measurable cases.

Each case is one pass through the package's public operators, called as a program calls them: device tensors in,
fresh device tensors out (or a cache updated in place), nothing synchronised. A case is a dict of plain values whose
"op" says which part of the package it stands for:

  norm      RMSNorm / LayerNorm over [rows, cols] activations
  softmax   softmax over the rows of [rows, cols]
  linear    dense 16-bit matmul, B stored [K, N] ("nn") or [N, K] ("nt": x @ W.T), with or without bias and residual
  w8a16     16-bit activations against int8 weights, with or without zero points
  flash     self-attention over [Z, H, S, D], causal or not
  attend    attention of Sq rows over Skv keys with or without an additive mask (a prompt taken in pieces, padding)
  block     one GPT-2 style transformer block over a batch of prompts (prefill)
  decode    one decoder layer with int8 weights for one new token of each sequence of a batch (decode)

listed() are fixed sizes, draw() picks others from the ranges they stand for. The package has no backward pass.
"""
import math
import os
import sys

import torch

sys.path.insert(0, os.path.join(os.getcwd(), "hexagon-mlir_amd"))
import hexmi  # noqa: E402

_DTYPES = {"f16": torch.float16, "bf16": torch.bfloat16, "f32": torch.float32}


def listed():
    return [
        # The smallest calls: the layer norm inside one block of a 768-wide model over a 512-token prompt. Host time
        # per call and one launch are all there is.
        {"name": "layer_norm_f16_512x768", "op": "norm", "kind": "layer", "rows": 512, "cols": 768, "dtype": "f16"},
        # A norm over the activations of a large batch (the package's own benchmark configuration).
        {"name": "rms_norm_f16_8192x4096", "op": "norm", "kind": "rms", "rows": 8192, "cols": 4096, "dtype": "f16"},
        # Probabilities over a 50257-token vocabulary: rows that are no multiple of anything.
        {"name": "softmax_f16_1024x50257", "op": "softmax", "rows": 1024, "cols": 50257, "dtype": "f16"},
        # The square matmul of the benchmark configuration.
        {"name": "gemm_f16_nn_4096", "op": "linear", "M": 4096, "N": 4096, "K": 4096, "dtype": "f16", "layout": "nn",
         "bias": False, "residual": False},
        # Logits of a ragged prompt against a tied [vocabulary, 768] embedding.
        {"name": "linear_bf16_nt_1021x50257x768", "op": "linear", "M": 1021, "N": 50257, "K": 768, "dtype": "bf16",
         "layout": "nt", "bias": False, "residual": False},
        # The down projection of a 4096 / 11008 feed-forward for a batch of 32 sequences decoding together.
        {"name": "linear_f16_nt_32x4096x11008", "op": "linear", "M": 32, "N": 4096, "K": 11008, "dtype": "f16",
         "layout": "nt", "bias": False, "residual": True},
        # Weight-only int8: decode batch and short prompt against the up projection (benchmark configurations).
        {"name": "w8a16_16x11008x4096", "op": "w8a16", "M": 16, "N": 11008, "K": 4096, "zero_points": False},
        {"name": "w8a16_256x11008x4096", "op": "w8a16", "M": 256, "N": 11008, "K": 4096, "zero_points": False},
        # Causal attention over long prompts (benchmark configuration).
        {"name": "flash_f16_causal_4x32x4096x128", "op": "flash", "Z": 4, "H": 32, "S": 4096, "D": 128,
         "dtype": "f16", "causal": True},
        # The next 509 tokens of a prompt against the 2555 keys so far, causal by mask, 32 heads.
        {"name": "attend_f16_32x509x2555x128", "op": "attend", "B": 32, "Sq": 509, "Skv": 2555, "D": 128,
         "dtype": "f16", "mask": True},
        # Prefill of one GPT-2 style block, two prompts of 1000 tokens.
        {"name": "block_bf16_2x1000x768", "op": "block", "B": 2, "S": 1000, "heads": 12, "dtype": "bf16"},
        # Decode of one layer, 16 sequences with up to 2048 tokens behind them.
        {"name": "decode_16x2048x4096", "op": "decode", "B": 16, "context": 2048, "heads": 32, "ffn": 11008},
    ]


def _log(rng, lo, hi):
    """A whole number of [lo, hi], even over the logarithm."""
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def _rounded(rng, value, *steps):
    """value, or its nearest multiple of one of steps: sizes in use are often, not always, multiples of something."""
    step = rng.choice(steps)
    return max(step, value // step * step)


# A drawn case does at most about as much as the largest listed one of its kind.
_MOST_FLOPS = {"flash": 5.5e11, "attend": 2.2e10}
_MOST_BYTES = {"flash": 5.4e8, "decode": 7.4e8}


def draw(rng):
    while True:
        case = _draw(rng)
        w = work(case)
        if w["flops"] <= _MOST_FLOPS.get(case["op"], 1.4e11) and w["bytes"] <= _MOST_BYTES.get(case["op"], 2.2e8):
            return case


def _draw(rng):
    op = rng.choice(("norm", "softmax", "linear", "linear", "w8a16", "flash", "attend", "block", "decode"))
    if op == "norm":
        return {"op": op, "kind": rng.choice(("rms", "layer")), "rows": _log(rng, 1, 16384),
                "cols": _rounded(rng, _log(rng, 256, 12288), 1, 8, 64, 256), "dtype": rng.choice(("f16", "bf16", "f32"))}
    if op == "softmax":
        return {"op": op, "rows": _log(rng, 1, 8192), "cols": _rounded(rng, _log(rng, 64, 65536), 1, 1, 8, 64),
                "dtype": rng.choice(("f16", "bf16", "f32"))}
    if op == "linear":
        layout = rng.choice(("nn", "nt"))
        return {"op": op, "M": _rounded(rng, _log(rng, 1, 8192), 1, 1, 16, 128),
                "N": _rounded(rng, _log(rng, 256, 51200), 1, 8, 64, 128), "K": _rounded(rng, _log(rng, 256, 12288), 8, 64, 64),
                "dtype": rng.choice(("f16", "bf16")), "layout": layout, "bias": rng.random() < 0.4,
                "residual": rng.random() < 0.3}
    if op == "w8a16":
        return {"op": op, "M": _rounded(rng, _log(rng, 1, 1024), 1, 1, 16), "N": _rounded(rng, _log(rng, 512, 14336), 1, 16, 128),
                "K": _rounded(rng, _log(rng, 512, 14336), 16, 64, 128), "zero_points": rng.random() < 0.25}
    if op == "flash":
        return {"op": op, "Z": _log(rng, 1, 8), "H": rng.choice((8, 12, 16, 32, 40)),
                "S": _rounded(rng, _log(rng, 64, 8192), 1, 16, 128), "D": rng.choice((64, 128, 128, 80, 96, 256)),
                "dtype": rng.choice(("f16", "bf16")), "causal": rng.random() < 0.75}
    if op == "attend":
        Sq = _log(rng, 1, 2048)
        return {"op": op, "B": _log(rng, 8, 256), "Sq": Sq, "Skv": _rounded(rng, max(Sq, _log(rng, 64, 8192)), 1, 8, 64),
                "D": rng.choice((64, 128)), "dtype": rng.choice(("f16", "bf16")), "mask": rng.random() < 0.6}
    if op == "block":
        return {"op": op, "B": _log(rng, 1, 8), "S": _log(rng, 16, 1024), "heads": rng.choice((8, 12, 16, 20, 25)),
                "dtype": rng.choice(("f16", "bf16"))}
    heads = rng.choice((16, 24, 32, 40))
    return {"op": op, "B": _log(rng, 1, 64), "context": _log(rng, 64, 8192), "heads": heads,
            "ffn": _rounded(rng, heads * 128 * 8 // 3, 128, 256)}


class _Random:
    """Seeded inputs, made on the GPU."""

    def __init__(self, seed):
        self.g = torch.Generator(device="cuda").manual_seed(seed)

    def normal(self, *shape, dtype, std=1.0, mean=0.0):
        return torch.randn(*shape, generator=self.g, device="cuda").mul_(std).add_(mean).to(dtype)

    def uniform(self, *shape, dtype, lo=-1.0, hi=1.0):
        return torch.rand(*shape, generator=self.g, device="cuda").mul_(hi - lo).add_(lo).to(dtype)

    def int8(self, *shape, lo=-127, hi=128):
        return torch.randint(lo, hi, shape, generator=self.g, device="cuda", dtype=torch.int8)

    def w8(self, N, K, rms=1.0):
        """int8 weights with a scale per channel that keep unit-variance activations at about `rms`."""
        mid = rms / (73.0 * math.sqrt(K))
        return self.int8(N, K), self.uniform(N, dtype=torch.float16, lo=0.5 * mid, hi=1.5 * mid)


def prepare(case, seed):
    r, op = _Random(seed), case["op"]
    if op == "norm":
        dt, C = _DTYPES[case["dtype"]], case["cols"]
        s = {"x": r.normal(case["rows"], C, dtype=dt), "weight": r.normal(C, dtype=dt, std=0.1, mean=1.0)}
        if case["kind"] == "layer":
            s["bias"] = r.normal(C, dtype=dt, std=0.1)
    elif op == "softmax":
        s = {"x": r.normal(case["rows"], case["cols"], dtype=_DTYPES[case["dtype"]], std=2.0)}
    elif op == "linear":
        dt, M, N, K = _DTYPES[case["dtype"]], case["M"], case["N"], case["K"]
        s = {"a": r.uniform(M, K, dtype=dt), "b": r.uniform(*((N, K) if case["layout"] == "nt" else (K, N)), dtype=dt),
             "trans_b": case["layout"] == "nt",
             "bias": r.normal(N, dtype=dt) if case["bias"] else None,
             "residual": r.normal(M, N, dtype=dt) if case["residual"] else None}
    elif op == "w8a16":
        M, N, K = case["M"], case["N"], case["K"]
        s = {"a": r.normal(M, K, dtype=torch.float16), "w": r.int8(N, K),
             "scales": r.uniform(N, dtype=torch.float16, lo=0.001, hi=0.02),
             "zero_points": r.int8(N, lo=-20, hi=20) if case["zero_points"] else None}
    elif op == "flash":
        dt, shape = _DTYPES[case["dtype"]], (case["Z"], case["H"], case["S"], case["D"])
        s = {n: r.normal(*shape, dtype=dt) for n in ("q", "k", "v")}
        s["sm_scale"], s["causal"] = 1.0 / math.sqrt(case["D"]), case["causal"]
    elif op == "attend":
        dt, B, Sq, Skv, D = _DTYPES[case["dtype"]], case["B"], case["Sq"], case["Skv"], case["D"]
        s = {"q": r.normal(B, Sq, D, dtype=dt), "k": r.normal(B, Skv, D, dtype=dt), "v": r.normal(B, Skv, D, dtype=dt),
             "mask": None}
        if case["mask"]:                                     # query i stands at key Skv - Sq + i
            after = torch.arange(Skv, device="cuda")[None, :] > torch.arange(Sq, device="cuda")[:, None] + (Skv - Sq)
            s["mask"] = torch.zeros(Sq, Skv, device="cuda", dtype=dt).masked_fill_(after, -math.inf).expand(B, Sq, Skv).contiguous()
    elif op == "block":
        dt, B, S, H = _DTYPES[case["dtype"]], case["B"], case["S"], case["heads"]
        E = 64 * H
        s = {"shape": (B, S, H), "x": r.normal(B * S, E, dtype=dt)}
        for n in ("ln1", "ln2"):
            s[n] = (r.normal(E, dtype=dt, std=0.1, mean=1.0), r.normal(E, dtype=dt, std=0.1))
        for n, rows, cols in (("qkv", E, 3 * E), ("o", E, E), ("fc", E, 4 * E), ("proj", 4 * E, E)):
            s[n] = (r.normal(rows, cols, dtype=dt, std=0.02), r.normal(cols, dtype=dt, std=0.02))
    else:
        B, T, H, F = case["B"], case["context"], case["heads"], case["ffn"]
        E = 128 * H
        s = {"shape": (B, H), "x": r.normal(B, E, dtype=torch.float16),
             "norm1": r.normal(E, dtype=torch.float16, std=0.1, mean=1.0),
             "norm2": r.normal(E, dtype=torch.float16, std=0.1, mean=1.0),
             "k_cache": r.normal(B * H, T, 128, dtype=torch.float16), "v_cache": r.normal(B * H, T, 128, dtype=torch.float16)}
        for n, N, K in (("qkv", 3 * E, E), ("o", E, E), ("gate", F, E), ("up", F, E), ("down", E, F)):
            s[n] = r.w8(N, K)
        # the prompts are padded on the left, so that every new token stands at the caches' last place
        pad = torch.randint(0, T // 2 + 1, (B,), generator=r.g, device="cuda")
        masked = torch.arange(T, device="cuda")[None, :] < pad[:, None]
        s["mask"] = (torch.zeros(B, T, device="cuda", dtype=torch.float16).masked_fill_(masked, -math.inf)
                     .repeat_interleave(H, 0).reshape(B * H, 1, T).contiguous())
    s["op"] = op
    return s


def run(s):
    op = s["op"]
    if op == "norm":
        if "bias" in s:
            return hexmi.layer_norm(s["x"], s["weight"], s["bias"], 1e-5)
        return hexmi.rms_norm(s["x"], s["weight"], 1e-5)
    if op == "softmax":
        return hexmi.softmax(s["x"])
    if op == "linear":
        return hexmi.matmul(s["a"], s["b"], trans_b=s["trans_b"], bias=s["bias"], residual=s["residual"])
    if op == "w8a16":
        return hexmi.w8a16_matmul(s["a"], s["w"], s["scales"], zero_points=s["zero_points"])
    if op == "flash":
        return hexmi.flash_attention(s["q"], s["k"], s["v"], s["sm_scale"], s["causal"])
    if op == "attend":
        return hexmi.attention(s["q"], s["k"], s["v"], s["mask"])
    return _block(s) if op == "block" else _decode(s)


def _block(s):
    B, S, H = s["shape"]
    x, E = s["x"], 64 * H
    h = hexmi.layer_norm(x, *s["ln1"], 1e-5)
    qkv = hexmi.matmul(h, s["qkv"][0], bias=s["qkv"][1])
    q, k, v = (t.view(B, S, H, 64).transpose(1, 2) for t in qkv.split(E, dim=-1))
    a = hexmi.flash_attention(q, k, v, 0.125, True)
    a = a.transpose(1, 2).reshape(B * S, E)
    x = hexmi.matmul(a, s["o"][0], bias=s["o"][1], residual=x)
    h = hexmi.layer_norm(x, *s["ln2"], 1e-5)
    m = hexmi.gelu(hexmi.matmul(h, s["fc"][0], bias=s["fc"][1]))
    return {"x": hexmi.matmul(m, s["proj"][0], bias=s["proj"][1], residual=x), "k": k, "v": v}


def _decode(s):
    B, H = s["shape"]
    x, E = s["x"], 128 * H
    h = hexmi.rms_norm(x, s["norm1"], 1e-5)
    qkv = hexmi.w8a16_matmul(h, *s["qkv"])
    q, k, v = (t.reshape(B * H, 128) for t in qkv.split(E, dim=-1))
    s["k_cache"][:, -1] = k
    s["v_cache"][:, -1] = v
    a = hexmi.attention(q.unsqueeze(1), s["k_cache"], s["v_cache"], s["mask"]).reshape(B, E)
    x = hexmi.binary("add", x, hexmi.w8a16_matmul(a, *s["o"]))
    h = hexmi.rms_norm(x, s["norm2"], 1e-5)
    m = hexmi.binary("mul", hexmi.silu(hexmi.w8a16_matmul(h, *s["gate"])), hexmi.w8a16_matmul(h, *s["up"]))
    return {"x": hexmi.binary("add", x, hexmi.w8a16_matmul(m, *s["down"])), "k_cache": s["k_cache"], "v_cache": s["v_cache"]}


def work(case):
    op, size = case["op"], 4 if case.get("dtype") == "f32" else 2
    if op in ("norm", "softmax"):
        n = case["rows"] * case["cols"]
        vectors = {"rms": 1, "layer": 2}.get(case.get("kind"), 0)
        return {"bytes": size * (2 * n + vectors * case["cols"]), "flops": 5 * n}
    if op == "linear":
        M, N, K = case["M"], case["N"], case["K"]
        return {"bytes": 2 * (M * K + N * K + M * N * (2 if case["residual"] else 1) + (N if case["bias"] else 0)),
                "flops": 2 * M * N * K}
    if op == "w8a16":
        M, N, K = case["M"], case["N"], case["K"]
        return {"bytes": N * K + 2 * (M * K + M * N + N) + (N if case["zero_points"] else 0), "flops": 2 * M * N * K}
    if op == "flash":
        n = case["Z"] * case["H"] * case["S"] * case["D"]
        pairs = (case["S"] + 1) / 2 if case["causal"] else case["S"]
        return {"bytes": 2 * 4 * n, "flops": 4 * n * pairs}
    if op == "attend":
        B, Sq, Skv, D = case["B"], case["Sq"], case["Skv"], case["D"]
        return {"bytes": 2 * B * (2 * Sq * D + 2 * Skv * D + (Sq * Skv if case["mask"] else 0)),
                "flops": 4 * B * Sq * Skv * D}
    if op == "block":
        T, S, E = case["B"] * case["S"], case["S"], 64 * case["heads"]
        return {"bytes": 2 * (12 * E * E + 13 * E + 4 * T * E), "flops": 24 * T * E * E + 2 * T * (S + 1) * E}
    B, T, E, F = case["B"], case["context"], 128 * case["heads"], case["ffn"]
    weights = 4 * E * E + 3 * E * F
    return {"bytes": weights + 2 * (5 * E + 2 * F) + 2 * B * (2 * T * E + 4 * E + T * case["heads"]),
            "flops": 2 * B * weights + 4 * B * T * E}


def tolerance(case):
    """Four times the error against the same pass in 64 bits, over the listed cases and forty drawn ones.

    A result rounded to f16 shows rel 2.1e-4 and max 4.9e-4 by that rounding alone, bf16 1.7e-3 and 3.9e-3, and f32
    1.0e-7 and 2.3e-7. Attention also rounds its probabilities (f16 2.9e-4 and 4.6e-3, bf16 2.3e-3 and 2.0e-2), the
    layers round between their operators (block f16 3.7e-4 and 1.5e-3, bf16 2.8e-3 and 1.2e-2; decode 4.7e-4 and
    2.4e-3)."""
    op, bf16 = case["op"], case.get("dtype") == "bf16"
    if case.get("dtype") == "f32":
        return {"rel": 4e-7, "max": 1e-6}
    if op in ("flash", "attend"):
        return {"rel": 9e-3, "max": 8e-2} if bf16 else {"rel": 1.2e-3, "max": 1.8e-2}
    if op == "block":
        return {"rel": 1.1e-2, "max": 5e-2} if bf16 else {"rel": 1.5e-3, "max": 6e-3}
    if op == "decode":
        return {"rel": 1.9e-3, "max": 1e-2}
    return {"rel": 7e-3, "max": 1.6e-2} if bf16 else {"rel": 8e-4, "max": 2e-3}
