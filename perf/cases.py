"""The work a model with packed weights has this package do, as cases that can be timed and compared.

A case is a dict of plain values; its `kind` names the layer it goes through:

  linear      one `QuantizedLinear` (nuvec_amd.layers), with or without a bias
  mlp         the gated MLPs of `layers` blocks of a model, gate and up projections fused at load time
  head        a tied table: the rows of a step's tokens (`QuantizedEmbedding`), then the logits of its last states
  moe         the mixture-of-experts MLPs of `layers` blocks, router included (`MoeMlp`)
  attention   attention of new queries over a quantized key / value cache (`layers.quantized_attention`)
  codec       a dense weight quantized, and the packed one dequantized (`quantize`, `dequantize`)

`listed()` holds one case for each way these are met in earnest, `draw()` takes others from the same ranges: one token to
a 2048-token prompt, every packed format, the three element types, sizes that are whole tiles and sizes that are not.
"""
from __future__ import annotations

import math

import torch

import nuvec_amd as nv
from nuvec_amd import layers

DTYPES = {"bfloat16": torch.bfloat16, "float16": torch.float16, "float32": torch.float32}
DTYPE_BYTES = {"bfloat16": 2, "float16": 2, "float32": 4}
BLOCK_FORMATS = {"mxfp4": (32, 4), "mxfp8": (32, 8), "nvfp4": (16, 4)}

# The largest work of a drawn case: that of the largest listed ones, a 2048-token prompt through a [14336, 4096] weight,
# 512 float32 rows through a [4096, 4096] one (the float32 matrix rate is a sixteenth of bfloat16's), 512 queries of 32 heads
# over 2048 positions, and the bytes of a prompt through 32 experts.
MOST_PRODUCT = 2048 * 14336 * 4096
MOST_PRODUCT_F32 = 512 * 4096 * 4096
MOST_WEIGHT = 151936 * 1024
MOST_SCORES = 32 * 512 * 2048
MOST_CACHE = 16 * 8192 * 8 * 128
MOST_BYTES = 420_000_000


def listed():
    return [
        # One token through a key projection of a model with grouped key heads: the smallest product of a decode step,
        # where the call itself is what counts.
        {"name": "linear_one_token", "kind": "linear", "mode": "affine", "group": 64, "bits": 4, "dtype": "bfloat16",
         "m": 1, "n": 1024, "k": 4096, "bias": True},
        # One token through the MLPs of four blocks, the bulk of a decode step: every weight comes from memory.
        {"name": "mlp_one_token", "kind": "mlp", "mode": "affine", "group": 64, "bits": 4, "dtype": "bfloat16",
         "m": 1, "dims": 4096, "hidden": 14336, "layers": 4},
        # Sixteen requests decoded together through 8-bit float16 weights.
        {"name": "mlp_batch_8bit", "kind": "mlp", "mode": "affine", "group": 32, "bits": 8, "dtype": "float16",
         "m": 16, "dims": 4096, "hidden": 11008, "layers": 2},
        # A 2048-token prompt through an up projection: the largest product.
        {"name": "linear_prompt", "kind": "linear", "mode": "affine", "group": 64, "bits": 4, "dtype": "bfloat16",
         "m": 2048, "n": 14336, "k": 4096, "bias": False},
        # The last, ragged chunk of a prompt through 3-bit codes, which cross word boundaries.
        {"name": "linear_ragged_3bit", "kind": "linear", "mode": "affine", "group": 64, "bits": 3, "dtype": "bfloat16",
         "m": 517, "n": 4096, "k": 4096, "bias": False},
        # A few rows in float32, as a check against a float32 model runs them.
        {"name": "linear_float32", "kind": "linear", "mode": "affine", "group": 64, "bits": 4, "dtype": "float32",
         "m": 33, "n": 4096, "k": 4096, "bias": False},
        # A step of four requests at both ends of a small model with tied embeddings: the lookup and the logits.
        {"name": "head_tied", "kind": "head", "mode": "affine", "group": 64, "bits": 4, "dtype": "bfloat16",
         "m": 4, "vocab": 151936, "dims": 1024},
        # One token through the experts of four blocks: 4 experts of 32, MXFP4, biases, the clamped gate.
        {"name": "moe_one_token", "kind": "moe", "mode": "mxfp4", "group": 32, "bits": 4, "dtype": "bfloat16",
         "m": 1, "dims": 2880, "hidden": 2880, "experts": 32, "top": 4, "bias": True, "activation": "swiglu_oai", "layers": 4},
        # 256 tokens of a prompt through the same experts.
        {"name": "moe_prompt", "kind": "moe", "mode": "mxfp4", "group": 32, "bits": 4, "dtype": "bfloat16",
         "m": 256, "dims": 2880, "hidden": 2880, "experts": 32, "top": 4, "bias": True, "activation": "swiglu_oai", "layers": 1},
        # A decode step of sixteen long requests over their 4-bit caches.
        {"name": "attention_decode", "kind": "attention", "group": 64, "bits": 4, "dtype": "bfloat16",
         "batch": 16, "heads": 32, "key_heads": 8, "queries": 1, "positions": 8192, "dim": 128},
        # A 512-token chunk of a prompt over an 8-bit cache of 2048 positions, causal.
        {"name": "attention_prompt", "kind": "attention", "group": 64, "bits": 8, "dtype": "bfloat16",
         "batch": 1, "heads": 32, "key_heads": 8, "queries": 512, "positions": 2048, "dim": 128},
        # A weight packed at load time, and another unpacked.
        {"name": "codec_weight", "kind": "codec", "mode": "affine", "group": 64, "bits": 4, "dtype": "bfloat16",
         "rows": 14336, "cols": 4096},
    ]


def _log(rng, low, high):
    return max(low, min(high, round(math.exp(rng.uniform(math.log(low), math.log(high))))))


def _format(rng):
    mode = rng.choice(["affine"] * 5 + list(BLOCK_FORMATS))
    if mode == "affine":
        return {"mode": mode, "group": rng.choice([32, 64, 64, 128]), "bits": rng.choice([2, 3, 4, 4, 4, 5, 6, 8, 8])}
    return {"mode": mode, "group": BLOCK_FORMATS[mode][0], "bits": BLOCK_FORMATS[mode][1]}


def _dtype(rng):
    return rng.choice(["bfloat16"] * 3 + ["float16", "float32"])


def draw(rng):
    """One more case: its kind, format and element type by how often they are met, its sizes over the whole range."""
    while True:
        case = _draw(rng)
        if work(case)["bytes"] <= MOST_BYTES:
            return case


def _draw(rng):
    kind = rng.choice(["linear", "linear", "linear", "mlp", "mlp", "head", "moe", "moe", "attention", "attention", "codec"])
    c = {"kind": kind, **_format(rng), "dtype": _dtype(rng)}
    group = max(c["group"], 32)
    most = MOST_PRODUCT_F32 if c["dtype"] == "float32" else MOST_PRODUCT
    if kind == "linear":
        n, k = _log(rng, 256, 16384), group * _log(rng, 512 // group, 14336 // group)
        c.update(m=_log(rng, 1, max(1, min(2048, most // (n * k)))), n=n, k=k, bias=rng.random() < 0.5)
    elif kind == "mlp":
        # (the hidden size is the down projection's row length, a whole number of groups)
        dims, hidden = group * _log(rng, 512 // group, 5120 // group), 64 * max(1, group // 64) * _log(rng, 16, 14336 // max(64, group))
        layers_ = rng.choice([1, 2, 4])
        c.update(m=_log(rng, 1, max(1, min(512, most // (3 * layers_ * dims * hidden)))), dims=dims, hidden=hidden, layers=layers_)
    elif kind == "head":
        dims = group * _log(rng, 512 // group, 4096 // group)
        c.update(m=_log(rng, 1, 64), vocab=_log(rng, 8192, MOST_WEIGHT // dims), dims=dims)
        if c["dtype"] == "float32":
            c["m"] = min(c["m"], max(1, MOST_PRODUCT_F32 // (c["vocab"] * dims)))
    elif kind == "moe":
        if c["dtype"] == "float32":  # (experts are run in half precision)
            c["dtype"] = "bfloat16"
        dims, hidden = group * _log(rng, 512 // group, 2880 // group), group * _log(rng, 512 // group, 2880 // group)
        top, layers_ = rng.choice([2, 4, 8]), rng.choice([1, 2])
        c.update(m=_log(rng, 1, max(1, min(512, most // (3 * layers_ * top * dims * hidden)))), dims=dims, hidden=hidden,
                 experts=rng.choice([8, 16, 32]), top=top, bias=rng.random() < 0.5,
                 activation=rng.choice(["swiglu", "swiglu_oai"]), layers=layers_)
    elif kind == "attention":
        del c["mode"]  # (caches are affine)
        dim, key_heads, per = rng.choice([64, 128]), rng.choice([2, 4, 8]), rng.choice([1, 2, 4, 8])
        c.update(group=rng.choice([32, 64]), bits=rng.choice([4, 4, 8, 8, 3]), heads=key_heads * per, key_heads=key_heads, dim=dim)
        if rng.random() < 0.5:
            batch = _log(rng, 1, 32)
            c.update(batch=batch, queries=1, positions=_log(rng, 128, min(32768, MOST_CACHE // (batch * key_heads * dim))))
        else:
            positions = _log(rng, 128, 8192)
            scores = MOST_SCORES // (16 if c["dtype"] == "float32" else 1)
            queries = _log(rng, 2, max(2, min(512, positions, scores // (positions * c["heads"]))))
            c.update(batch=rng.randint(1, max(1, min(4, scores // (queries * positions * c["heads"])))), queries=queries, positions=positions)
    else:
        cols = group * _log(rng, 128 // group, 8192 // group)
        size = 14336 * 4096 * 2 // DTYPE_BYTES[c["dtype"]]
        c.update(rows=_log(rng, 64, size // cols), cols=cols)
    return c


def _quant(case):
    if case.get("mode", "affine") == "affine":
        return nv.Quant.affine(case["group"], case["bits"])
    return nv.Quant.new(nv.QuantMode.parse(case["mode"]))


def _packed_bytes(case, rows, cols):
    """Bytes of a packed [rows, cols] weight: codes, scales and, for affine formats, biases."""
    scale = 2 * DTYPE_BYTES[case["dtype"]] if case.get("mode", "affine") == "affine" else 1
    return rows * cols * case["bits"] // 8 + rows * (cols // case["group"]) * scale


class _Inputs:
    """Tensors of one seed on the GPU: activations of unit variance, weights of a model's 0.02."""

    def __init__(self, case, seed):
        self.device, self.dtype, self.quant = torch.device("cuda"), DTYPES[case["dtype"]], _quant(case)
        self.gen = torch.Generator(device=self.device)
        self.gen.manual_seed(seed)

    def normal(self, *shape, std=1.0):
        return (torch.randn(shape, device=self.device, generator=self.gen) * std).to(self.dtype)

    def packed(self, *shape, std=0.02):
        return nv.quantize(self.normal(*shape, std=std), self.quant)

    def linear(self, n, k, bias=False):
        q = self.packed(n, k)
        return layers.QuantizedLinear(q.weight, q.scales, q.biases, self.normal(n, std=0.02) if bias else None, q.quant)

    def experts(self, e, n, k, bias):
        q = self.packed(e, n, k)
        return layers.SwitchProjection(q.weight, q.scales, q.biases, self.normal(e, n, std=0.02) if bias else None, q.quant)


def prepare(case, seed):
    """The weights, caches and activations of one pass."""
    put, kind = _Inputs(case, seed), case["kind"]
    if kind == "linear":
        return kind, put.linear(case["n"], case["k"], case["bias"]), put.normal(case["m"], case["k"])
    if kind == "mlp":
        blocks = []
        for _ in range(case["layers"]):
            mlp = layers.Mlp(put.linear(case["hidden"], case["dims"]), put.linear(case["hidden"], case["dims"]),
                             put.linear(case["dims"], case["hidden"]))
            blocks.append((mlp.fuse_gate_up(), put.normal(case["m"], case["dims"])))
        return kind, blocks
    if kind == "head":
        q = put.packed(case["vocab"], case["dims"])
        ids = torch.randint(case["vocab"], (case["m"],), device=put.device, generator=put.gen, dtype=torch.int32)
        return kind, layers.QuantizedEmbedding(q.weight, q.scales, q.biases, q.quant), ids, put.normal(case["m"], case["dims"])
    if kind == "moe":
        blocks = []
        for _ in range(case["layers"]):
            d, h, e = case["dims"], case["hidden"], case["experts"]
            experts = layers.SwitchGlu(put.experts(e, h, d, case["bias"]), put.experts(e, h, d, case["bias"]),
                                       put.experts(e, d, h, case["bias"]), activation=case["activation"]).fuse_gate_up()
            blocks.append((layers.MoeMlp(put.normal(e, d, std=0.02), experts, case["top"]), put.normal(1, case["m"], d)))
        return kind, blocks
    if kind == "attention":
        b, hq, hkv, l, s, d = (case[f] for f in ("batch", "heads", "key_heads", "queries", "positions", "dim"))
        return kind, put.normal(b, hq, l, d), put.packed(b, hkv, s, d, std=1.0), put.packed(b, hkv, s, d, std=1.0), d ** -0.5
    return kind, put.normal(case["rows"], case["cols"], std=0.02), put.quant, put.packed(case["rows"], case["cols"])


def run(state):
    """One pass; its results."""
    kind = state[0]
    if kind == "linear":
        _, layer, x = state
        return layer(x)
    if kind in ("mlp", "moe"):
        return [block(x) for block, x in state[1]]
    if kind == "head":
        _, table, ids, x = state
        return table(ids), table.as_linear(x)
    if kind == "attention":
        _, q, k, v, scale = state
        return layers.quantized_attention(q, k, v, scale, causal=True)
    _, dense, quant, packed = state
    q = nv.quantize(dense, quant)
    return q.weight.view(torch.int32), q.scales, q.biases, nv.dequantize(packed, dense.dtype)


def work(case):
    """Bytes and operations of one pass: each weight, input and result once, the products' multiplications and additions."""
    kind, e = case["kind"], DTYPE_BYTES[case["dtype"]]
    if kind == "linear":
        m, n, k = case["m"], case["n"], case["k"]
        return {"bytes": _packed_bytes(case, n, k) + e * (m * (n + k) + (n if case["bias"] else 0)), "flops": 2 * m * n * k}
    if kind == "mlp":
        m, d, h, blocks = case["m"], case["dims"], case["hidden"], case["layers"]
        return {"bytes": blocks * (2 * _packed_bytes(case, h, d) + _packed_bytes(case, d, h) + e * 2 * m * d),
                "flops": blocks * 6 * m * d * h}
    if kind == "head":
        m, n, k = case["m"], case["vocab"], case["dims"]
        rows_out = e if case["mode"] == "affine" else 2
        return {"bytes": _packed_bytes(case, n, k) + e * m * (n + k) + m * (4 + rows_out * k) + _packed_bytes(case, m, k), "flops": 2 * m * n * k}
    if kind == "moe":
        m, d, h, n, top = case["m"], case["dims"], case["hidden"], case["experts"], case["top"]
        met = n * (1 - (1 - top / n) ** m)  # experts that some token chose, were the choice even
        expert = 2 * _packed_bytes(case, h, d) + _packed_bytes(case, d, h) + (e * (2 * h + d) if case["bias"] else 0)
        return {"bytes": case["layers"] * (met * expert + e * (n * d + 2 * m * d)),
                "flops": case["layers"] * (6 * m * top * d * h + 2 * m * n * d)}
    if kind == "attention":
        b, hq, hkv, l, s, d = (case[f] for f in ("batch", "heads", "key_heads", "queries", "positions", "dim"))
        seen = l * (s - l) + l * (l + 1) // 2  # query i of l sees the first s - l + i + 1 positions
        return {"bytes": 2 * _packed_bytes(case, b * hkv * s, d) + 2 * e * b * hq * l * d, "flops": 4 * b * hq * seen * d}
    dense, packed = case["rows"] * case["cols"] * e, _packed_bytes(case, case["rows"], case["cols"])
    return {"bytes": 2 * (dense + packed), "flops": 2 * case["rows"] * case["cols"]}


def tolerance(case):
    """Codecs are bit-exact.  Products round their results (and, by kernel, the dequantized weights and what goes from one
    product to the next) to the element type and sum in float32."""
    if case["kind"] == "codec":
        return "exact"
    return {"bfloat16": {"rel": 1e-2}, "float16": {"rel": 2e-3}, "float32": {"rel": 1e-5}}[case["dtype"]]
