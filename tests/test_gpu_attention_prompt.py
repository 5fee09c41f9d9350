"""Attention of several query rows on the matrix cores (csrc/qattn_prompt.hip) against float64 attention over the cache's values
s c + b, unrounded.  Bound, with u the element type's unit roundoff: the weights p of the softmax are rounded (relative error u) and
the values too, so a row's error is at most 2 u sum p |v| <= 2 u max |v|, and the output is rounded once more: u |out|.  A key's values
are rounded where the composition rounds them (keys_rounded below), which moves a score by at most u scale sum |q| |k| and a weight by
as much relatively: e = that bound's largest, e sum p |v| more; two terms elsewhere leave nothing.  A tenth more for the float32 sums
and exponentials."""
import numpy as np
import pytest
import torch

import nuvec_amd as nv
from nuvec_amd import layers, ops

pytestmark = pytest.mark.gpu

# batch, query heads, key heads, queries, positions, head size, bits, group, causal, sinks
CASES = [
    (1, 2, 2, 2, 2, 64, 4, 32, True, False),         # fewer rows and keys than a tile
    (1, 4, 2, 31, 31, 128, 8, 64, True, True),       # 62 rows: a tile and a ragged one
    (2, 6, 2, 33, 95, 64, 3, 64, True, False),       # three heads per key head
    (1, 1, 1, 32, 32, 128, 4, 128, False, False),    # exactly one tile
    (1, 2, 1, 5, 4100, 128, 8, 32, True, True),      # few rows of a long cache: splits over the grid
    (3, 8, 8, 3, 1023, 64, 6, 32, False, True),
    (1, 32, 8, 257, 600, 128, 4, 64, True, False),
    (4, 32, 4, 320, 320, 64, 8, 64, True, True),     # two and four row groups a block
    (2, 32, 8, 512, 700, 128, 5, 64, True, False),
    (1, 8, 2, 40, 64, 64, 1, 32, False, False),
    (1, 8, 2, 9, 33, 128, 2, 32, True, False),
    (1, 4, 1, 17, 1024, 64, 4, 64, True, False),     # (float16: keys of two terms)
    (2, 8, 2, 16, 1500, 128, 8, 64, False, True),    # (both types)
    (1, 8, 2, 24, 8192, 128, 3, 32, True, False),    # (both types, many positions)
    (4, 64, 4, 130, 1056, 128, 6, 128, False, False),  # two and four row groups a block
    (8, 64, 8, 200, 1100, 64, 4, 64, True, False),
    (11, 8, 8, 3, 16500, 128, 4, 64, True, False),   # more heads than one workspace holds: slices, the last one smaller
]


def keys_rounded(dtype, l, s):
    return s < 1024 or (dtype == torch.bfloat16 and l > 16 and s < 8192)


def unrounded(t):
    """s c + b in float64."""
    codes = nv.dequantize(nv.Quantized(t.weight, torch.ones_like(t.scales, dtype=torch.float32), torch.zeros_like(t.scales, dtype=torch.float32), t.quant))
    spread = lambda x: x.double().repeat_interleave(t.quant.group_size, dim=-1)
    return codes.double() * spread(t.scales) + spread(t.biases)


@pytest.mark.parametrize("case", CASES, ids=str)
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_prompt_attention(case, dtype):
    b, hq, hkv, l, s, d, bits, group, causal, with_sinks = case
    torch.manual_seed(l * s)
    put = lambda *shape: torch.randn(shape, device="cuda").to(dtype)
    quant = nv.Quant.affine(group, bits)
    k, v, q = nv.quantize(put(b, hkv, s, d), quant), nv.quantize(put(b, hkv, s, d), quant), put(b, hq, l, d)
    sinks = put(hq) if with_sinks else None
    got = layers.quantized_attention(q, k, v, d ** -0.5, sinks, causal=causal)
    assert got.dtype == dtype and got.shape == q.shape
    assert torch.equal(got, ops.quantized_attention_prompt(q, k, v, d ** -0.5, sinks, causal))
    rep, u = hq // hkv, 2.0 ** (-8 if dtype == torch.bfloat16 else -11)
    kf, vf = (unrounded(t) for t in (k, v))
    for i in range(b):  # (a batch at a time: float64 scores)
        kd, vd = (t[i].repeat_interleave(rep, dim=0).contiguous() for t in (kf, vf))
        qd = q[i].double()
        scores = d ** -0.5 * (qd @ kd.transpose(-1, -2).contiguous())
        if causal:
            hidden = torch.arange(s, device="cuda")[None, :] > (s - l + torch.arange(l, device="cuda"))[:, None]
            scores = scores.masked_fill(hidden, float("-inf"))
        if with_sinks:
            scores = torch.cat([scores, sinks.double().view(hq, 1, 1).expand(hq, l, 1)], dim=-1)
        p = torch.softmax(scores, dim=-1)[..., :s].contiguous()
        want = p @ vd
        bound = u * (2 * vf[i].abs().max() + want.abs())
        if keys_rounded(dtype, l, s):
            e = u * d ** -0.5 * (qd.abs() @ kd.abs().transpose(-1, -2).contiguous()).amax(-1, keepdim=True)
            bound = bound + e * (p @ vd.abs() + want.abs())  # (a weight and the denominator)
        off = (got[i].double() - want).abs()
        assert (off <= 1.1 * bound).all(), off.max().item()


@pytest.mark.parametrize("case", [(1, 6, 2, 61, 600, 128, 4, 64, True, True), (1, 3, 1, 43, 2048, 64, 8, 32, True, True),
                                  (1, 2, 1, 67, 2304, 128, 4, 64, False, False), (2, 2, 1, 33, 1300, 64, 3, 64, True, False)], ids=str)
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_merged_splits(case, dtype):
    """Two, eight, nine and five splits of rows that are no whole blocks of the merge."""
    test_prompt_attention(case, dtype)


@pytest.mark.parametrize("dtype,l,s", [(torch.float16, 2, 1024), (torch.float16, 200, 1100), (torch.bfloat16, 16, 1100), (torch.bfloat16, 40, 8200)])
@pytest.mark.parametrize("d", [64, 128])
def test_keys_of_two_terms(dtype, l, s, d):
    """Keys that need 16 bits, whose scores differ by what one rounding of them loses: half the keys score d more than the others,
    their values are 1 and -1, the output is tanh(d / 2) to the rounding of the weights."""
    quant, ulp = nv.Quant.affine(32, 8), 2.0 ** (-7 if dtype == torch.bfloat16 else -10)
    delta = 0.5 if dtype == torch.bfloat16 else 13 / 256
    words = torch.full((1, 1, s, d // 4), -1, dtype=torch.int32, device="cuda").view(torch.uint32)
    put = lambda value: torch.full((1, 1, s, d // 32), float(value), device="cuda", dtype=dtype)
    biases, signs = put(0), put(1)
    biases[:, :, ::2, 0] = delta
    signs[:, :, 1::2] = -1
    k = nv.Quantized(words, put(1 + ulp), biases, quant)
    v = nv.Quantized(torch.full_like(words.view(torch.int32), 0x01010101).view(torch.uint32), signs, put(0), quant)
    q = torch.zeros(1, 4, l, d, device="cuda", dtype=dtype)
    q[..., 0], q[..., 32] = 1, -1  # (of the first and the second group: the codes' part cancels)
    got = layers.quantized_attention(q, k, v, 1.0)
    want = float(np.tanh(delta / 2))
    assert ((got.double() - want).abs() <= 1.1 * 2.0 ** (-8 if dtype == torch.bfloat16 else -11) * (1 + want)).all(), (got[0, 0, 0, 0].item(), want)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_workspace_is_bounded(dtype):
    """32 batches of 8 key heads over 32768 positions: 4.3 GB of operands, which pass through one workspace slice by slice."""
    import ctypes as C

    from nuvec_amd import _lib
    ops._init(torch.empty(1, device="cuda"))
    for batch, queries in ((1, 2), (32, 2), (32, 512)):
        d = _lib.AttentionPromptDescC(_lib.AttentionDescC(ops._CODE[dtype], 4, 64, 128, batch, 32, 8, 32768, 0.1), queries, 1)
        need = _lib.load().nvq_quantized_attention_prompt_workspace_bytes(C.byref(d))
        assert 0 < need <= 320 << 20, need  # (256 MB of operands; the splits' states beside them)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("sinks", [False, True])
def test_more_queries_than_positions(dtype, sinks):
    """Causal rows that see no key: NaN, as their softmax is; with a sink, which takes all the weight, zero."""
    l, s, d = 70, 33, 64
    k, v = (nv.quantize(torch.randn(2, 2, s, d, device="cuda").to(dtype), nv.Quant.affine(32, 4)) for _ in range(2))
    q, sink = torch.randn(2, 8, l, d, device="cuda").to(dtype), torch.randn(8, device="cuda").to(dtype) if sinks else None
    got = layers.quantized_attention(q, k, v, 0.125, sink, causal=True)
    composed = layers.quantized_attention(q, k, v, 0.125, sink, causal=True, fused=False)
    blind = got[:, :, : l - s]
    assert (blind == 0).all() if sinks else torch.isnan(blind).all()
    assert torch.equal(torch.isnan(got), torch.isnan(composed)) and torch.isfinite(got[:, :, l - s:]).all()
    rest = layers.quantized_attention(q[:, :, l - s:].contiguous(), k, v, 0.125, sink, causal=True)  # (in other tiles: a rounding either way)
    u = 2.0 ** (-7 if dtype == torch.bfloat16 else -10)
    assert ((got[:, :, l - s:] - rest).float().abs() <= 2 * u * (rest.float().abs() + 1)).all()


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("s", [300, 2000])
def test_infinities_and_nans_stay_where_they_are(dtype, s):
    """A NaN or an infinity in a query is its row's; keys whose scores are -inf weigh nothing."""
    torch.manual_seed(s)
    l, d, quant = 9, 128, nv.Quant.affine(64, 8)
    k, v = (nv.quantize(torch.randn(2, 2, s, d, device="cuda").to(dtype), quant) for _ in range(2))
    q = torch.randn(2, 8, l, d, device="cuda").to(dtype).abs_()
    run = lambda k=k, v=v: layers.quantized_attention(q, k, v, d ** -0.5)
    plain, u = run(), 2.0 ** (-7 if dtype == torch.bfloat16 else -10)  # (rows of a tile rescale together: one rounding either way)
    for bad in (float("nan"), float("inf")):
        keep = q[0, 1, 4, 5].clone()
        q[0, 1, 4, 5] = bad
        got = run()
        q[0, 1, 4, 5] = keep
        assert torch.isnan(got[0, 1, 4]).all()
        got[0, 1, 4] = plain[0, 1, 4]
        assert ((got - plain).float().abs() <= 2 * u * (plain.float().abs() + 1)).all() and torch.equal(got[1], plain[1])
    k.biases[:, :, :100] = float("-inf")
    rest = [nv.Quantized(t.weight[:, :, 100:].contiguous(), t.scales[:, :, 100:].contiguous(), t.biases[:, :, 100:].contiguous(), quant) for t in (k, v)]
    got, want = run(), run(*rest)
    assert ((got - want).float().abs() <= 2 * u * (want.float().abs() + 1)).all()


def test_strided_queries_and_what_the_kernels_do_not_take():
    k, v = (nv.quantize(torch.randn(1, 2, 50, 64, device="cuda").bfloat16(), nv.Quant.affine(32, 4)) for _ in range(2))
    q = torch.randn(1, 10, 4, 64, device="cuda").bfloat16().transpose(1, 2)  # [1, 4, 10, 64], not dense
    got = layers.quantized_attention(q, k, v, 0.125, causal=True)
    assert torch.equal(got, layers.quantized_attention(q.contiguous(), k, v, 0.125, causal=True))
    for dtype, d in ((torch.float32, 64), (torch.bfloat16, 96)):  # the composition
        kk, vv = (nv.quantize(torch.randn(1, 2, 50, d, device="cuda").to(dtype), nv.Quant.affine(32, 4)) for _ in range(2))
        qq = torch.randn(1, 4, 10, d, device="cuda").to(dtype)
        with pytest.raises(nv.Unsupported):
            ops.quantized_attention_prompt(qq, kk, vv, 0.125)
        assert layers.quantized_attention(qq, kk, vv, 0.125).shape == qq.shape
