"""Attention of several query rows on the matrix cores (csrc/qattn_prompt.hip) against float32 attention over the
dequantized cache.  Bound: keys and values are `dequantize`'s bits, the weights p of the softmax are rounded to the element
type (relative error u, its unit roundoff) before the product with the values, so a row's error is at most u sum p |v| <=
u max |v|, and the output is rounded once more: u |out|; a tenth more for the float32 sums and exponentials."""
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
]


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
    rep = hq // hkv
    kf, vf = (nv.dequantize(t).float().repeat_interleave(rep, dim=1).contiguous() for t in (k, v))
    scores = d ** -0.5 * (q.float() @ kf.transpose(-1, -2).contiguous())
    if causal:
        hidden = torch.arange(s, device="cuda")[None, :] > (s - l + torch.arange(l, device="cuda"))[:, None]
        scores = scores.masked_fill(hidden, float("-inf"))
    if with_sinks:
        scores = torch.cat([scores, sinks.float().view(1, hq, 1, 1).expand(b, hq, l, 1)], dim=-1)
    want = torch.softmax(scores, dim=-1)[..., :s].contiguous() @ vf
    u = 2.0 ** (-8 if dtype == torch.bfloat16 else -11)
    assert ((got.float() - want).abs() <= 1.1 * u * (vf.abs().max() + want.abs())).all(), (got.float() - want).abs().max().item()


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
