"""The decode attention kernel (csrc/qattn.hip) at the edges of its tiles and column layouts against float64 attention over
the dequantized cache.  Bound, of the largest value: the codes, the float32 queries' three bfloat16 terms and their products
are exact; the sums are float32 over operands of at most 143 x scale (the scores' of 8 bits 255, with a scale a sixteenth as large), 2^-24 of
that a rounding, with scale <= 2 max / 15, i.e. 1.1e-6 max, and their roundings are random: sixteen of them.  In the 16-bit types one rounding of the output beside it, and the
weights' 16 bits (2^-17)."""
import pytest
import torch

import nuvec_amd as nv
from nuvec_amd import ops

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("heads,key_heads,d,group", [(8, 1, 128, 32), (16, 2, 128, 64), (8, 1, 128, 128), (2, 2, 128, 32), (8, 2, 64, 32), (8, 1, 64, 64)])
@pytest.mark.parametrize("bits", [3, 4, 8])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
def test_edges(heads, key_heads, d, group, bits, dtype):
    quant = nv.Quant.affine(group, bits)
    for s in (1, 3, 16, 31, 32, 33, 129, 700):
        torch.manual_seed(s)
        put = lambda *shape: torch.randn(shape, device="cuda").to(dtype)
        k, v, q = nv.quantize(put(2, key_heads, s, d), quant), nv.quantize(put(2, key_heads, s, d), quant), put(2, heads, 1, d)
        sinks = put(heads) if s % 2 else None
        got = ops.quantized_attention(q, k, v, d ** -0.5, sinks)
        # scale * code + bias unrounded: the dequantized values in float64
        def dense(t):
            codes = nv.dequantize(nv.Quantized(t.weight, torch.ones_like(t.scales, dtype=torch.float32), torch.zeros_like(t.scales, dtype=torch.float32), quant))
            spread = lambda x: x.double().repeat_interleave(group, dim=-1)
            return (codes.double() * spread(t.scales) + spread(t.biases)).repeat_interleave(heads // key_heads, dim=1)
        kf, vf = dense(k), dense(v)
        scores = d ** -0.5 * (q.double() * kf).sum(-1)
        if sinks is not None:
            scores = torch.cat([scores, sinks.double().view(1, heads, 1).expand(2, heads, 1)], dim=-1)
        want = (torch.softmax(scores, -1)[..., :s, None] * vf).sum(-2, keepdim=True)
        u = {torch.float32: 0.0, torch.bfloat16: 2.0 ** -8, torch.float16: 2.0 ** -11}[dtype]
        bound = (16 * 1.1e-6 + (0 if dtype == torch.float32 else 2.0 ** -17)) * vf.abs().max() + u * want.abs()
        assert ((got.double() - want).abs() <= bound).all(), (s, (got.double() - want).abs().max().item())


@pytest.mark.parametrize("splits", [2, 3, 5, 31, 33, 64])
def test_merged_splits(splits):
    """One key head over 256 positions a split, up to the 64 splits that the kernel takes: lanes and groups of the merge that are
    full, partly used and idle.  The queries are zeros: the weights are equal and the output is the mean of the values."""
    s, d, quant = 256 * splits, 64, nv.Quant.affine(64, 4)
    v = nv.quantize(torch.randn(1, 1, s, d, device="cuda"), quant)
    k = nv.quantize(torch.randn(1, 1, s, d, device="cuda"), quant)
    got = ops.quantized_attention(torch.zeros(1, 2, 1, d, device="cuda"), k, v, 1.0)
    want = nv.dequantize(v).double().mean(-2, keepdim=True)
    # (as above: the float32 sums' random roundings)
    assert (got.double() - want).abs().max() <= 16 * 1.1e-6 * nv.dequantize(v).abs().max()
