"""The decode attention kernels (csrc/qattn.hip) at the edges of their tiles and column layouts against float64 attention over
the dequantized cache.  Bound, of the largest value: the codes, the queries' and the weights' bfloat16 terms and their products
are exact; the sums are float32 over operands of at most 143 x scale (the scores' of 8 bits 255, with a scale a sixteenth as large), 2^-24 of
that a rounding, with scale <= 2 max / 15, i.e. 1.1e-6 max, and their roundings are random: sixteen of them.  In the 16-bit types one rounding
of the output beside it."""
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
        check(heads, key_heads, d, quant, dtype, 2, s)


@pytest.mark.parametrize("heads,key_heads,d,group", [(8, 1, 128, 32), (16, 2, 128, 64), (8, 1, 128, 128), (4, 1, 128, 32), (8, 2, 64, 32), (8, 1, 64, 64)])
@pytest.mark.parametrize("bits", [3, 4, 8])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
def test_edges_of_many(heads, key_heads, d, group, bits, dtype):
    """Four and eight query heads per key head over 60000 positions in all (the matrix cores), few of them a batch."""
    for s in (1, 3, 31, 33, 129, 700):
        check(heads, key_heads, d, nv.Quant.affine(group, bits), dtype, -(-60000 * 128 // (s * key_heads * d)) if s > 3 else 60000, s)


def check(heads, key_heads, d, quant, dtype, batch, s):
    torch.manual_seed(s)
    group = quant.group_size
    put = lambda *shape: torch.randn(shape, device="cuda").to(dtype)
    k, v, q = nv.quantize(put(batch, key_heads, s, d), quant), nv.quantize(put(batch, key_heads, s, d), quant), put(batch, heads, 1, d)
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
        scores = torch.cat([scores, sinks.double().view(1, heads, 1).expand(batch, heads, 1)], dim=-1)
    want = (torch.softmax(scores, -1)[..., :s, None] * vf).sum(-2, keepdim=True)
    u = {torch.float32: 0.0, torch.bfloat16: 2.0 ** -8, torch.float16: 2.0 ** -11}[dtype]
    bound = 16 * 1.1e-6 * vf.abs().max() + u * want.abs()
    assert ((got.double() - want).abs() <= bound).all(), (s, (got.double() - want).abs().max().item())


@pytest.mark.parametrize("batch", [16, 32768])  # (fewer and more positions)
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
def test_weights_of_24_bits(dtype, batch):
    """Two keys whose scores differ by a little, and values of 1 and -1: the output is tanh of half the difference, what is left of
    weights that nearly cancel.  They come as codes of 1 that are counted from 128 (the kernels' middle of eight bits), so an error of a weight
    is seen 127-fold: 16 bits of it would show 127 x 2^-18 on average, float32 shows the exponential's and the sums' 2^-24, sixteen of them here."""
    torch.manual_seed(11)
    quant, heads, d = nv.Quant.affine(64, 8), 8, 128
    q = torch.zeros(batch, heads, 1, d, device="cuda")
    q[..., 0] = torch.rand(batch, heads, 1, device="cuda") * 2.0 ** -6
    q = q.to(dtype)
    put = lambda value: torch.full((batch, 1, 2, 2), float(value), device="cuda", dtype=dtype)
    codes = torch.zeros(batch, 1, 2, d // 4, dtype=torch.int32, device="cuda")
    codes[:, :, 0, 0] = 1
    k = nv.Quantized(codes.view(torch.uint32), put(1), put(0), quant)
    signs = put(1)
    signs[:, :, 1] = -1
    v = nv.Quantized(torch.full_like(codes, 0x01010101).view(torch.uint32), signs, put(0), quant)
    got = ops.quantized_attention(q, k, v, 1.0).double()
    want = torch.tanh(q[..., :1].double() / 2).expand_as(got)
    u = {torch.float32: 0.0, torch.bfloat16: 2.0 ** -8, torch.float16: 2.0 ** -11}[dtype]
    assert ((got - want).abs() <= u * want.abs() + 16 * 128 * 2.0 ** -24).all(), (got - want).abs().max().item()


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


@pytest.mark.parametrize("splits", [2, 7, 8, 9])
@pytest.mark.parametrize("heads,dim", [(1, 64), (5, 64), (3, 128)])
def test_merged_splits_up_to_eight(splits, heads, dim):
    """Both sides of the splits that a row's own threads merge, heads that are no whole blocks of them, weights that differ by split:
    the second half of the keys has scores 3 above the first."""
    s, quant = 256 * splits, nv.Quant.affine(64, 4)
    keys = torch.zeros(1, heads, s, dim, device="cuda")
    keys[:, :, s // 2:, 0] = 3.0
    v = nv.quantize(torch.randn(1, heads, s, dim, device="cuda"), quant)
    q = torch.zeros(1, heads, 1, dim, device="cuda")
    q[..., 0] = 1.0
    k, sinks = nv.quantize(keys, quant), torch.full((heads,), 7.0, device="cuda")
    scores = nv.dequantize(k).double()[..., 0]
    weights = torch.softmax(torch.cat([scores, sinks.double().view(1, heads, 1)], dim=-1), dim=-1)[..., :s]
    want = (weights.unsqueeze(-1) * nv.dequantize(v).double()).sum(-2, keepdim=True)
    got = ops.quantized_attention(q, k, v, 1.0, sinks)
    # (the float32 sums' random roundings, as above)
    assert (got.double() - want).abs().max() <= 16 * 1.1e-6 * nv.dequantize(v).abs().max()


@pytest.mark.parametrize("heads,batch", [(2, 1), (8, 300)])  # the vector kernel, the matrix cores
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
def test_infinities_and_nans_stay_where_they_are(dtype, heads, batch):
    """A NaN or an infinity in one head's query or one group of a value reaches what attention over it reaches and nothing else: other
    batches and groups keep the bits that they have without it, other heads of a block (whose sums may be rescaled at another key) their
    values to a rounding.  Keys whose scores are -inf weigh nothing; a row of them alone is NaN, as its softmax is."""
    torch.manual_seed(9)
    s, d, group = 300, 128, 64
    quant = nv.Quant.affine(group, 4)
    put = lambda *shape: torch.randn(shape, device="cuda").to(dtype)
    k, v, q = nv.quantize(put(batch, 2, s, d), quant), nv.quantize(put(batch, 2, s, d), quant), put(batch, 2 * heads, 1, d)
    run = lambda: ops.quantized_attention(q, k, v, d ** -0.5)
    plain = run()
    u = {torch.float32: 2.0 ** -20, torch.bfloat16: 2.0 ** -7, torch.float16: 2.0 ** -10}[dtype]  # (sums in another order; one rounding either way)
    near = lambda a, b: ((a - b).float().abs() <= u * (b.float().abs() + 1)).all()
    for bad in (float("nan"), float("inf")):
        keep = q[0, 1, 0, 5].clone()
        q[0, 1, 0, 5] = bad
        got = run()
        q[0, 1, 0, 5] = keep
        assert torch.isnan(got[0, 1]).all() and near(got[0, 0], plain[0, 0]) and near(got[0, 2:], plain[0, 2:])
        assert torch.equal(got[0, heads:], plain[0, heads:]) and torch.equal(got[1:], plain[1:])
    # a value's second group: its 64 outputs of every head over it
    keep = v.biases[0, 0, 7, 1].clone()
    v.biases[0, 0, 7, 1] = float("nan")
    got = run()
    v.biases[0, 0, 7, 1] = keep
    assert torch.isnan(got[0, :heads, 0, group:]).all() and torch.equal(got[0, :heads, 0, :group], plain[0, :heads, 0, :group])
    assert torch.equal(got[0, heads:], plain[0, heads:]) and torch.equal(got[1:], plain[1:])
    # keys at -inf: every query positive in one place, the first 200 keys' biases there -inf
    q.abs_()
    biases = k.biases.clone()
    k.biases[0, 0, :200] = float("-inf")
    got = run()
    rest = [nv.Quantized(t.weight[:1, :1, 200:].contiguous(), t.scales[:1, :1, 200:].contiguous(), t.biases[:1, :1, 200:].contiguous(), quant) for t in (k, v)]
    want = ops.quantized_attention(q[:1, :heads].contiguous(), *rest, d ** -0.5)
    assert near(got[:1, :heads], want)
    k.biases[0, 0] = float("-inf")
    assert torch.isnan(run()[0, :heads]).all()
    k.biases.copy_(biases)
