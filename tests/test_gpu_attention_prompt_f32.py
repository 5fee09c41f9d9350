"""Attention of several float32 query rows over a quantized cache (`prompt_attention_f32_kernel`; crates/nuvec-core/src/fast/imp.rs:3996-4035)
against float64 attention over the cache as the CPU's product dequantizes it, and against the composition of the library's products."""
import pytest
import torch

import nuvec_amd as nv
from nuvec_amd import layers

pytestmark = pytest.mark.gpu


def cache(b, hkv, s, d, group, bits, gen):
    return nv.quantize(torch.randn(b, hkv, s, d, device="cuda", generator=gen), nv.Quant.affine(group, bits))


def exact(q, k, v, scale, sinks, causal):
    b, hq, l, d = q.shape
    rep = hq // k.weight.shape[1]
    kd, vd = (nv.dequantize(t, torch.float32).double().repeat_interleave(rep, 1) for t in (k, v))
    scores = (q.double() * scale) @ kd.transpose(-1, -2)
    s = scores.shape[-1]
    if causal:
        scores = scores.masked_fill(torch.arange(s, device="cuda")[None, :] > (s - l + torch.arange(l, device="cuda"))[:, None], float("-inf"))
    if sinks is not None:
        scores = torch.cat([scores, sinks.double().reshape(1, hq, 1, 1).expand(b, hq, l, 1)], -1)
    return torch.softmax(scores, -1)[..., :s] @ vd


@pytest.mark.parametrize("dim", [64, 128])
@pytest.mark.parametrize("group,bits", [(32, 4), (64, 8), (64, 3), (32, 6), (64, 5), (32, 2), (64, 1)])
def test_against_float64(group, bits, dim):
    """Rows and keys at the ends of their tiles, four row groups a block and four wavefronts a row group, the keys split over the grid or
    not.  A score takes about 2 sqrt(D) roundings of 2^-25 of its partial sums and two of its own size (under 8 bits of 2^-24 here), a
    weight the same absolutely, an output as many again of its sum over the keys: 16 units of 2^-24 (0.9e-7 to 3e-7 measured)."""
    gen = torch.Generator(device="cuda")
    gen.manual_seed(100 * bits + dim)
    shapes = [(1, 8, 2, 34, 1218), (2, 4, 4, 2, 33), (4, 4, 1, 17, 64), (1, 2, 2, 281, 284), (3, 2, 2, 5, 2), (8, 64, 8, 70, 65), (1, 1, 1, 16, 4096)]
    for b, hq, hkv, l, s in shapes:
        q = torch.randn(b, hq, l, dim, device="cuda", generator=gen)
        k, v = (cache(b, hkv, s, dim, group, bits, gen) for _ in range(2))
        sinks = torch.randn(hq, device="cuda", generator=gen)
        for causal, sink in ((True, None), (False, sinks), (True, sinks)):
            if causal and l > s:
                continue  # (rows that see no key: below)
            got = layers.quantized_attention(q, k, v, dim ** -0.5, sink, causal=causal)
            want = exact(q, k, v, dim ** -0.5, sink, causal)
            assert (got.double() - want).norm() <= 16 * 2.0 ** -24 * want.norm(), (b, hq, hkv, l, s, causal)
            assert torch.equal(got, layers.quantized_attention(q.transpose(1, 2).contiguous().transpose(1, 2), k, v, dim ** -0.5, sink, causal=causal))


@pytest.mark.parametrize("scale", [0.125, -0.125, 0.0, 3.0])
def test_like_the_composition(scale):
    """Scales of either sign, none, and ones that make the weights one key's; rows that see no key; infinities and NaN in a row."""
    gen = torch.Generator(device="cuda")
    gen.manual_seed(9)
    q = torch.randn(2, 8, 40, 64, device="cuda", generator=gen)
    k, v = (cache(2, 4, 100, 64, 64, 4, gen) for _ in range(2))
    got, want = (layers.quantized_attention(q, k, v, scale, causal=True, fused=f) for f in (True, False))
    # (3.0: a score of 24 x 8 takes an error of 2^-17 into its weight, of either side)
    assert (got - want).norm() <= (1e-4 if scale == 3.0 else 2e-6) * want.norm()
    short = nv.Quantized(k.weight[:, :, :30].contiguous(), k.scales[:, :, :30].contiguous(), k.biases[:, :, :30].contiguous(), k.quant)
    vshort = nv.Quantized(v.weight[:, :, :30].contiguous(), v.scales[:, :, :30].contiguous(), v.biases[:, :, :30].contiguous(), v.quant)
    got, want = (layers.quantized_attention(q, short, vshort, scale, causal=True, fused=f) for f in (True, False))
    assert torch.equal(got.isnan(), want.isnan()) and got.isnan()[:, :, :10].all() and not got.isnan()[:, :, 10:].any()
    odd = q.clone()
    odd[0, 3, 7, 5] = float("nan")
    odd[1, 2, 9, 1] = float("inf")
    plain, got = layers.quantized_attention(q, k, v, scale, causal=True), layers.quantized_attention(odd, k, v, scale, causal=True)
    assert got[0, 3, 7].isnan().all() and got[1, 2, 9].isnan().all()
    got[0, 3, 7], got[1, 2, 9] = plain[0, 3, 7], plain[1, 2, 9]
    assert torch.equal(got, plain)


@pytest.mark.parametrize("dim", [64, 128])
@pytest.mark.parametrize("s", [300, 2000])
@pytest.mark.parametrize("sign", [1.0, -1.0])
def test_keys_whose_scores_are_minus_infinity_weigh_nothing(dim, s, sign):
    """Whatever the scale's sign and the sign of what its rounding leaves (positive at head size 64, negative at 128), in whole tiles and
    between other keys; a row of such keys alone is NaN, as the composition has it, or its sink's.  The bound is that of test_against_float64
    for two sums, the other keys lying in other tiles."""
    gen = torch.Generator(device="cuda")
    gen.manual_seed(s + dim)
    quant = nv.Quant.affine(64, 8)
    k, v = (cache(2, 2, s, dim, 64, 8, gen) for _ in range(2))
    q = torch.randn(2, 8, 9, dim, device="cuda", generator=gen).abs_()
    seen = torch.ones(s, dtype=torch.bool, device="cuda")
    seen[:100], seen[170], seen[s - 1] = False, False, False
    k.biases[:, :, ~seen] = sign * float("-inf")
    take = lambda t: nv.Quantized(t.weight.view(torch.int32)[:, :, seen].contiguous().view(torch.uint32), t.scales[:, :, seen].contiguous(),
                                  t.biases[:, :, seen].contiguous(), quant)
    got, want = layers.quantized_attention(q, k, v, sign * dim ** -0.5), exact(q, take(k), take(v), sign * dim ** -0.5, None, False)
    assert (got.double() - want).norm() <= 32 * 2.0 ** -24 * want.norm()
    k.biases[:] = sign * float("-inf")
    assert layers.quantized_attention(q, k, v, sign * dim ** -0.5).isnan().all()
    sinks = torch.randn(8, device="cuda", generator=gen)
    assert (layers.quantized_attention(q, k, v, sign * dim ** -0.5, sinks) == 0).all()


@pytest.mark.parametrize("dim", [64, 128])
@pytest.mark.parametrize("s", [45, 2000])
@pytest.mark.parametrize("size", [1e4, 1e7, -1e7, 1e10, -1e10, 1e20, 1e33, -1e33, -1e36])
def test_scores_of_any_size(dim, s, size):
    """The largest scores weigh alike however large they are: beyond 2^31 a score's own rounding is more than exp2 holds, and all of
    a row may lie below any finite value that a maximum could start from.  Keys of ones and of twos: the mean of half of the values."""
    gen = torch.Generator(device="cuda")
    gen.manual_seed(s + dim)
    k, v = (cache(1, 2, s, dim, 64, 8, gen) for _ in range(2))
    k.scales.zero_()
    k.biases.copy_(torch.randint(1, 3, (1, 2, s, 1), device="cuda", generator=gen).float().expand(k.biases.shape))
    q = torch.full((1, 8, 7, dim), size, device="cuda")
    sinks = torch.randn(8, device="cuda", generator=gen)
    for causal, sink in ((False, None), (True, None), (False, sinks)):
        got, want = layers.quantized_attention(q, k, v, dim ** -0.5, sink, causal=causal), exact(q, k, v, dim ** -0.5, sink, causal)
        assert (got.double() - want).norm() <= 16 * 2.0 ** -24 * want.norm() + 1e-30, (causal, sink is None)
