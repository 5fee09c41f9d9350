"""Sorted pairs on the grouped kernel where its tiles, windows, tables and groups end: passes of 1 to 4 tiles of rows, experts with no
row and with more than a pass, K of part of a window, of windows that the groups of a block share unevenly and of tables that begin off
16 bytes, N off whole stores of four, and K split over one, two and four groups.  Held to the CPU product
(crates/nuvec-core/src/kernels.rs:1091-1142) at the bar of the element type."""
import numpy as np
import pytest
import torch

import nuvec_amd as nv
from nuvec_amd import layers
from oracle import ref
from tests.hip_backend import to_dev, to_host
from tests.test_gpu_half_steps import MODES, unrounded
from tests.test_gpu_parity import make_w, make_x

pytestmark = pytest.mark.gpu

ROWS = [0, 1, 16, 17, 33, 48, 0, 49, 64, 65]


def packed(rng, n, k, dtype, fmt):
    """A weight and the oracle's product of rows with it."""
    w = make_w(rng, n, k, dtype)
    if isinstance(fmt, str):
        codes, scales = ref.fp_quantize(w, dtype, MODES[fmt])
        group, bits = ref.FP_PARAMS[MODES[fmt]]
        want = lambda x: ref.quantized_matmul(x, codes, scales, None, mode=MODES[fmt], group=group, bits=bits, dtype=dtype, threads=8)
        return nv.Quantized(to_dev(codes), to_dev(scales), None, nv.Quant.new(getattr(nv.QuantMode, fmt))), want
    group, bits = fmt
    codes, scales, biases = ref.affine_quantize(w, dtype, group, bits)
    if n < 1024:
        want = lambda x: ref.quantized_matmul(x, codes, scales, biases, group=group, bits=bits, dtype=dtype, threads=8)
    else:
        want = lambda x: ref.quantized_matmul_device(x, codes, scales, biases, group=group, bits=bits, dtype=dtype, rounded_weights=True)
    return nv.Quantized(to_dev(codes), to_dev(scales), to_dev(biases), nv.Quant.affine(group, bits)), want


def stacked(experts):
    stack = lambda f: None if f(experts[0][0]) is None else torch.stack([f(q) for q, _ in experts])
    return nv.Quantized(stack(lambda q: q.weight), stack(lambda q: q.scales), stack(lambda q: q.biases), experts[0][0].quant)


# (groups of a block: 1 off whole blocks of 128 columns, else 2 from four windows and 4 from twelve)
@pytest.mark.parametrize("fmt", [(64, 1), (64, 2), (128, 3), (64, 4), (128, 5), (32, 6), (32, 8), "MXFP4", "MXFP8", "NVFP4"], ids=str)
@pytest.mark.parametrize("dtype,n,k", [(ref.BF16, 1030, 384), (ref.F16, 1024, 640), (ref.BF16, 1026, 1664), (ref.BF16, 1152, 2432), (ref.F16, 200, 640), (ref.BF16, 128, 1664), (ref.BF16, 1024, 128)])
def test_passes_and_windows(fmt, dtype, n, k):
    rng = np.random.default_rng(9100 + n + k)
    experts = [packed(rng, n, k, dtype, fmt) for _ in ROWS]
    q = stacked(experts)
    ids = np.repeat(np.arange(len(ROWS)), ROWS).astype(np.int32)
    tokens = rng.integers(0, 40, size=ids.size).astype(np.int32)  # (rows of x that several pairs take)
    x = make_x(rng, 40, k, dtype)
    place = rng.permutation(ids.size).astype(np.int32)
    dev = lambda a: torch.from_numpy(a).cuda()
    got = to_host(nv.gather_qmm_grouped(to_dev(x), q, dev(tokens), dev(ids), nv.sorted_offsets(dev(ids), len(ROWS)), out_rows=dev(place)))[place]
    for e, rows in enumerate(ROWS):
        if rows > 0:
            want = ref.to_f32(experts[e][1](x[tokens[ids == e]]), dtype)
            bound = (2.0 ** -7 if dtype == ref.BF16 else 2.0 ** -10) * np.max(np.abs(want), axis=1, keepdims=True)
            assert np.all(np.abs(ref.to_f32(got[ids == e], dtype) - want) <= bound), (e, rows)


# What a block's tail rows, pieces of codes and tables read lies inside their tensors' own lines: the last expert's last rows are right
# whatever lies after them, and every pair's sums are its own, whatever the pairs beside it.
@pytest.mark.parametrize("fmt", [(32, 4), (32, 8), "MXFP4"], ids=str)
@pytest.mark.parametrize("n,k", [(1024, 1536), (1152, 2432), (1030, 640)])
def test_a_pair_alone_has_the_bits_it_has_among_others(fmt, n, k):
    rng = np.random.default_rng(9200 + n + k)
    experts = [packed(rng, n, k, ref.BF16, fmt) for _ in range(3)]
    q = stacked(experts)
    ids = np.repeat(np.arange(3), [40, 3, 20]).astype(np.int32)  # (all fewer than 64, whose affine weights are float32)
    x = to_dev(make_x(rng, ids.size, k, ref.BF16))
    dev = lambda a: torch.from_numpy(a).cuda()
    rows = torch.arange(ids.size, dtype=torch.int32, device="cuda")
    whole = nv.gather_qmm_grouped(x, q, rows, dev(ids), nv.sorted_offsets(dev(ids), 3))
    for first, last in [(0, 17), (38, 45), (43, 63)]:
        some = dev(ids[first:last])
        part = nv.gather_qmm_grouped(x, q, rows[first:last].contiguous(), some, nv.sorted_offsets(some, 3))
        assert torch.equal(part, whole[first:last])


QUANTS = {"4 bits": nv.Quant.affine(64, 4), "8 bits": nv.Quant.affine(32, 8), **{mode: nv.Quant.new(getattr(nv.QuantMode, mode)) for mode in MODES}}


@pytest.mark.parametrize("quant", list(QUANTS))
@pytest.mark.parametrize("tokens,choices,count,dims,hidden,ordered", [(2, 2, 16, 2176, 2368, False), (5, 8, 8, 1088, 2368, True), (31, 2, 8, 1024, 1088, True)])
def test_few_pairs(quant, tokens, choices, count, dims, hidden, ordered):
    """The layer's experts, in whichever order the rule picks, against the products of every pair: bfloat16 products of the same weights,
    exact or in float32 on both sides, whose sums may fall to the next value, twice."""
    torch.manual_seed(tokens)
    quant = QUANTS[quant]

    def projection(n, k):
        q = nv.quantize((torch.randn(count, n, k, device="cuda") * 0.05).bfloat16(), quant)
        return layers.SwitchProjection(q.weight, q.scales, q.biases, (torch.randn(count, n, device="cuda") * 0.1).bfloat16(), q.quant)
    glu = layers.SwitchGlu(projection(hidden, dims), projection(hidden, dims), projection(dims, hidden))
    x = torch.randn(1, tokens, dims, device="cuda").bfloat16()
    ids = torch.stack([torch.randperm(count, device="cuda")[:choices] for _ in range(tokens)]).to(torch.int32).reshape(1, tokens, choices)
    assert nv.ops.moe_ordered(glu.up_proj.quantized(), x.dtype, tokens, choices, count, 3 * hidden * dims) == ordered
    xe = x.reshape(1, tokens, 1, 1, dims)
    gate, up = (p.forward(xe, ids, add_bias=False) for p in (glu.gate_proj, glu.up_proj))
    want = glu.down_proj.forward(glu.gated(gate, up, ids), ids).squeeze(-2).float()
    for block in (glu, glu.fuse_gate_up()):
        got = block.forward(x, ids).float()
        # (a hidden state that falls to the next value moves an output by 2^-8 of one of its terms, at random over them)
        assert (got - want).abs().max() <= 2 * 2.0 ** -7 * want.abs().max()


def test_few_pairs_hold_affine_weights_in_float32():
    """Against float64: few sorted pairs as far from it as pairs one by one, whose kernel holds float32 weights; the outputs' rounding
    (values are at most 2^-7 of them apart, errors uniform: 2^-7 / sqrt(12) in the mean square) is all that is left."""
    torch.manual_seed(11)
    quant = nv.Quant.affine(64, 4)
    q = nv.quantize((torch.randn(3, 1152, 1024, device="cuda") * 0.02 + 0.3).bfloat16(), quant)  # (biases far above the codes' steps)
    x = torch.randn(21, 1024, device="cuda").bfloat16()
    ids = torch.arange(3, device="cuda").repeat_interleave(7).to(torch.int32)
    rows = torch.arange(21, dtype=torch.int32, device="cuda")
    got = nv.gather_qmm_grouped(x, q, rows, ids, nv.sorted_offsets(ids, 3)).double()
    codes = nv.dequantize(nv.Quantized(q.weight, torch.ones_like(q.scales, dtype=torch.float32), torch.zeros_like(q.scales, dtype=torch.float32), quant))
    spread = lambda t: t.double().repeat_interleave(64, dim=-1)
    dense = codes.double() * spread(q.scales) + spread(q.biases)
    want = torch.einsum("rk,rnk->rn", x.double().cpu(), dense.cpu()[ids.long().cpu()]).cuda()
    assert (got - want).norm() <= 2.0 ** -7 / 12 ** 0.5 * want.norm()


# Fewer than 64 pairs, whose affine weights are terms: groups of a block that split K (1024 and 1152 columns), a window's part at the end
# (K = 1504), weights of which one term is all, and a weight of zero.
@pytest.mark.parametrize("fmt", [(64, 1), (32, 2), (32, 3), (32, 4), (32, 5), (32, 6), (32, 8)], ids=str)
@pytest.mark.parametrize("dtype,n,k", [(torch.bfloat16, 1024, 512), (torch.float16, 1152, 1664), (torch.bfloat16, 1030, 640), (torch.float16, 1024, 1504)])
def test_infinities_in_few_pairs(fmt, dtype, n, k):
    """What is infinite or no number in a row of x gives that row what its product with the weights gives, and no other row anything."""
    if k % fmt[0]:
        pytest.skip("K is not whole groups")
    torch.manual_seed(n + k)
    dense = (torch.randn(2, n, k, device="cuda") * 0.05).to(dtype)
    q = nv.quantize(dense, nv.Quant.affine(*fmt))
    q.biases[:, 5], q.scales[0, 7, :] = 0.0, 1.0
    q.biases[0, 7, :] = -1.0 if fmt[1] > 1 else 0.0  # (weights of zero where the code is 1)
    x = torch.randn(40, k, device="cuda").to(dtype)
    ids = torch.tensor([0] * 17 + [1] * 23, dtype=torch.int32, device="cuda")
    run = lambda x: nv.gather_qmm_grouped(x, q, torch.arange(40, dtype=torch.int32, device="cuda"), ids, nv.sorted_offsets(ids, 2))
    odd = {0: {3: "inf"}, 4: {k - 1: "-inf"}, 16: {k // 2: "nan"}, 17: {0: "inf", 1: "inf"}, 39: {40: "-inf", k - 33: "inf"}}
    plain = run(x)
    for row, values in odd.items():
        for at, value in values.items():
            x[row, at] = float(value)
    got = run(x)
    same = [row for row in range(40) if row not in odd]
    assert torch.equal(got[same], plain[same])
    for row in odd:
        e = int(ids[row])
        want = (x[row].double().cpu() * unrounded(nv.Quantized(q.weight[e], q.scales[e], q.biases[e], q.quant)).cpu()).sum(-1)
        assert torch.equal(got[row].double().cpu().nan_to_num(nan=7.0), want.nan_to_num(nan=7.0)), row


@pytest.mark.parametrize("fmt", [(64, 2), (128, 3), (64, 4), (32, 5), (64, 6), (32, 8)], ids=str)
@pytest.mark.parametrize("dtype,k", [(torch.bfloat16, 1024), (torch.float16, 384)])
def test_sorted_gathers_round_each_weight_once(fmt, dtype, k):
    """However few their pairs are, where nobody asks for float32 weights: the bits that a pair has among 80, and far from those of
    float32 weights (biases above the codes' steps, rows of x that sum to nothing: what rounding does to a weight is not lost in the sum)."""
    torch.manual_seed(k)
    n = 1100  # (off whole blocks: one group of wavefronts, however many pairs)
    q = nv.quantize(torch.randn(2, n, k, device="cuda") * 0.02 + 0.3, nv.Quant.affine(*fmt))
    q = nv.Quantized(q.weight, q.scales.to(dtype), q.biases.to(dtype), q.quant)
    x = torch.randn(80, k // 2, device="cuda").to(dtype)
    x = torch.stack([x, -x], dim=-1).reshape(80, 1, k)
    ids = torch.tensor([0] * 30 + [1] * 50, dtype=torch.int32, device="cuda")
    gather = lambda rows: nv.gather_qmm(x[rows], q, None, ids[rows], nv.GatherQmm(sorted_indices=True))[:, 0]
    every, few = gather(slice(0, 80)), gather(slice(10, 60))
    assert torch.equal(few, every[10:60])
    exact = torch.stack([unrounded(nv.Quantized(q.weight[e], q.scales[e], q.biases[e], q.quant)) for e in range(2)])
    product = lambda weights: torch.matmul(weights[ids[10:60].long()], x[10:60].double().transpose(1, 2))[..., 0]
    want, unit = product(exact.to(dtype).double()), 2.0 ** (-8 if dtype == torch.bfloat16 else -11)
    # (an output's rounding is half a unit of it at most; a weight's, 2^-10 or 2^-13 of 0.3 at random, is some 3 % or 0.4 % of these sums)
    assert (few.double() - want).norm() <= unit * want.norm()
    assert (few.double() - product(exact)).norm() >= 2 * unit * want.norm()


def test_order_of_few_pairs():
    rule = nv.ops.moe_ordered
    q = lambda quant, scale=None: nv.Quantized(None, None, None, quant, scale)
    mx, affine, nvfp4 = nv.Quant.new(nv.QuantMode.MXFP4), nv.Quant.affine(64, 4), nv.Quant.new(nv.QuantMode.NVFP4)
    many = 3 * 2880 * 2880
    assert rule(q(mx), torch.bfloat16, 5, 8, 8, many) and rule(q(nvfp4), torch.float16, 5, 8, 8, many) and rule(q(affine), torch.bfloat16, 5, 8, 8, many)
    assert not rule(q(mx), torch.bfloat16, 1, 32, 32, many) and not rule(q(mx), torch.float32, 5, 8, 8, many)
    assert not rule(q(nvfp4, torch.ones(8)), torch.bfloat16, 5, 8, 8, many)
    assert rule(q(affine), torch.float32, 64, 1, 8, 1) and not rule(q(affine), torch.bfloat16, 63, 1, 64, many)


@pytest.mark.parametrize("mode,size", [("MXFP8", 1e-4), ("MXFP4", 1e-7)])
def test_few_float16_pairs_of_small_scales(mode, size):
    """Block scales so small that float16 does not hold a code times its scale: the layer gives what the kernel of pairs one by one
    gives, whose scales multiply in float32 (its products within float32 sums and an output's rounding of float64)."""
    torch.manual_seed(3)
    quant, (count, dims, hidden) = nv.Quant.new(getattr(nv.QuantMode, mode)), (8, 1088, 2368)

    def projection(n, k, size):
        q = nv.quantize(torch.randn(count, n, k, device="cuda") * size, quant)
        return layers.SwitchProjection(q.weight, q.scales, q.biases, None, q.quant)
    glu = layers.SwitchGlu(projection(hidden, dims, size), projection(hidden, dims, size), projection(dims, hidden, 0.05))
    x = (torch.randn(1, 5, dims, device="cuda") * 5e3).half()
    ids = torch.stack([torch.randperm(count, device="cuda") for _ in range(5)]).to(torch.int32).reshape(1, 5, 8)
    xe = x.reshape(1, 5, 1, 1, dims)
    gate, up = (p.forward(xe, ids, add_bias=False) for p in (glu.gate_proj, glu.up_proj))
    exact = nv.dequantize(glu.up_proj.quantized(), torch.float32)[ids.long()[0]].double()
    want = torch.matmul(exact, x.double().reshape(5, 1, dims, 1))[..., 0]
    assert ((up.reshape(5, 8, hidden).double() - want).abs() <= 2.0 ** -10 * want.abs() + 1e-6 * want.abs().max()).all()
    want = glu.down_proj.forward(glu.gated(gate, up, ids), ids).squeeze(-2)
    assert torch.equal(glu.forward(x, ids), want)
    got = glu.fuse_gate_up().forward(x, ids)
    assert torch.equal(got, want)


@pytest.mark.parametrize("fmt,n,k", [((32, 8), 2176, 4096), ((64, 4), 2048, 8192), ((32, 2), 2304, 4128), ((32, 3), 2048, 4096), ("NVFP4", 2048, 8192)], ids=str)
@pytest.mark.parametrize("pairs", [40, 90])
def test_gated_pairs_of_long_rows(fmt, n, k, pairs):
    """Rows whose groups' scales are many: the gated product is bit for bit its two products and the activation, however long they are."""
    torch.manual_seed(k + pairs)
    quant = nv.Quant.new(getattr(nv.QuantMode, fmt)) if isinstance(fmt, str) else nv.Quant.affine(*fmt)
    gate, up = (nv.quantize((torch.randn(3, n // 2, k, device="cuda") * k ** -0.5).bfloat16(), quant) for _ in range(2))
    pair = lambda a, b: None if a is None else nv.ops.pair_rows(a, b, 1)
    both = nv.Quantized(pair(gate.weight, up.weight), pair(gate.scales, up.scales), pair(gate.biases, up.biases), quant)
    x = torch.randn(pairs, k, device="cuda").bfloat16()
    ids = torch.sort(torch.randint(0, 3, (pairs,), device="cuda")).values.to(torch.int32)
    rows, offsets = torch.arange(pairs, dtype=torch.int32, device="cuda"), nv.sorted_offsets(ids, 3)
    product = lambda q: nv.gather_qmm_grouped(x, q, rows, ids, offsets)
    assert torch.equal(nv.ops.gather_qmm_glu(x, both, rows, ids, offsets, "swiglu"), nv.ops.glu(product(gate), product(up), "swiglu"))


@pytest.mark.parametrize("quant,dims,hidden,taken", [("NVFP4", 2896, 2864, False), ("NVFP4", 2896, 2880, True), ("NVFP4", 2880, 2864, True), ("NVFP4", 2880, 2848, True), ("4 bits", 4096, 2048, True)])
def test_few_pairs_are_ordered_for_the_grouped_kernel_alone(quant, dims, hidden, taken, monkeypatch):
    """Rows that it does not take (NVFP4 of half a block of 32) run one by one in either order: without the order where no projection gains."""
    torch.manual_seed(hidden)
    quant, count = QUANTS[quant], 8

    def projection(n, k):
        q = nv.quantize((torch.randn(count, n, k, device="cuda") * 0.02).bfloat16(), quant)
        return layers.SwitchProjection(q.weight, q.scales, q.biases, None, q.quant)
    glu = layers.SwitchGlu(projection(hidden, dims), projection(hidden, dims), projection(dims, hidden))
    x = torch.randn(1, 5, dims, device="cuda").bfloat16()
    ids = torch.stack([torch.randperm(count, device="cuda") for _ in range(5)]).to(torch.int32).reshape(1, 5, 8)
    ordered = []
    order = nv.ops.moe_order
    monkeypatch.setattr(nv.ops, "moe_order", lambda *args: ordered.append(1) or order(*args))
    glu.forward(x, ids)
    assert bool(ordered) == taken
    for p, k in ((glu.up_proj, dims), (glu.gate_proj, dims), (glu.down_proj, hidden)):
        assert nv.ops.gather_sorted_takes(p.quantized(), x.dtype, 40) == (k % 32 == 0)


def test_few_pairs_are_ordered_where_all_three_projections_gain():
    """A gate whose weights the ordered kernel would hold less precisely keeps the block's pairs one by one."""
    torch.manual_seed(5)
    count, dims, hidden = 8, 1088, 2368

    def projection(n, k, quant, size):
        q = nv.quantize(torch.randn(count, n, k, device="cuda") * size, quant)
        parts = (q.scales.half(), q.biases.half()) if q.biases is not None else (q.scales, None)
        return layers.SwitchProjection(q.weight, *parts, None, q.quant)
    affine = nv.Quant.affine(64, 4)
    glu = layers.SwitchGlu(projection(hidden, dims, nv.Quant.new(nv.QuantMode.MXFP8), 1e-4), projection(hidden, dims, affine, 0.05), projection(dims, hidden, affine, 0.05))
    x = (torch.randn(1, 5, dims, device="cuda") * 30).half()
    ids = torch.stack([torch.randperm(count, device="cuda") for _ in range(5)]).to(torch.int32).reshape(1, 5, 8)
    xe = x.reshape(1, 5, 1, 1, dims)
    gate, up = (p.forward(xe, ids, add_bias=False) for p in (glu.gate_proj, glu.up_proj))
    assert torch.equal(glu.forward(x, ids), glu.down_proj.forward(glu.gated(gate, up, ids), ids).squeeze(-2))


# The first term alone, or two of three, are far from this: rows of x that sum to nothing leave nothing of the biases but what their rounding
# to the terms lost (a weight of 0.3 to one term, a hundred times the bound and more).  `wide`: 8-bit codes of 248 to 255 beside a bias
# that a term holds, their sum with it within half a unit of that term: sixteen bits are left for the others (two terms: nine times the bound).
@pytest.mark.parametrize("fmt,dtype,n,k,wide", [((64, 2), torch.bfloat16, 1100, 1024, False), ((64, 4), torch.float16, 1152, 1664, False), ((128, 5), torch.bfloat16, 1030, 512, False),
                                                ((32, 8), torch.float16, 1100, 1024, False), ((32, 8), torch.bfloat16, 1152, 1664, True), ((32, 8), torch.bfloat16, 1030, 512, True)], ids=str)
def test_few_pairs_hold_every_term_of_their_weights(fmt, dtype, n, k, wide):
    """Every output within its own rounding and float32 sums of float64's product of the float32 weights."""
    torch.manual_seed(n + fmt[1])
    q = nv.quantize(torch.randn(2, n, k, device="cuda") * 0.02 + 0.3, nv.Quant.affine(*fmt))
    codes, scales, biases = q.weight, q.scales.to(dtype), q.biases.to(dtype)
    if wide:
        codes = (codes.view(torch.int32) | -0x07070708).view(codes.dtype)  # (0xF8F8F8F8)
        scales, biases = torch.full_like(scales, 1.42 * 2.0 ** -18), torch.full_like(biases, 0.71)
    q = nv.Quantized(codes, scales, biases, q.quant)
    x = torch.randn(40, k // 2, device="cuda").to(dtype)
    x = torch.stack([x, -x], dim=-1).reshape(40, k)
    ids = torch.tensor([0] * 17 + [1] * 23, dtype=torch.int32, device="cuda")
    got = nv.gather_qmm_grouped(x, q, torch.arange(40, dtype=torch.int32, device="cuda"), ids, nv.sorted_offsets(ids, 2)).double().cpu()
    weights = torch.stack([unrounded(nv.Quantized(q.weight[e], q.scales[e], q.biases[e], q.quant)) for e in range(2)]).float().double().cpu()
    unit = 2.0 ** (-8 if dtype == torch.bfloat16 else -11)
    for row in range(40):
        terms = weights[int(ids[row])] * x[row].double().cpu()
        want = terms.sum(-1)
        # half a unit of the output; and up to three matrix instructions for 32 values of K, each of whose sums is within 2^-24 of a partial
        # sum, which neighbours that cancel keep within four products of the sum itself: at random, five deviations
        bound = unit * want.abs() + 5 * (3 * k / 32) ** 0.5 * 2.0 ** -24 * (4 * terms.abs().amax(-1) + want.abs())
        assert ((got[row] - want).abs() <= bound).all(), row
