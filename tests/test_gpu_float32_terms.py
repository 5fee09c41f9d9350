"""float32 products on the bfloat16 matrix instruction (`qmm_f32_kernel`): codes are exact bfloat16 operands, x is three of them.
Against a product in float64 of the weights as real numbers, at the ends of its windows, spans, tiles and splits."""
import numpy as np
import pytest
import torch

import nuvec_amd as nv
from nuvec_amd import ops
from oracle import ref
from tests.hip_backend import to_dev, to_host
from tests.test_gpu_parity import make_w, make_x

pytestmark = pytest.mark.gpu

# A block's sum takes at most thirteen roundings (two a matrix instruction, one for its scale), an output one more per block of 64 or 32
# and two per split; each is off by 2^-25 in the mean of a partial sum no longer than the result, and they add as their root: under
# four units of 2^-24 up to K = 2048.  (0.7e-7 to 1.8e-7 measured.)
LIMIT = 4 * 2.0 ** -24


def quantized(fmt, w):
    if isinstance(fmt, str):
        packed, scales = ref.fp_quantize(w, ref.F32, getattr(ref, fmt))
        q = nv.Quantized(to_dev(packed), to_dev(scales), None, nv.Quant.new(getattr(nv.QuantMode, fmt)))
        return q, ref.fp_dequantize(packed, scales, getattr(ref, fmt), ref.F32).astype(np.float64)  # (a code times its scale is exact)
    group, bits = fmt
    packed, scales, biases = ref.affine_quantize(w, ref.F32, group, bits)
    n, k = w.shape
    streams = np.unpackbits(packed.view(np.uint8).reshape(n, -1), axis=1, bitorder="little").reshape(n, k, bits)
    codes = (streams * (1 << np.arange(bits))).sum(-1).reshape(n, k // group, group).astype(np.float64)
    dense = codes * scales.reshape(n, -1, 1).astype(np.float64) + biases.reshape(n, -1, 1).astype(np.float64)
    return nv.Quantized(to_dev(packed), to_dev(scales), to_dev(biases), nv.Quant.affine(group, bits)), dense.reshape(n, k)


@pytest.mark.parametrize("fmt", [(32, 1), (64, 2), (32, 3), (128, 4), (32, 4), (32, 5), (64, 6), (32, 8), "MXFP4", "MXFP8", "NVFP4"], ids=str)
@pytest.mark.parametrize("m,n,k", [(65, 5000, 160), (33, 5001, 224), (64, 4099, 288), (50, 6000, 352), (100, 3000, 1056), (300, 130, 1920), (17, 20000, 1024)])
def test_ends_of_windows_spans_and_splits(fmt, m, n, k):
    """K that ends inside a chunk of codes, a window, a step, a span; rows and weight rows that are no whole tiles; splits of K."""
    group, bits = ref.FP_PARAMS[getattr(ref, fmt)] if isinstance(fmt, str) else fmt
    k = -(-k // max(group, 32)) * max(group, 32)
    if m > 128:
        k = -(-k // 64) * 64
    rng = np.random.default_rng(6100 + m + k)
    x = make_x(rng, m, k, ref.F32)
    q, dense = quantized(fmt, make_w(rng, n, k, ref.F32))
    assert ops.quantized_matmul_route(m, n, k, q.quant, torch.float32) == "qmm_f32_kernel"
    want = x.astype(np.float64) @ dense.T
    for scratch in (True, False):  # K split over the grid, and not
        got = to_host(ops.quantized_matmul(to_dev(x), q, scratch=scratch)).astype(np.float64)
        assert np.linalg.norm(got - want) <= LIMIT * np.linalg.norm(want)


@pytest.mark.parametrize("fmt,m,n,k", [((32, 3), 801, 700, 1120), ((32, 8), 129, 2001, 1056), ("MXFP8", 132, 1989, 864), ("MXFP4", 160, 968, 544),
                                       ("MXFP4", 4, 5208, 160), ("MXFP4", 3, 12990, 512), ((64, 4), 32, 4099, 2048), ((128, 5), 6, 5858, 2048),
                                       ((64, 6), 21, 1731, 2048), ((128, 2), 2, 11651, 1920), ((128, 1), 3, 16001, 2048), ("MXFP8", 2, 13742, 1376)], ids=str)
def test_products_that_keep_the_vector_kernels_route(fmt, m, n, k):
    rng = np.random.default_rng(6150 + m + k)
    x = make_x(rng, m, k, ref.F32)
    q, dense = quantized(fmt, make_w(rng, n, k, ref.F32))
    assert ops.quantized_matmul_route(m, n, k, q.quant, torch.float32).startswith("qmv_")
    assert ops.quantized_matmul_kernel(m, n, k, q.quant, torch.float32) == "qmm_f32_kernel"
    want = x.astype(np.float64) @ dense.T
    for scratch in (True, False):
        got = to_host(ops.quantized_matmul(to_dev(x), q, scratch=scratch)).astype(np.float64)
        assert np.linalg.norm(got - want) <= LIMIT * np.linalg.norm(want)


@pytest.mark.parametrize("fmt", [(64, 4), (32, 8), "MXFP4", "MXFP8", "NVFP4"], ids=str)
def test_magnitudes_that_three_terms_do_not_hold(fmt):
    """Infinities, NaN and values near the end of float32's range give what the CPU's product gives; the other rows keep their bits."""
    rng = np.random.default_rng(6200)
    m, n, k = 40, 5000, 512
    x = make_x(rng, m, k, ref.F32)
    q, dense = quantized(fmt, make_w(rng, n, k, ref.F32))
    plain = to_host(nv.quantized_matmul(to_dev(x), q))
    odd = x.copy()
    odd[1, 7], odd[3, 200], odd[5, 511] = np.inf, -np.inf, np.nan
    odd[8, 100], odd[20, 0] = 3.0e38, -3.2e38
    got = to_host(nv.quantized_matmul(to_dev(odd), q))
    mode = getattr(ref, fmt) if isinstance(fmt, str) else ref.AFFINE
    want = ref.quantized_matmul(odd, to_host(q.weight), to_host(q.scales), None if q.biases is None else to_host(q.biases), mode=mode,
                                group=q.quant.group_size, bits=q.quant.bits, dtype=ref.F32, threads=8)
    assert np.array_equal(np.isnan(got), np.isnan(want)) and np.array_equal(np.isinf(got), np.isinf(want))
    infinite = np.isinf(want)
    assert np.array_equal(np.sign(got[infinite]), np.sign(want[infinite]))
    for row in (8, 20):
        exact = odd[row].astype(np.float64) @ dense.T
        assert np.linalg.norm(got[row] - exact) <= LIMIT * np.linalg.norm(exact)
    same = [r for r in range(m) if r not in (1, 3, 5, 8, 20)]
    assert np.array_equal(got[same], plain[same])


@pytest.mark.parametrize("fmt", [(64, 4), (32, 3), (128, 8), (64, 1), "MXFP4", "MXFP8", "NVFP4"], ids=str)
@pytest.mark.parametrize("k", [512, 2048])
def test_magnitudes_at_the_low_end_of_float32(fmt, k):
    """Rows of x down to the subnormal numbers keep all of their bits, alone and (block formats, where a zero is code zero and not a
    difference) beside ordinary values whose weights are zero.  A result of the least rows is itself near the end, 2^-149: half of
    that is allowed beside the bound above."""
    rng = np.random.default_rng(6250)
    m, n = 48, 5000
    w = make_w(rng, n, k, ref.F32) * np.float32(256.0)
    w[:, :128] = 0.0
    powers = np.array([0, -60, -95, -100, -104, -109, -112, -116, -120, -124, -126, -128], dtype=np.int32)
    x = np.ldexp(make_x(rng, m, k, ref.F32), powers[np.arange(m) % len(powers)][:, None]).astype(np.float32)
    if isinstance(fmt, str):
        x[24:, :128] = make_x(rng, 24, 128, ref.F32)
    q, dense = quantized(fmt, w)
    assert ops.quantized_matmul_route(m, n, k, q.quant, torch.float32) == "qmm_f32_kernel"
    want = x.astype(np.float64) @ dense.T
    for scratch in (True, False):
        got = to_host(ops.quantized_matmul(to_dev(x), q, scratch=scratch)).astype(np.float64)
        for row in range(m):
            assert np.linalg.norm(got[row] - want[row]) <= LIMIT * np.linalg.norm(want[row]) + np.sqrt(n) * 2.0 ** -150, (row, powers[row % len(powers)])


@pytest.mark.parametrize("fmt", [(64, 4), (32, 3), (128, 8), (32, 5), "MXFP4", "MXFP8", "NVFP4"], ids=str)
@pytest.mark.parametrize("m,n,k", [(70, 5001, 544), (33, 4096, 2048)])
def test_a_batch_of_infinities_and_nans(fmt, m, n, k):
    """What the split of x does not hold in every row: the outputs are those of the CPU's product, and take no more than a few times as
    long as others (W[4096,4096] of 4 bits at 33 rows 54 us against 17, at 512 rows 480 against 85)."""
    group = 32 if isinstance(fmt, str) else fmt[0]
    k = -(-k // group) * group
    rng = np.random.default_rng(6300 + k)
    x = make_x(rng, m, k, ref.F32)
    q, _ = quantized(fmt, make_w(rng, n, k, ref.F32))
    odd = x.copy()
    odd[np.arange(0, m, 2), rng.integers(0, k, len(range(0, m, 2)))] = np.inf
    odd[np.arange(1, m, 2), rng.integers(0, k, len(range(1, m, 2)))] = np.nan
    xd, od = to_dev(x), to_dev(odd)
    got = to_host(nv.quantized_matmul(od, q))
    mode = getattr(ref, fmt) if isinstance(fmt, str) else ref.AFFINE
    want = ref.quantized_matmul(odd, to_host(q.weight), to_host(q.scales), None if q.biases is None else to_host(q.biases), mode=mode,
                                group=q.quant.group_size, bits=q.quant.bits, dtype=ref.F32, threads=8)
    assert np.array_equal(np.isnan(got), np.isnan(want)) and np.array_equal(got[0::2][~np.isnan(want[0::2])], want[0::2][~np.isnan(want[0::2])])

    def us(t):
        times = []
        for _ in range(7):
            a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            a.record()
            for _ in range(5):
                nv.quantized_matmul(t, q)
            b.record()
            b.synchronize()
            times.append(a.elapsed_time(b))
        return min(times)

    assert us(od) < 12 * us(xd)
