"""Products of a few to a few dozen rows on the split-K kernel (`qms_kernel`), which the few-row and tiled routes hand what it is estimated
faster at: against the CPU's product (crates/nuvec-core/src/kernels.rs:1091-1142), at the ends of its turns of 256 values, its chunks
of codes, its tiles of rows and weight rows; and in every shape of block that it has, with K split over the grid and not."""
import ctypes as C

import numpy as np
import pytest
import torch

import nuvec_amd as nv
from nuvec_amd import _lib, ops
from oracle import ref
from tests.hip_backend import to_dev, to_host
from tests.test_gpu_parity import assert_rows_close, make_w, make_x

pytestmark = pytest.mark.gpu


def product(rng, fmt, m, n, k, dtype):
    w, x = make_w(rng, n, k, dtype), make_x(rng, m, k, dtype)
    if isinstance(fmt, str):
        mode = getattr(ref, fmt)
        group, bits = ref.FP_PARAMS[mode]
        packed, scales = ref.fp_quantize(w, dtype, mode)
        q = nv.Quantized(to_dev(packed), to_dev(scales), None, nv.Quant.new(getattr(nv.QuantMode, fmt)))
        return q, x, ref.quantized_matmul(x, packed, scales, None, mode=mode, group=group, bits=bits, dtype=dtype, threads=8)
    group, bits = fmt
    packed, scales, biases = ref.affine_quantize(w, dtype, group, bits)
    q = nv.Quantized(to_dev(packed), to_dev(scales), to_dev(biases), nv.Quant.affine(group, bits))
    return q, x, ref.quantized_matmul(x, packed, scales, biases, group=group, bits=bits, dtype=dtype, threads=8)


def workspace_bytes(m, n, k, quant, dtype):
    lib = _lib.load()
    d = _lib.QmmDescC()
    d.quant = _lib.QuantC(int(quant.mode.value), quant.group_size, quant.bits)
    d.dtype, d.transpose, d.m, d.item_rows, d.n, d.k = dtype, 1, m, m, n, k
    return lib.nvq_quantized_matmul_workspace_bytes(C.byref(d))


# One, two and four tiles of rows with tails; one and four wavefronts a group; K in and off whole turns, steps, chunks; splits of K.
SHAPES = [(5, 1130, 1184), (16, 4100, 11104), (9, 18734, 1600), (24, 1100, 2336), (20, 9001, 2112), (33, 2050, 5984), (62, 1030, 11072),
          (64, 5000, 480), (96, 1200, 2400), (7, 3536, 12832)]


@pytest.mark.parametrize("dtype", [ref.BF16, ref.F16])
@pytest.mark.parametrize("fmt", [(64, 2), (32, 3), (64, 4), (32, 4), (128, 5), (32, 6), (32, 8), (64, 8), "MXFP4", "MXFP8", "NVFP4"], ids=str)
def test_every_format_against_the_cpu_product(fmt, dtype):
    rng = np.random.default_rng(7300)
    unit = max(fmt[0], 32) if not isinstance(fmt, str) else 32
    for m, n, k in SHAPES:
        k = k // unit * unit
        q, x, want = product(rng, fmt, m, n, k, dtype)
        for scratch in (True, False):
            got = to_host(ops.quantized_matmul(to_dev(x), q, scratch=scratch))
            assert_rows_close(got, want, dtype, f"split rows {fmt} M={m} N={n} K={k} scratch={scratch}", exact_weights=isinstance(fmt, str))


@pytest.mark.parametrize("shape,split,fmt,dtype,m,n,k", [
    ("1,1,1", False, (64, 4), ref.BF16, 9, 18734, 1600),
    ("1,2,1", False, (64, 3), ref.BF16, 16, 7039, 1984),
    ("1,2,1", True, "MXFP4", ref.F16, 12, 5333, 8224),
    ("1,2,1", True, (64, 2), ref.BF16, 8, 1825, 8064),
    ("1,1,4", False, "MXFP8", ref.F16, 9, 13587, 736),
    ("1,1,4", True, (32, 8), ref.F16, 10, 1491, 5056),
    ("2,1,1", False, (64, 4), ref.F16, 20, 9001, 2112),
    ("2,1,1", True, (64, 8), ref.F16, 20, 4822, 8064),
    ("2,1,4", False, (32, 4), ref.BF16, 19, 15569, 576),
    ("2,1,4", True, (128, 4), ref.F16, 27, 1644, 4608),
    ("2,2,4", True, (128, 6), ref.F16, 30, 4432, 6528),
    ("2,2,4", True, (32, 2), ref.BF16, 20, 5737, 5408),
    ("4,1,4", False, (32, 4), ref.BF16, 64, 5000, 480),
    ("4,1,4", True, (64, 4), ref.BF16, 62, 1030, 11072),
    ("4,2,4", False, "NVFP4", ref.F16, 70, 11444, 928),
    ("4,2,4", True, (128, 3), ref.F16, 39, 5444, 1664),
])
def test_every_shape_of_block(shape, split, fmt, dtype, m, n, k):
    rng = np.random.default_rng(7350 + m)
    q, x, want = product(rng, fmt, m, n, k, dtype)
    if torch.cuda.get_device_properties(0).multi_processor_count == 256:  # (the cut is chosen by the compute units)
        assert ops.quantized_matmul_kernel(m, n, k, q.quant, torch.bfloat16 if dtype == ref.BF16 else torch.float16) == f"qms_kernel<{shape}>"
        assert (workspace_bytes(m, n, k, q.quant, dtype) > 0) == split
    for scratch in (True, False):
        got = to_host(ops.quantized_matmul(to_dev(x), q, scratch=scratch))
        assert_rows_close(got, want, dtype, f"split rows {shape} {fmt} M={m} N={n} K={k} scratch={scratch}", exact_weights=isinstance(fmt, str))


@pytest.mark.parametrize("m,n,k", [(16, 4096, 11008), (62, 2560, 11072), (31, 404, 13792)])
def test_bias_determinism_and_both_entry_points(m, n, k):
    """QuantizedLinear's bias is the separate addition bit for bit (crates/nuvec-nn/src/layers.rs:155-162) after a split of K as before it;
    two launches give the same bits; a row past the end of x, or a NaN in another row, changes nothing."""
    rng = np.random.default_rng(7400 + m)
    quant = nv.Quant.new(nv.QuantMode.NVFP4)
    if workspace_bytes(m, n, k, quant, 10) == 0:
        pytest.skip("K is not split on this device")
    q, x, _ = product(rng, "NVFP4", m, n, k, ref.BF16)
    xd = to_dev(x)
    plain = nv.quantized_matmul(xd, q)
    assert torch.equal(plain, nv.quantized_matmul(xd, q))
    bias = torch.randn(n, device="cuda").to(torch.bfloat16)
    from nuvec_amd.layers import QuantizedLinear
    assert torch.equal(QuantizedLinear(q.weight, q.scales, None, bias, q.quant)(xd), plain + bias)
    xd[m // 2, 3] = float("nan")
    odd = nv.quantized_matmul(xd, q)
    assert odd[m // 2].isnan().all()
    keep = [r for r in range(m) if r != m // 2]
    assert torch.equal(odd[keep], plain[keep])


def test_the_query_names_the_kernel_that_runs():
    """The routes of several 16-bit rows keep their names; the kernel behind them has its own query."""
    both = lambda *a, **k: (ops.quantized_matmul_route(*a, **k), ops.quantized_matmul_kernel(*a, **k))
    q4, bf16 = nv.Quant.affine(64, 4), torch.bfloat16
    route, kernel = both(20, 9001, 2112, q4, bf16)
    assert route in ("qmf_kernel", "qmm_kernel") and kernel.startswith("qms_kernel<2,")
    assert both(31, 404, 13792, nv.Quant.new(nv.QuantMode.NVFP4), bf16)[1].startswith("qms_kernel<")
    assert both(517, 4096, 4096, nv.Quant.affine(64, 3), bf16) == ("qmm_kernel", "qmm_dense_kernel")
    assert both(300, 64, 128, q4, bf16) == ("qmm_kernel", "qmm_kernel")
    for same in ((1, 14336, 4096, q4, bf16), (16, 4096, 4096, q4, bf16), (64, 14336, 4096, q4, bf16), (33, 4096, 4096, q4, torch.float32)):
        assert len(set(both(*same))) == 1
    assert len(set(both(4, 4096, 4096, q4, bf16, transpose=False))) == 1
    with pytest.raises(nv.Unsupported):
        ops.quantized_matmul_kernel(1, 64, 64, q4, bf16, batch=70000)


@pytest.mark.parametrize("m,n,k,fmt,dtype,route", [
    (4, 8118, 3328, (64, 8), torch.float16, "qmf_kernel"),     # 12.5 us there, 20.2 on the split-K kernel
    (13, 12640, 1920, (64, 8), torch.float16, "qmf_kernel"),   # 12.2 / 18.9
    (10, 6907, 3712, (128, 8), torch.bfloat16, "qmf_kernel"),  # 11.6 / 17.9
    (7, 4249, 3968, "MXFP8", torch.bfloat16, "qmf_kernel"),    # 9.6 / 12.1
    (14, 5482, 13824, "MXFP8", torch.bfloat16, "qmf_kernel"),  # 28.6 / 34.1
    (126, 7681, 6016, "MXFP8", torch.float16, "qmm_kernel"),   # 28.3 / 38.3
    (220, 3113, 5440, "MXFP8", torch.bfloat16, "qmm_kernel"),  # 26.9 / 35.4
])
def test_what_the_estimates_alone_would_take(m, n, k, fmt, dtype, route):
    """Products that the bare estimates hand to the split-K kernel, and that are faster on their route's own."""
    quant = nv.Quant.new(getattr(nv.QuantMode, fmt)) if isinstance(fmt, str) else nv.Quant.affine(*fmt)
    assert ops.quantized_matmul_route(m, n, k, quant, dtype) == ops.quantized_matmul_kernel(m, n, k, quant, dtype) == route


@pytest.mark.parametrize("dtype", [ref.BF16, ref.F16])
@pytest.mark.parametrize("fmt", [(64, 2), (32, 3), (64, 4), (32, 4), (128, 5), (32, 6), (32, 8), (64, 8), "MXFP4", "MXFP8", "NVFP4"], ids=str)
def test_the_few_row_kernel_keeps_batches(fmt, dtype):
    """The split-K kernel takes one product: batches stay on the few-row kernel, with weights rounded once and (fewer than 1024 outputs)
    with the CPU's."""
    rng = np.random.default_rng(7450)
    for b, m, n, k in ((2, 12, 1100, 2304), (3, 7, 2060, 1152), (2, 16, 700, 6272)):
        items = [product(rng, fmt, m, n, k, dtype) for _ in range(b)]
        stack = lambda of: None if of(items[0]) is None else torch.stack([of(i) for i in items])
        q = nv.Quantized(stack(lambda i: i[0].weight), stack(lambda i: i[0].scales), stack(lambda i: i[0].biases), items[0][0].quant)
        kernel = ops.quantized_matmul_kernel(m, n, k, q.quant, torch.bfloat16 if dtype == ref.BF16 else torch.float16, batch=b)
        assert kernel == "qmf_kernel", (b, m, n, k)
        got = to_host(ops.quantized_matmul(stack(lambda i: to_dev(i[1])), q))
        for i in range(b):
            assert_rows_close(got[i], items[i][2], dtype, f"few rows {fmt} item {i} of {b}, M={m} N={n} K={k}", exact_weights=isinstance(fmt, str))


def test_no_rounding_where_the_weights_and_sums_are_exact():
    """Small whole numbers: every cut of K gives the exact sums."""
    m, n, k = 20, 3000, 4128
    x = torch.randint(-2, 3, (m, k), device="cuda").to(torch.float16)
    w = torch.randint(-2, 3, (n, k), device="cuda").to(torch.float16)
    q = nv.quantize(w, nv.QuantMode.MXFP8)
    dense = nv.dequantize(q, torch.float32)
    assert torch.equal(dense, w.float())
    want = (x.double() @ dense.double().t()).to(torch.float16)
    assert torch.equal(nv.quantized_matmul(x, q), want)
