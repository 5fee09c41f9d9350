"""The tiles of the products that expand codes themselves (csrc/qmm_kernel.h, csrc/qmk_kernel.h): which of them a product runs on, and
qmk_kernel's, whose wavefronts take quarters of K, against float64 over the weights they multiply."""
import ctypes as C

import numpy as np
import pytest
import torch

import nuvec_amd as nv
from nuvec_amd import _lib, ops
from nuvec_amd.layers import QuantizedLinear

pytestmark = pytest.mark.gpu


def quant_of(form):
    return nv.Quant.new(getattr(nv.QuantMode, form)) if isinstance(form, str) else nv.Quant.affine(*form)


@pytest.mark.parametrize("m,n,k,form,dtype,tile", [
    (2048, 14336, 4096, (64, 4), torch.bfloat16, "qmm_kernel<256,256>"),
    (258, 16291, 1408, "MXFP4", torch.bfloat16, "qmm_kernel<128,128>"),
    (512, 4096, 14336, (64, 4), torch.bfloat16, "qmk_kernel<128,128>"),
    (126, 7681, 6016, "MXFP8", torch.float16, "qmk_kernel<128,128>"),
    (300, 64, 128, (64, 4), torch.bfloat16, "qmk_kernel<64,128>"),
    (700, 1500, 2048, "NVFP4", torch.float16, "qmk_kernel<64,128>"),
])
def test_the_query_tells_the_tiled_kernels_apart(m, n, k, form, dtype, tile):
    quant = quant_of(form)
    assert ops.quantized_matmul_kernel(m, n, k, quant, dtype) == "qmm_kernel"
    assert nv.quantized_matmul_tile(m, n, k, quant, dtype) == tile


def test_other_kernels_keep_their_names():
    q4, bf16 = nv.Quant.affine(64, 4), torch.bfloat16
    for p in ((1, 14336, 4096, q4, bf16), (16, 4096, 4096, q4, bf16), (64, 14336, 4096, q4, bf16), (33, 4096, 4096, q4, torch.float32),
              (20, 9001, 2112, q4, bf16), (517, 4096, 4096, nv.Quant.affine(64, 3), bf16)):
        assert ops.quantized_matmul_tile(*p) == ops.quantized_matmul_kernel(*p)
    with pytest.raises(nv.Unsupported):
        ops.quantized_matmul_tile(1, 64, 64, q4, bf16, batch=70000)


@pytest.mark.parametrize("m,n,k,bits,dense", [
    (517, 4096, 4096, 1, True), (517, 4096, 4096, 2, True), (517, 4096, 4096, 4, True), (517, 4096, 4096, 8, True),  # us 39 / 48, 39 / 45, 41 / 46, 42 / 45
    (768, 6144, 8192, 4, True), (768, 6144, 8192, 8, True),      # 120 / 134, 122 / 136
    (640, 4096, 4096, 4, False), (640, 6144, 8192, 8, False),    # 49 / 43, 100 / 82
    (512, 4096, 4096, 4, False), (768, 4096, 8192, 8, False),    # 43 / 34, 88 / 77
])
def test_the_weight_is_dequantized_once_where_that_is_faster(m, n, k, bits, dense):
    """Timed on both sides (us, dequantized / codes expanded in the product)."""
    quant = nv.Quant.affine(64, bits)
    assert (nv.quantized_matmul_kernel(m, n, k, quant, torch.bfloat16) == "qmm_dense_kernel") == dense


FORMS = [(32, 1), (128, 2), (32, 3), (64, 4), (32, 5), (32, 6), (64, 8), "MXFP4", "MXFP8", "NVFP4"]


def weights(q, dtype):
    """The weights that a product of two matrices multiplies, in float64: the CPU's of rows that take those (fewer than 1024 outputs, bfloat16 fewer than
    8192), else code * scale + bias rounded once; block formats exactly."""
    if q.quant.mode != nv.QuantMode.AFFINE or q.weight.shape[-2] < (8192 if dtype == torch.bfloat16 else 1024):
        return nv.dequantize(q, dtype).double()
    group = q.quant.group_size
    codes = nv.dequantize(nv.Quantized(q.weight, torch.ones_like(q.scales, dtype=torch.float32), torch.zeros_like(q.biases, dtype=torch.float32), q.quant)).double()
    spread = lambda t: t.double().repeat_interleave(group, dim=-1)
    exact = codes * spread(q.scales) + spread(q.biases)  # (codes, scales and biases of 16 bits: exact)
    if dtype == torch.float16:
        return torch.from_numpy(exact.cpu().numpy().astype(np.float16)).cuda().double()
    return exact.float().to(dtype).double()


def product(m, n, k, form, dtype):
    gen = torch.Generator(device="cuda").manual_seed(m + n + k)
    make = lambda *s: torch.randn(*s, generator=gen, device="cuda")
    return nv.quantize((make(n, k) * 0.02).to(dtype), quant_of(form)), make(m, k).to(dtype), make(n).to(dtype)


def split_of(m, n, k, quant, dtype):
    """The parts of K of a tiled product, by the size of the float32 partial sums."""
    d = _lib.QmmDescC()
    d.quant, d.dtype, d.transpose, d.m, d.n, d.k = quant._c(), ops._CODE[dtype], 1, m, n, k
    return max(1, _lib.load().nvq_quantized_matmul_workspace_bytes(C.byref(d)) // (4 * m * n))


def first_on(tile, split, shapes, form, dtype):
    quant, group = quant_of(form), max(quant_of(form).group_size, 32)
    for m, n, k in shapes:
        if k % group == 0 and nv.quantized_matmul_tile(m, n, k, quant, dtype) == tile and (split_of(m, n, k, quant, dtype) > 1) == split:
            return m, n, k
    if torch.cuda.get_device_properties(0).multi_processor_count != 256:
        pytest.skip("another number of compute units: other tiles")
    raise AssertionError(f"no product of {form} on {tile}")


# Tails of rows and of weight rows; a last window of K of one quarter, two, three and four; one window and fewer than the stages under way
WHOLE_128 = [(3000, 1001, 1440), (2050, 1290, 1984), (2050, 1001, 2144), (2050, 1290, 2048), (1500, 1290, 1024), (1100, 2050, 1024), (641, 5100, 512), (1300, 2500, 640), (1200, 2700, 1152)]
SPLIT_128 = [(897, 515, 16544), (641, 1040, 8256), (641, 1040, 8192)]
WHOLE_64 = [(1300, 700, 1056), (700, 390, 96), (700, 900, 832), (700, 900, 704), (700, 900, 768)]


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("form", FORMS, ids=str)
@pytest.mark.parametrize("tile,split,shapes", [("qmk_kernel<128,128>", False, WHOLE_128), ("qmk_kernel<128,128>", True, SPLIT_128), ("qmk_kernel<64,128>", False, WHOLE_64)],
                         ids=["128", "128 split", "64"])
def test_quarters_against_float64(tile, split, shapes, form, dtype):
    """The tiles whose wavefronts take quarters of K.  Bound: one rounding of the output, u |out|, one more for the bias, and float32 sums of K products,
    their roundings random: 2^-24 x sqrt(K) x the product of the operands' norms."""
    m, n, k = first_on(tile, split, shapes, form, dtype)
    q, x, bias = product(m, n, k, form, dtype)
    w = weights(q, dtype)
    rows = torch.cat([torch.arange(0, m, 17, device="cuda"), torch.arange(max(0, m - 130), m, device="cuda")])
    want = x[rows].double() @ w.T
    u, sums = 2.0 ** (-8 if dtype == torch.bfloat16 else -11), 2.0 ** -24 * k ** 0.5 * x[rows].double().norm(dim=1, keepdim=True) * w.norm(dim=1)
    got = nv.quantized_matmul(x, q)
    assert ((got[rows].double() - want).abs() <= u * want.abs() + sums).all()
    with_bias = QuantizedLinear(q.weight, q.scales, q.biases, bias, q.quant)(x)[rows].double()
    assert ((with_bias - want - bias.double()).abs() <= u * (want.abs() + (want + bias.double()).abs()) * 1.01 + sums).all()
    # the entry point without a workspace: the same bits
    d, y, p = _lib.QmmDescC(), torch.empty_like(got), ops._ptr
    d.quant, d.dtype, d.transpose, d.m, d.n, d.k = q.quant._c(), ops._CODE[dtype], 1, m, n, k
    _lib.check(_lib.load().nvq_quantized_matmul_static(C.byref(d), p(x), p(q.weight), p(q.scales), p(q.biases), p(y), ops._stream()))
    assert torch.equal(y, got)


@pytest.mark.parametrize("m,n,k,form,dtype", [(65, 8256, 896, (64, 4), torch.bfloat16), (80, 9000, 640, (32, 3), torch.bfloat16), (40, 24000, 320, (64, 6), torch.float16)])
def test_few_rows_of_a_short_k(m, n, k, form, dtype):
    """Up to 80 rows and K < 1100 products take the plan's tile as others do; before a bias affine ones sum in qmm_kernel's order.  Both within their
    roundings of float64 (test_quarters_against_float64)."""
    first_on("qmk_kernel<64,128>", False, [(m, n, k)], form, dtype)
    q, x, bias = product(m, n, k, form, dtype)
    w = weights(q, dtype)
    want, u = x.double() @ w.T, 2.0 ** (-8 if dtype == torch.bfloat16 else -11)
    sums = 2.0 ** -24 * k ** 0.5 * x.double().norm(dim=1, keepdim=True) * w.norm(dim=1)
    assert ((nv.quantized_matmul(x, q).double() - want).abs() <= u * want.abs() + sums).all()
    with_bias = QuantizedLinear(q.weight, q.scales, q.biases, bias, q.quant)(x).double()
    assert ((with_bias - want - bias.double()).abs() <= u * (want.abs() + (want + bias.double()).abs()) * 1.01 + sums).all()


@pytest.mark.parametrize("tile,m,n,k", [("qmk_kernel<128,128>", 700, 1290, 1984), ("qmk_kernel<64,128>", 300, 700, 704)])
@pytest.mark.parametrize("form", [(64, 4), (64, 3), "MXFP8", "NVFP4"], ids=str)
def test_items_of_a_batch(form, tile, m, n, k):
    """Each item of a batch on the quarters' tiles: within one rounding and the float32 sums of float64, and another item's operands do not reach it."""
    gen = torch.Generator(device="cuda").manual_seed(m)
    make = lambda *s: torch.randn(*s, generator=gen, device="cuda")
    items = [(nv.quantize((make(n, k) * 0.02 * (i + 1)).bfloat16(), quant_of(form)), make(m, k).bfloat16()) for i in range(3)]
    if torch.cuda.get_device_properties(0).multi_processor_count == 256:
        assert nv.quantized_matmul_tile(m, n, k, quant_of(form), torch.bfloat16, batch=3) == tile
    stack = lambda name: None if getattr(items[0][0], name) is None else torch.stack([getattr(i[0], name) for i in items])
    x = torch.stack([i[1] for i in items])
    got = nv.quantized_matmul(x, nv.Quantized(stack("weight"), stack("scales"), stack("biases"), items[0][0].quant))
    for i, (q, xi) in enumerate(items):
        w = weights(q, torch.bfloat16)
        want, sums = xi.double() @ w.T, 2.0 ** -24 * k ** 0.5 * xi.double().norm(dim=1, keepdim=True) * w.norm(dim=1)
        assert ((got[i].double() - want).abs() <= 2.0 ** -8 * want.abs() + sums).all()
    again = x.clone()
    again[1, 5] = float("nan")
    odd = nv.quantized_matmul(again, nv.Quantized(stack("weight"), stack("scales"), stack("biases"), items[0][0].quant))
    assert torch.equal(odd[0], got[0]) and torch.equal(odd[2], got[2]) and odd[1, 5].isnan().all()


@pytest.mark.parametrize("tile,m,n,k", [("qmk_kernel<128,128>", 2050, 1290, 1984), ("qmk_kernel<64,128>", 700, 900, 704)])
@pytest.mark.parametrize("form,dtype", [((64, 8), torch.float16), ("MXFP4", torch.bfloat16)], ids=str)
def test_values_without_a_number(form, dtype, tile, m, n, k):
    """An infinity or a NaN in one row of x stays in that row, also in the last window of K, half of which lies past the end."""
    first_on(tile, False, [(m, n, k)], form, dtype)
    q, x, _ = product(m, n, k, form, dtype)
    plain, w = nv.quantized_matmul(x, q), weights(q, dtype)
    odd = x.clone()
    odd[7, 0], odd[150, k - 1], odd[m - 1, k - 40] = float("inf"), float("nan"), float("-inf")
    y = nv.quantized_matmul(odd, q)
    keep = [r for r in range(m) if r not in (7, 150, m - 1)]
    assert torch.equal(y[keep], plain[keep]) and y[150].isnan().all()
    for row, at, sign in ((7, 0, 1), (m - 1, k - 40, -1)):
        some = w[:, at] != 0  # (zero times infinity is no number)
        assert y[row][some].isinf().all() and (y[row][some] > 0).equal(sign * w[some, at] > 0)


@pytest.mark.parametrize("m,n,k,form,dtype", [
    (517, 4096, 4096, (64, 4), torch.bfloat16),    # the whole copy fits the scratch
    (1138, 4578, 12800, (64, 4), torch.bfloat16),  # two parts of whole tiles, the last one ragged
    (1809, 8191, 13696, (64, 3), torch.bfloat16),  # four
    (4096, 8191, 28672, (32, 1), torch.bfloat16),  # eight, of whole tiles but the last
    (2049, 1023, 14400, (64, 5), torch.float16),   # one; float16, the CPU's weights of fewer than 1024 outputs
])
def test_dequantized_in_the_scratch(m, n, k, form, dtype):
    """The entry point without a workspace dequantizes a weight in parts that fit the library's scratch: the same bits."""
    quant = quant_of(form)
    if torch.cuda.get_device_properties(0).multi_processor_count == 256:
        assert nv.quantized_matmul_kernel(m, n, k, quant, dtype) == "qmm_dense_kernel"
    gen = torch.Generator(device="cuda").manual_seed(n)
    words = torch.randint(-(1 << 31), 1 << 31, (n, k * quant.bits // 32), generator=gen, device="cuda", dtype=torch.int64).to(torch.int32).view(torch.uint32)
    scales = (torch.rand(n, k // quant.group_size, generator=gen, device="cuda") * 0.01 + 0.001).to(dtype)
    q = nv.Quantized(words, scales, -scales * 2, quant)
    x = torch.randn(m, k, generator=gen, device="cuda").to(dtype)
    want, y, p = nv.quantized_matmul(x, q), torch.empty(m, n, dtype=dtype, device="cuda"), ops._ptr
    d = _lib.QmmDescC()
    d.quant, d.dtype, d.transpose, d.m, d.n, d.k = quant._c(), ops._CODE[dtype], 1, m, n, k
    _lib.check(_lib.load().nvq_quantized_matmul_static(C.byref(d), p(x), p(q.weight), p(q.scales), p(q.biases), p(y), ops._stream()))
    assert torch.equal(y, want)
