"""The tiles whose wavefronts take quarters of K (csrc/qmk_kernel.h), against float64 over the weights they multiply: the CPU's for affine
rows of fewer than 1024 outputs (round(round(code * scale) + bias), crates/nuvec-core/src/kernels.rs:835-859), the exact ones of the
block formats.  Bound: one rounding of the output, u |out|, one more for the bias, and float32 sums of K products, their roundings
random: 2^-24 x sqrt(K) x the product of the operands' norms."""
import ctypes as C

import pytest
import torch

import nuvec_amd as nv
from nuvec_amd import _lib, ops
from nuvec_amd.layers import QuantizedLinear

pytestmark = pytest.mark.gpu

FORMS = [(32, 1), (64, 2), (32, 3), (64, 4), (128, 5), (32, 6), (64, 8), "MXFP4", "MXFP8", "NVFP4"]


# Tails of rows and of weight rows; K of one quarter past whole windows of 128, of two and of three; one window, fewer than the stages
# under way, and many; K in several parts; tiles of 64 and of 128 rows
@pytest.mark.parametrize("m,n,k", [(129, 130, 128), (300, 700, 384), (700, 259, 800), (1500, 390, 1088), (517, 1000, 992), (150, 640, 6272), (1030, 1001, 2048)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("form", FORMS, ids=str)
def test_against_float64(form, dtype, m, n, k):
    quant = nv.Quant.new(getattr(nv.QuantMode, form)) if isinstance(form, str) else nv.Quant.affine(*form)
    unit = 32 if isinstance(form, str) else max(form[0], 32)
    k = k // unit * unit
    gen = torch.Generator(device="cuda").manual_seed(m + k)
    make = lambda *s: torch.randn(*s, generator=gen, device="cuda").to(dtype)
    q = nv.quantize((make(n, k).float() * 0.02).to(dtype), quant)
    x, bias = make(m, k), make(n)
    w = nv.dequantize(q, dtype).double()
    want = x.double() @ w.T
    got, with_bias = nv.quantized_matmul(x, q), QuantizedLinear(q.weight, q.scales, q.biases, bias, quant)(x)
    u = 2.0 ** (-8 if dtype == torch.bfloat16 else -11)
    sums = 2.0 ** -24 * k ** 0.5 * x.double().norm(dim=1, keepdim=True) * w.norm(dim=1)
    assert ((got.double() - want).abs() <= u * want.abs() + sums).all()
    assert ((with_bias.double() - want - bias.double()).abs() <= u * (want.abs() + (want + bias.double()).abs()) * 1.01 + sums).all()
    # the entry point without a workspace: the same bits
    d, y, p = _lib.QmmDescC(), torch.empty_like(got), ops._ptr
    d.quant, d.dtype, d.transpose, d.m, d.n, d.k = quant._c(), ops._CODE[dtype], 1, m, n, k
    _lib.check(_lib.load().nvq_quantized_matmul_static(C.byref(d), p(x), p(q.weight), p(q.scales), p(q.biases), p(y), ops._stream()))
    assert torch.equal(y, got)


@pytest.mark.parametrize("form", [(64, 4), "MXFP8"], ids=str)
def test_a_batch_and_values_without_a_number(form):
    """Items of a batch are the single products bit for bit; an infinity or a NaN in one row of x stays in that row, also where a row's
    last window is a part of one."""
    quant = nv.Quant.new(getattr(nv.QuantMode, form)) if isinstance(form, str) else nv.Quant.affine(*form)
    m, n, k = 200, 520, 704
    gen = torch.Generator(device="cuda").manual_seed(3)
    make = lambda *s: torch.randn(*s, generator=gen, device="cuda").bfloat16()
    items = [nv.quantize((make(n, k).float() * 0.02).bfloat16(), quant) for _ in range(2)]
    x = make(2, m, k)
    stack = lambda name: None if getattr(items[0], name) is None else torch.stack([getattr(i, name) for i in items])
    got = nv.quantized_matmul(x, nv.Quantized(stack("weight"), stack("scales"), stack("biases"), quant))
    plain = nv.quantized_matmul(x[0], items[0])
    w = [nv.dequantize(i, torch.bfloat16).double() for i in items]
    for i in range(2):
        want, sums = x[i].double() @ w[i].T, 2.0 ** -24 * k ** 0.5 * x[i].double().norm(dim=1, keepdim=True) * w[i].norm(dim=1)
        assert ((got[i].double() - want).abs() <= 2.0 ** -8 * want.abs() + sums).all()
    odd = x[0].clone()
    odd[7, 0], odd[150, k - 1] = float("inf"), float("nan")
    y = nv.quantized_matmul(odd, items[0])
    keep = [r for r in range(m) if r not in (7, 150)]
    assert torch.equal(y[keep], plain[keep]) and y[150].isnan().all()
    first = w[0][:, 0] != 0  # (zero times infinity is no number)
    assert y[7][first].isinf().all() and (y[7][first] > 0).equal(w[0][first, 0] > 0)
