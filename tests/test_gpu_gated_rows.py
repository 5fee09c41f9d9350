"""The gate and up projections of several rows in one product with the gated epilogue (`quantized_matmul_glu_rows`) against the
two products and `glu`, at the edges of its tiles: weights and roundings are the same, so what differs is the order in which K
is summed."""
import pytest
import torch

pytestmark = pytest.mark.gpu

nv = pytest.importorskip("nuvec_amd")
from nuvec_amd import _lib, layers, ops  # noqa: E402

FORMS = [(64, 4), (32, 8), (64, 3), (128, 2), (32, 6), "MXFP4", "MXFP8", "NVFP4"]


def _projections(quant, hidden, k, dtype, bias, seed):
    gen = torch.Generator(device="cuda").manual_seed(seed)
    make = lambda *s: torch.randn(*s, generator=gen, device="cuda")
    out = []
    for _ in range(2):
        q = nv.quantize((make(hidden, k) * k ** -0.5).to(dtype), quant)
        out.append(layers.QuantizedLinear(q.weight, q.scales, q.biases, make(hidden).to(dtype) if bias else None, quant))
    return out, make


@pytest.mark.parametrize("form", FORMS, ids=str)
@pytest.mark.parametrize("rows,hidden,k,dtype,activation,bias", [
    (6, 1088, 640, torch.bfloat16, "swiglu", False),    # the fewest rows; off whole blocks of 128 outputs; few-row route
    (16, 1024, 4096, torch.float16, "geglu", True),     # a whole pass; eight slices of 512 values
    (17, 2752, 2048, torch.bfloat16, "swiglu_oai", False),  # one row into the second pass
    (31, 1088, 1152, torch.float16, "swiglu", True),    # K off slices of 512
    (12, 1216, 7168, torch.float16, "swiglu", False),   # K in two chunks
    (65, 640, 896, torch.bfloat16, "geglu", True),      # the CPU's weights (fewer than 1024 outputs); a second pass of four tiles
    (130, 4864, 896, torch.float16, "swiglu", False),
])
def test_equals_two_products_and_glu(form, rows, hidden, k, dtype, activation, bias):
    quant = nv.Quant.new(getattr(nv.QuantMode, form)) if isinstance(form, str) else nv.Quant.affine(*form)
    (gate, up), make = _projections(quant, hidden, k, dtype, bias, rows + hidden)
    pair = lambda a, b: None if a is None else ops.pair_rows(a, b, 0)
    both = layers.QuantizedLinear(pair(gate.weight, up.weight), pair(gate.scales, up.scales), pair(gate.biases, up.biases), pair(gate.bias, up.bias), quant)
    x = make(rows, k).to(dtype)
    try:
        y = ops.quantized_matmul_glu_rows(x, both.quantized(), activation, bias=both.bias)
    except nv.Unsupported:  # (left to the two products: estimated faster, or weights held otherwise)
        assert (rows, k) != (31, 1152)
        return
    g, u = gate(x), up(x)
    want = ops.glu(g, u, activation)
    assert y.shape == want.shape and y.dtype == want.dtype
    # Two orders of a float32 sum: K / 32 matrix instructions and up to 16 parts, each within half a unit of float32 of the sum
    # of magnitudes S, which moves a projection by d <= 2 (K / 32 + 16) 2^-24 S and, where that crosses a rounding boundary, the
    # rounded one by one unit more; the activation's slopes are at most 1.2 (|up| + 1) in the gate and |gate| + 1 in the up.
    unit = 2.0 ** (-7 if dtype == torch.bfloat16 else -10)
    magnitudes = [x.double().abs() @ nv.dequantize(p.quantized(), dtype=torch.float32).double().abs().T for p in (gate, up)]
    dg, du = [2.0 * (k / 32 + 16) * 2.0 ** -24 * s for s in magnitudes]
    g, u, want = g.double(), u.double(), want.double()
    tolerance = (dg + unit * g.abs()) * 1.2 * (u.abs() + 1) + (du + unit * u.abs()) * (g.abs() + 1) + unit * want.abs()
    assert ((y.double() - want).abs() <= tolerance).all()
    assert (y.double() != want).float().mean() < 0.2


@pytest.mark.parametrize("rows,hidden,k,form", [(16, 11008, 1024, (32, 8)), (9, 14336, 512, (64, 4)), (33, 8192, 2048, (64, 4)), (40, 11008, 2560, (32, 4))])
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
def test_beside_the_batched_decode_kernel(rows, hidden, k, form, dtype):
    """That kernel rounds each weight once; the gated product holds them at least as precisely: no larger an error against the
    float64 product of the unrounded weights (the outputs' own rounding in both)."""
    quant = nv.Quant.affine(*form)
    (gate, up), make = _projections(quant, hidden, k, dtype, False, rows)
    assert ops.quantized_matmul_route(rows, hidden, k, quant, dtype) == "qmr_kernel"
    both = nv.Quantized(*(ops.pair_rows(getattr(gate, name), getattr(up, name), 0) for name in ("weight", "scales", "biases")), quant)
    x = make(rows, k).to(dtype)
    try:
        y = ops.quantized_matmul_glu_rows(x, both, "swiglu")
    except nv.Unsupported:
        return
    wide = lambda p: nv.dequantize(nv.Quantized(p.weight, p.scales.float(), p.biases.float(), quant)).double()
    g, u = x.double() @ wide(gate).T, x.double() @ wide(up).T
    want = torch.nn.functional.silu(g) * u
    error = lambda v: ((v.double() - want).norm() / want.norm()).item()
    assert error(y) <= 1.02 * error(ops.glu(gate(x), up(x), "swiglu"))


@pytest.mark.parametrize("form", [(64, 4), (32, 8), "MXFP4"], ids=str)
@pytest.mark.parametrize("shape", [(16,), (2, 9), (40,), (7, 1), (300,)])
def test_block_native_and_composed_agree(form, shape, monkeypatch):
    quant = nv.Quant.new(getattr(nv.QuantMode, form)) if isinstance(form, str) else nv.Quant.affine(*form)
    (gate, up), make = _projections(quant, 2752, 2048, torch.bfloat16, False, 3)
    q = nv.quantize((make(2048, 2752) * 0.02).to(torch.bfloat16)[:, :2752 // 64 * 64].contiguous(), quant)
    down = layers.QuantizedLinear(q.weight, q.scales, q.biases, None, quant)
    mlp = layers.Mlp(gate, up, down).fuse_gate_up()
    x = make(*shape, 2048).to(torch.bfloat16)
    y = mlp(x)

    class Declines:
        def __getattr__(self, name):
            return lambda *args: None
    monkeypatch.setattr(_lib, "_native", Declines())
    monkeypatch.setattr(layers, "_native", Declines())
    assert torch.equal(y, mlp(x))
