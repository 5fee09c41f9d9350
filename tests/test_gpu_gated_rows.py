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
@pytest.mark.parametrize("rows,hidden,k,dtype,activation,bias,affine", [
    (6, 1088, 640, torch.bfloat16, "swiglu", False, True),    # the fewest rows; off whole blocks of 128 outputs; few-row route
    (31, 1088, 1152, torch.float16, "swiglu", True, True),    # a row short of two tiles; K of four turns of 256 and a half
    (17, 8192, 1152, torch.bfloat16, "geglu", True, True),    # a row into the second tile
    (65, 8256, 896, torch.bfloat16, "swiglu_oai", True, True),  # a second pass of four tiles of rows
    (130, 4864, 896, torch.float16, "swiglu", False, True),   # a third
    (256, 2048, 640, torch.float16, "geglu", False, True),    # the most rows
    # affine formats are left to the two products: the direct few-row kernel, which never rounds a weight, or the CPU's weights
    (16, 1024, 4096, torch.float16, "geglu", True, False),    # sixteen whole turns of 256
    (17, 2752, 2048, torch.bfloat16, "swiglu_oai", False, False),
    (12, 1216, 7168, torch.float16, "swiglu", False, False),  # a long K
    (65, 640, 896, torch.bfloat16, "geglu", True, False),     # fewer than 1024 outputs
])
def test_equals_two_products_and_glu(form, rows, hidden, k, dtype, activation, bias, affine):
    quant = nv.Quant.new(getattr(nv.QuantMode, form)) if isinstance(form, str) else nv.Quant.affine(*form)
    (gate, up), make = _projections(quant, hidden, k, dtype, bias, rows + hidden)
    pair = lambda a, b: None if a is None else ops.pair_rows(a, b, 0)
    both = layers.QuantizedLinear(pair(gate.weight, up.weight), pair(gate.scales, up.scales), pair(gate.biases, up.biases), pair(gate.bias, up.bias), quant)
    x = make(rows, k).to(dtype)
    if not affine and not isinstance(form, str):
        with pytest.raises(nv.Unsupported):
            ops.quantized_matmul_glu_rows(x, both.quantized(), activation, bias=both.bias)
        return
    y = ops.quantized_matmul_glu_rows(x, both.quantized(), activation, bias=both.bias)
    g, u = gate(x), up(x)
    want = ops.glu(g, u, activation)
    assert y.shape == want.shape and y.dtype == want.dtype
    # Two orders of a float32 sum: K / 32 matrix instructions and up to 16 parts, each within half a unit of float32 of the sum
    # of magnitudes S, which moves a projection by d <= 2 (K / 32 + 16) 2^-24 S and, where that crosses a rounding boundary, the
    # rounded one by one unit more; the activation's slopes are at most 1.2 (|up| + 1) in the gate and |gate| + 1 in the up.  Inside it
    # alpha times the gate, the sigmoid of that, its product with the gate, up + 1 and the last product are rounded as well, and each may
    # fall a unit aside: one unit more of the gate, three more of the result.
    unit = 2.0 ** (-7 if dtype == torch.bfloat16 else -10)
    magnitudes = [x.double().abs() @ nv.dequantize(p.quantized(), dtype=torch.float32).double().abs().T for p in (gate, up)]
    dg, du = [2.0 * (k / 32 + 16) * 2.0 ** -24 * s for s in magnitudes]
    g, u, want = g.double(), u.double(), want.double()
    tolerance = (dg + 2 * unit * g.abs()) * 1.2 * (u.abs() + 1) + (du + unit * u.abs()) * (g.abs() + 1) + 4 * unit * want.abs()
    assert ((y.double() - want).abs() <= tolerance).all()
    assert (y.double() != want).float().mean() < 0.2


@pytest.mark.parametrize("rows,hidden,k,form,taken", [
    (9, 14336, 512, (64, 4), True), (20, 14336, 1536, (32, 4), True),  # 4 bits: up to K = 1536
    (49, 8192, 2048, (64, 4), True),                                   # or beyond 48 rows
    (17, 8192, 1024, (32, 8), True), (32, 11008, 1024, (64, 8), True),  # 8 bits: K = 1024 from 17 rows on
    (33, 8192, 2048, (64, 4), False), (48, 11008, 2560, (32, 4), False), (16, 11008, 1024, (32, 8), False), (17, 8192, 2048, (64, 8), False),
])
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
def test_beside_the_batched_decode_kernel(rows, hidden, k, form, taken, dtype):
    """That kernel rounds each weight once; the gated product holds them at least as precisely: no larger an error against the
    float64 product of the unrounded weights (the outputs' own rounding in both).  What it is slower at is refused."""
    quant = nv.Quant.affine(*form)
    (gate, up), make = _projections(quant, hidden, k, dtype, False, rows)
    assert ops.quantized_matmul_route(rows, hidden, k, quant, dtype) == "qmr_kernel"
    both = nv.Quantized(*(ops.pair_rows(getattr(gate, name), getattr(up, name), 0) for name in ("weight", "scales", "biases")), quant)
    x = make(rows, k).to(dtype)
    if not taken:
        with pytest.raises(nv.Unsupported):
            ops.quantized_matmul_glu_rows(x, both, "swiglu")
        return
    y = ops.quantized_matmul_glu_rows(x, both, "swiglu")
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


@pytest.mark.parametrize("rows", [4, 8, 16, 300])
def test_what_is_refused_costs_no_allocation(rows):
    """An MLP whose gate and up projections stay two products takes as many allocations with the pair beside them as without it."""
    quant = nv.Quant.affine(64, 4)
    (gate, up), make = _projections(quant, 1024, 512, torch.bfloat16, False, rows)
    q = nv.quantize((make(512, 1024) * 0.03).to(torch.bfloat16), quant)
    down = layers.QuantizedLinear(q.weight, q.scales, q.biases, None, quant)
    alone, paired = layers.Mlp(gate, up, down), layers.Mlp(gate, up, down).fuse_gate_up()
    x = make(rows, 512).to(torch.bfloat16)
    with pytest.raises(nv.Unsupported):
        p = paired.gate_up_proj
        ops.quantized_matmul_glu_rows(x, p.quantized(), "swiglu", bias=p.bias)

    def allocations(block):
        block(x)
        before = torch.cuda.memory_stats()["allocation.all.allocated"]
        block(x)
        return torch.cuda.memory_stats()["allocation.all.allocated"] - before

    assert allocations(paired) == allocations(alone)
