"""The gate and up projections of several rows as the one group of the grouped kernel, with the gated epilogue
(`quantized_matmul_glu_grouped`), against the two products and `glu` at the edges of its tiles, windows and groups."""
import ctypes as C
import random

import pytest
import torch

pytestmark = pytest.mark.gpu

nv = pytest.importorskip("nuvec_amd")
from nuvec_amd import _lib, layers, ops  # noqa: E402
from tests.test_gpu_gated_rows import _projections  # noqa: E402


def _check_gated(y, x, gate, up, activation, dtype):
    k = x.shape[1]
    g, u = gate(x), up(x)
    want = ops.glu(g, u, activation)
    assert y.shape == want.shape and y.dtype == want.dtype
    # (as beside the split-K kernel) Two orders of a float32 sum: K / 32 matrix instructions and up to 16 parts, each within half a unit of float32 of the sum
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


@pytest.mark.parametrize("rows,hidden,k,dtype,form,activation,bias", [
    (16, 11008, 4096, torch.float16, (32, 8), "swiglu", False),      # one whole tile of rows, four groups or two of whole windows
    (9, 8192, 1600, torch.bfloat16, (32, 8), "geglu", True),         # half a window at the end
    (34, 11712, 1984, torch.bfloat16, (64, 4), "swiglu", True),      # two rows into the third tile, 15 windows and a half
    (64, 9728, 1152, torch.float16, "MXFP4", "swiglu_oai", True),    # a whole pass
    (65, 9792, 2944, torch.bfloat16, (64, 3), "swiglu", False),      # a row into the second pass, 23 windows
    (144, 8704, 2240, torch.float16, "NVFP4", "geglu", True),
    (203, 9728, 3968, torch.bfloat16, "MXFP4", "swiglu", False),
    (256, 9728, 2944, torch.bfloat16, "MXFP8", "swiglu", True),      # the most rows
    (96, 14144, 2176, torch.bfloat16, (128, 4), "swiglu", True),
    (150, 11712, 2944, torch.float16, (64, 2), "geglu", False),
    (130, 8192, 1984, torch.bfloat16, (64, 6), "swiglu", True),      # a third pass of two rows
    (128, 13248, 4352, torch.float16, (64, 5), "swiglu", False),
])
def test_equals_two_products_and_glu(rows, hidden, k, dtype, form, activation, bias):
    """The grouped kernel with all rows as one group, which the block takes for these."""
    quant = nv.Quant.new(getattr(nv.QuantMode, form)) if isinstance(form, str) else nv.Quant.affine(*form)
    (gate, up), make = _projections(quant, hidden, k, dtype, bias, rows + hidden)
    pair = lambda a, b: None if a is None else ops.pair_rows(a, b, 0)
    both = layers.QuantizedLinear(pair(gate.weight, up.weight), pair(gate.scales, up.scales), pair(gate.biases, up.biases), pair(gate.bias, up.bias), quant)
    x = make(rows, k).to(dtype)
    y = ops.quantized_matmul_glu_grouped(x, both.quantized(), activation, bias=both.bias)
    _check_gated(y, x, gate, up, activation, dtype)


def test_refused():
    """Where the two products hold their weights more precisely, up to five rows, beyond 256, and K off whole steps."""
    for rows, hidden, k, form in [(5, 11008, 1024, (32, 8)), (257, 9728, 3968, "MXFP4"), (34, 11712, 1952, (32, 4)), (16, 14336, 4096, (64, 4)), (65, 640, 896, (64, 4))]:
        quant = nv.Quant.new(getattr(nv.QuantMode, form)) if isinstance(form, str) else nv.Quant.affine(*form)
        (gate, up), make = _projections(quant, hidden, k, torch.bfloat16, False, rows)
        both = nv.Quantized(*(None if getattr(gate, name) is None else ops.pair_rows(getattr(gate, name), getattr(up, name), 0) for name in ("weight", "scales", "biases")), quant)
        with pytest.raises(nv.Unsupported):
            ops.quantized_matmul_glu_grouped(make(rows, k).to(torch.bfloat16), both, "swiglu")


def test_float16_of_small_scales_stays_two_products():
    """MXFP4 where the two products' kernel multiplies a group's sum by its float32 scale: bfloat16 holds the weights as exactly, float16
    does not, so its block is bit for bit the composition."""
    rows, hidden, k = 64, 8192, 2048
    quant = nv.Quant.new(nv.QuantMode.MXFP4)
    for dtype in (torch.bfloat16, torch.float16):
        assert ops.quantized_matmul_route(rows, hidden, k, quant, dtype) == "qmd_kernel"
        torch.manual_seed(7)
        make = lambda *shape: torch.randn(shape, device="cuda")
        linear = lambda n, k, size: layers.QuantizedLinear(*(lambda q: (q.weight, q.scales, q.biases))(nv.quantize(make(n, k) * size, quant)), None, quant)
        gate, up, down = linear(hidden, k, 1e-7), linear(hidden, k, 1e-7), linear(k, hidden, 0.05)
        x = (make(rows, k) * 5e3).to(dtype)
        mlp = layers.Mlp(gate, up, down).fuse_gate_up()
        both = mlp.gate_up_proj.quantized()
        if dtype == torch.bfloat16:
            _check_gated(ops.quantized_matmul_glu_grouped(x, both, "swiglu"), x, gate, up, "swiglu", dtype)
        else:
            with pytest.raises(nv.Unsupported):
                ops.quantized_matmul_glu_grouped(x, both, "swiglu")
            assert torch.equal(mlp(x), down(ops.glu(gate(x), up(x), "swiglu")))


def test_both_questions_at_once():
    """`nvq_quantized_matmul_glu_several_takes` is the two questions it stands for, over the range of each."""
    rng, library = random.Random(4), _lib.load()
    seen = set()
    for _ in range(4000):
        mode = rng.choice(["affine"] * 4 + ["MXFP4", "MXFP8", "NVFP4"])
        quant = nv.Quant.affine(rng.choice([32, 64, 128]), rng.choice([1, 2, 3, 4, 5, 6, 8])) if mode == "affine" else nv.Quant.new(getattr(nv.QuantMode, mode))
        d = _lib.QmmDescC()
        d.quant, d.dtype, d.transpose = quant._c(), ops._CODE[rng.choice([torch.bfloat16, torch.float16, torch.float32])], 1
        d.m, d.n, d.k = rng.randint(1, 300), 128 * rng.randint(1, 230), rng.choice([32, 64, 128]) * rng.randint(1, 80)
        d.item_rows = d.m
        need, of_rows = C.c_size_t(7), C.c_size_t(7)
        got = library.nvq_quantized_matmul_glu_several_takes(C.byref(d), C.byref(need))
        rows = library.nvq_quantized_matmul_glu_rows_takes(C.byref(d), C.byref(of_rows))
        grouped = library.nvq_quantized_matmul_glu_grouped_takes(C.byref(d))
        assert got == (1 if grouped else 2 if rows else 0) and need.value == (of_rows.value if got == 2 else 0)
        assert library.nvq_quantized_matmul_glu_several_takes(C.byref(d), None) == got
        seen.add(got)
    assert seen == {0, 1, 2}
