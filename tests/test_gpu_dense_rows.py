"""Many rows against the CPU's weights, dequantized once and multiplied densely (csrc/qmm_dense.hip), against float64 over the
dequantized weight (round(round(code * scale) + bias), crates/nuvec-core/src/kernels.rs:835-859).  Bound: one rounding of the output,
u |out|, one more for the bias, and float32 sums of K products, their roundings random: 2^-24 x sqrt(K) x the product of the
operands' norms."""
import pytest
import torch

import nuvec_amd as nv
from nuvec_amd import ops
from nuvec_amd.layers import QuantizedLinear

pytestmark = pytest.mark.gpu


# Both tiles, tails of rows and of weight rows, one step of K (fewer than the stages under way) and many
@pytest.mark.parametrize("m,n,k", [(517, 4096, 4096), (513, 4099, 2048), (2050, 3970, 1024), (1100, 6145, 512), (9000, 1025, 192), (30000, 1100, 64), (1536, 4096, 2048)])
@pytest.mark.parametrize("bits,group", [(1, 32), (2, 64), (3, 64), (4, 32), (5, 64), (6, 32), (8, 64)])
def test_against_float64(m, n, k, bits, group):
    torch.manual_seed(m + bits)
    q = nv.quantize((torch.randn(n, k, device="cuda") * 0.02).bfloat16(), nv.Quant.affine(group, bits))
    x, bias = torch.randn(m, k, device="cuda").bfloat16(), torch.randn(n, device="cuda").bfloat16()
    w = nv.dequantize(q).double()
    rows = torch.cat([torch.arange(0, m, 97, device="cuda"), torch.arange(max(0, m - 40), m, device="cuda")])
    want = x[rows].double() @ w.T
    got, with_bias = nv.quantized_matmul(x, q)[rows].double(), QuantizedLinear(q.weight, q.scales, q.biases, bias, q.quant)(x)[rows].double()
    u, sums = 2.0 ** -8, 2.0 ** -24 * k ** 0.5 * x[rows].double().norm(dim=1, keepdim=True) * w.norm(dim=1)
    assert ((got - want).abs() <= u * want.abs() + sums).all()
    assert ((with_bias - want - bias.double()).abs() <= u * (want.abs() + (want + bias.double()).abs()) * 1.01 + sums).all()


def test_replays_in_a_graph():
    """The weight's copy belongs to one call: captured, replayed after other work, equal to the eager result."""
    q = nv.quantize((torch.randn(4096, 1024, device="cuda") * 0.02).bfloat16(), nv.Quant.affine(64, 4))
    x = torch.randn(2048, 1024, device="cuda").bfloat16()
    want = nv.quantized_matmul(x, q)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        y = nv.quantized_matmul(x, q)
    for _ in range(3):
        nv.quantized_matmul(torch.randn_like(x), q)
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(y, want)


def test_workspace_is_bounded():
    """Half a gigabyte at most; the products of larger weights expand codes in the tiled kernel."""
    import ctypes as C

    from nuvec_amd import _lib
    ops._init(torch.empty(1, device="cuda"))
    for n, k in ((4096, 4096), (8191, 28672), (8191, 65536), (8000, 1 << 18)):
        d = _lib.QmmDescC()
        d.quant, d.dtype, d.transpose, d.m, d.n, d.k = nv.Quant.affine(64, 4)._c(), ops._CODE[torch.bfloat16], 1, 4096, n, k
        need = _lib.load().nvq_quantized_matmul_workspace_bytes(C.byref(d))
        assert need == (2 * n * k if n * k <= 1 << 28 else 0), (n, k, need)


@pytest.mark.parametrize("m,n,k", [(517, 4096, 4096), (2048, 3970, 1024), (517, 4096, 14336), (517, 2048, 2048)])
def test_without_a_workspace(m, n, k):
    """`nvq_quantized_matmul_static` expands codes in the product: the same bits, whether K is split or not."""
    import ctypes as C

    from nuvec_amd import _lib
    q = nv.quantize((torch.randn(n, k, device="cuda") * 0.02).bfloat16(), nv.Quant.affine(64, 4))
    x = torch.randn(m, k, device="cuda").bfloat16()
    want, got = nv.quantized_matmul(x, q), torch.empty(m, n, dtype=torch.bfloat16, device="cuda")
    d = _lib.QmmDescC()
    d.quant, d.dtype, d.transpose, d.m, d.n, d.k = q.quant._c(), ops._CODE[x.dtype], 1, m, n, k
    p = ops._ptr
    _lib.check(_lib.load().nvq_quantized_matmul_static(C.byref(d), p(x), p(q.weight), p(q.scales), p(q.biases), p(got), ops._stream()))
    assert torch.equal(got, want)
