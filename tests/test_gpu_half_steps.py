"""K of whole 32 values off the matrix-core kernels' whole steps of 64 (windows of 128): the last step begins early and what it
repeats is zeros in both operands.  Held to the CPU product (crates/nuvec-core/src/kernels.rs:1091-1142) at the bar of the
element type; an infinity where values repeat reaches the sums once."""
import numpy as np
import pytest
import torch

import nuvec_amd as nv
from nuvec_amd import ops
from oracle import ref
from tests.hip_backend import to_dev, to_host
from tests.test_gpu_parity import assert_rows_close, make_w, make_x

pytestmark = pytest.mark.gpu

TORCH = {ref.BF16: torch.bfloat16, ref.F16: torch.float16}
MODES = {"MXFP4": ref.MXFP4, "MXFP8": ref.MXFP8, "NVFP4": ref.NVFP4}
FORMATS = [(32, b) for b in (1, 2, 3, 4, 5, 6, 8)] + list(MODES)


def packed(rng, n, k, dtype, fmt):
    """A weight, its quant and the oracle's product of rows with it."""
    w = make_w(rng, n, k, dtype)
    if isinstance(fmt, str):
        codes, scales = ref.fp_quantize(w, dtype, MODES[fmt])
        group, bits = ref.FP_PARAMS[MODES[fmt]]
        want = lambda x: ref.quantized_matmul(x, codes, scales, None, mode=MODES[fmt], group=group, bits=bits, dtype=dtype, threads=8)
        return nv.Quantized(to_dev(codes), to_dev(scales), None, nv.Quant.new(getattr(nv.QuantMode, fmt))), want
    group, bits = fmt
    codes, scales, biases = ref.affine_quantize(w, dtype, group, bits)
    want = lambda x: ref.quantized_matmul(x, codes, scales, biases, group=group, bits=bits, dtype=dtype, threads=8)
    return nv.Quantized(to_dev(codes), to_dev(scales), to_dev(biases), nv.Quant.affine(group, bits)), want


# One whole step and a half, both tiles, tails of rows and of weight rows, K split over the grid (the last split a half step)
@pytest.mark.parametrize("fmt", FORMATS, ids=str)
@pytest.mark.parametrize("dtype,m,n,k", [(ref.BF16, 33, 1030, 96), (ref.F16, 130, 200, 160), (ref.F16, 600, 4500, 224), (ref.BF16, 40, 256, 4128)])
def test_tiles(fmt, dtype, m, n, k):
    rng = np.random.default_rng(7100 + m + k)
    q, want = packed(rng, n, k, dtype, fmt)
    rest = not isinstance(fmt, str) and n >= 1024 and dtype == ref.F16  # (weights of two terms on the grouped kernel)
    assert ops.quantized_matmul_route(m, n, k, q.quant, TORCH[dtype]) == ("qmg_kernel" if rest else "qmm_kernel")
    x = make_x(rng, m, k, dtype)
    assert_rows_close(to_host(nv.quantized_matmul(to_dev(x), q)), want(x), dtype, f"half step {fmt} M={m} N={n} K={k}", exact_weights=isinstance(fmt, str))


# Windows of 128 and 32, 64 or 96 values more, one step alone; rows of fewer than 1024 outputs (the CPU's weights) and of more;
# experts with no rows, with one and with more than a pass of 64.
@pytest.mark.parametrize("fmt", FORMATS + [(64, 4), (128, 6)], ids=str)
@pytest.mark.parametrize("dtype,n,k", [(ref.BF16, 1100, 160), (ref.F16, 1024, 224), (ref.BF16, 300, 448), (ref.F16, 640, 256), (ref.BF16, 130, 64)])
def test_grouped(fmt, dtype, n, k):
    if not isinstance(fmt, str) and k % fmt[0] != 0:
        pytest.skip("K is not whole groups")
    rng = np.random.default_rng(7200 + n + k)
    experts = [packed(rng, n, k, dtype, fmt) for _ in range(4)]
    stack = lambda f: None if f(experts[0][0]) is None else torch.stack([f(q) for q, _ in experts])
    q = nv.Quantized(stack(lambda q: q.weight), stack(lambda q: q.scales), stack(lambda q: q.biases), experts[0][0].quant)
    ids = np.concatenate([np.zeros(70), np.ones(1), np.full(40, 3)]).astype(np.int32)  # (expert 2 has none)
    x = make_x(rng, ids.size, k, dtype)
    rows, sorted_ids = torch.arange(ids.size, dtype=torch.int32, device="cuda"), torch.from_numpy(ids).cuda()
    got = to_host(nv.gather_qmm_grouped(to_dev(x), q, rows, sorted_ids, nv.sorted_offsets(sorted_ids, 4)))
    for e in (0, 1, 3):
        if isinstance(fmt, str) or n < 1024:
            assert_rows_close(got[ids == e], experts[e][1](x[ids == e]), dtype, f"grouped {fmt} N={n} K={k}", exact_weights=isinstance(fmt, str))
        elif k % 64:
            assert_two_terms(torch.from_numpy(ref.to_f32(got[ids == e], dtype)), torch.from_numpy(ref.to_f32(x[ids == e], dtype)), experts[e][0], dtype, k)


def unrounded(q):
    """scale * code + bias in float64."""
    codes = nv.dequantize(nv.Quantized(q.weight, torch.ones_like(q.scales, dtype=torch.float32), torch.zeros_like(q.scales, dtype=torch.float32), q.quant))
    spread = lambda t: t.double().repeat_interleave(q.quant.group_size, dim=-1)
    return codes.double() * spread(q.scales) + spread(q.biases)


def assert_two_terms(got, x, q, dtype, k):
    """One rounding of the output (u |out|); float32 weights (two terms of them, exact here, may leave u^2 of each where a third does
    not) and float32 sums, whose errors are random over K."""
    u, w = {ref.BF16: 2.0 ** -8, ref.F16: 2.0 ** -11}[dtype], unrounded(q).cpu()
    want, norms = x.double() @ w.T, x.double().norm(dim=1, keepdim=True) * w.norm(dim=1)
    assert ((got.double() - want).abs() <= u * want.abs() + 4 * (u * u / 2 + 2.0 ** -24) * norms).all()


@pytest.mark.parametrize("bits", [1, 2, 3, 4, 5, 6, 8])
@pytest.mark.parametrize("dtype,m,n,k", [(torch.float16, 400, 5000, 160), (torch.float16, 130, 4099, 1056), (torch.bfloat16, 100, 8200, 352), (torch.float16, 300, 1100, 6944)])
def test_rows_on_weights_of_two_terms(bits, dtype, m, n, k):
    torch.manual_seed(bits + m)
    quant = nv.Quant.affine(32, bits)
    assert ops.quantized_matmul_route(m, n, k, quant, dtype) == "qmg_kernel"
    q = nv.quantize((torch.randn(n, k, device="cuda") * 0.02).to(dtype), quant)
    x = torch.randn(m, k, device="cuda").to(dtype)
    assert_two_terms(nv.quantized_matmul(x, q).cpu(), x.cpu(), q, ref.F16 if dtype == torch.float16 else ref.BF16, k)


@pytest.mark.parametrize("bits", [1, 2, 3, 4, 5, 6, 8])
@pytest.mark.parametrize("dtype,m,n,k", [(torch.float16, 400, 5000, 160), (torch.bfloat16, 100, 8200, 352)])
def test_rows_on_weights_of_three_terms(bits, dtype, m, n, k):
    """A bias far below its scale's largest multiple: the weight c s + b has up to 24 bits.  Groups take turns with b and with none, every
    code is the largest, and a row of x is 1 and -1 at one place of either kind: the output is b, exactly, if the weights are."""
    torch.manual_seed(bits)
    quant, ulp = nv.Quant.affine(32, bits), 2.0 ** (-10 if dtype == torch.float16 else -7)
    assert ops.quantized_matmul_route(m, n, k, quant, dtype) == "qmg_kernel"
    s = 1 + ulp
    b = 2.0 ** (int(np.floor(np.log2((2 ** bits - 1) * s))) - 13) * (1 + ulp)
    biases = torch.zeros(n, k // 32, device="cuda", dtype=dtype)
    biases[:, ::2] = b
    q = nv.Quantized(torch.full((n, k * bits // 32), -1, dtype=torch.int32, device="cuda").view(torch.uint32), torch.full_like(biases, s), biases, quant)
    x = torch.zeros(m, k)
    groups = torch.randint(0, k // 64, (m,))
    x[torch.arange(m), 64 * groups + torch.randint(0, 32, (m,))] = 1
    x[torch.arange(m), 64 * groups + 32 + torch.randint(0, 32, (m,))] = -1
    got = nv.quantized_matmul(x.to(dtype).cuda(), q)
    assert torch.equal(got, torch.full_like(got, b)), (got.float() - b).abs().max().item()


@pytest.mark.parametrize("fmt,dtype,m,n,k", [((32, 3), torch.bfloat16, 40, 256, 4128), ((32, 8), torch.float16, 90, 700, 8224), ("MXFP4", torch.bfloat16, 64, 1030, 6176)], ids=str)
def test_without_a_workspace(fmt, dtype, m, n, k):
    """`nvq_quantized_matmul_static` splits K as the call with a workspace does: the same bits."""
    import ctypes as C

    from nuvec_amd import _lib
    torch.manual_seed(k)
    quant = nv.Quant.new(getattr(nv.QuantMode, fmt)) if isinstance(fmt, str) else nv.Quant.affine(*fmt)
    q = nv.quantize((torch.randn(n, k, device="cuda") * 0.02).to(dtype), quant)
    x = torch.randn(m, k, device="cuda").to(dtype)
    want, got = nv.quantized_matmul(x, q), torch.empty(m, n, dtype=dtype, device="cuda")
    d = _lib.QmmDescC()
    d.quant, d.dtype, d.transpose, d.m, d.n, d.k = q.quant._c(), ops._CODE[dtype], 1, m, n, k
    assert _lib.load().nvq_quantized_matmul_workspace_bytes(C.byref(d)) > 0  # (K is split)
    p = ops._ptr
    _lib.check(_lib.load().nvq_quantized_matmul_static(C.byref(d), p(x), p(q.weight), p(q.scales), p(q.biases), p(got), ops._stream()))
    assert torch.equal(got, want)


@pytest.mark.parametrize("k", [160, 224])
def test_an_infinity_among_the_repeated_values(k):
    """x holds one infinity where the last step starts early: every output is that infinity times a weight's sign, none is NaN."""
    rng = np.random.default_rng(7300 + k)
    q, _ = packed(rng, 300, k, ref.BF16, (32, 8))
    x = torch.ones(40, k, dtype=torch.bfloat16, device="cuda")
    at = k - 40 if k % 128 else k - 1
    x[3, at] = float("inf")
    w = nv.dequantize(q)[:, at]
    sign = torch.where(w > 0, float("inf"), float("-inf"))
    ids = torch.zeros(40, dtype=torch.int32, device="cuda")
    grouped = nv.gather_qmm_grouped(x, nv.Quantized(q.weight[None], q.scales[None], q.biases[None], q.quant), torch.arange(40, dtype=torch.int32, device="cuda"),
                                    ids, nv.sorted_offsets(ids, 1))
    for y in (nv.quantized_matmul(x, q), grouped):
        sure = w.abs() > 1e-3  # (a weight near zero may round to either side)
        assert torch.equal(y[3][sure].float(), sign[sure]) and torch.isfinite(y[4]).all()
