"""The down products of a token's experts and their weighted sum in one kernel (`nvq_gather_qmm_sum`; MoeMlp::forward,
crates/nuvec-lm/src/model.rs:2248-2271): bit for bit `nvq_gather_qmm_expert_bias` and `nvq_weighted_sum`."""
import ctypes as C

import pytest
import torch

import nuvec_amd as nv
from nuvec_amd import _lib, ops

pytestmark = pytest.mark.gpu

p = lambda t: None if t is None else C.c_void_p(t.data_ptr())


def call(q, x, lhs, rhs, bias, scores, out, pairs, rows):
    n, k = q.weight.shape[1], x.shape[1]
    d = _lib.GatherDescC(q.quant._c(), ops._CODE[x.dtype], 1, 0, 0, 1, n, k, pairs, rows, q.weight.shape[0])
    return _lib.load().nvq_gather_qmm_sum(C.byref(d), p(x), p(q.weight), p(q.scales), p(q.biases), p(q.global_scale), p(lhs), p(rhs), p(bias),
                                          p(scores), scores.shape[1], p(out), ops._stream())


# n: rows that end inside a wavefront's, a block's; k: part of a step, of its second half, a second step
@pytest.mark.parametrize("quant,n,k", [("MXFP4", 2, 2080), ("MXFP4", 1025, 4128), ("MXFP8", 130, 2912), ("NVFP4", 67, 4096), ((64, 4), 1027, 2880), ((32, 8), 1030, 352),
                                       ((32, 2), 1026, 2144), ((32, 3), 1024, 4384), ((64, 5), 1035, 1088), ((128, 6), 1041, 640)], ids=str)
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_equals_the_products_and_their_sum(quant, n, k, dtype):
    torch.manual_seed(n + k)
    put = lambda *shape: torch.randn(shape, device="cuda").to(dtype)
    kind = nv.Quant.affine(*quant) if isinstance(quant, tuple) else nv.Quant.new(getattr(nv.QuantMode, quant))
    q = nv.quantize(put(5, n, k) * 0.1, kind)
    if quant == "NVFP4":
        q = nv.Quantized(q.weight, q.scales, None, q.quant, torch.rand(5, device="cuda") * 3 + 0.5)
    for tokens, choices in ((1, 1), (3, 1), (1, 2), (2, 3), (1, 4), (2, 4)):
        pairs = tokens * choices
        rhs = torch.randint(0, 5, (pairs,), device="cuda", dtype=torch.int32)
        for rows, lhs in ((pairs, torch.arange(pairs, device="cuda", dtype=torch.int32)), (2, torch.randint(0, 2, (pairs,), device="cuda", dtype=torch.int32))):
            for bias in (None, put(5, n)):
                x, scores, out = put(rows, k), torch.rand(tokens, choices, device="cuda").to(dtype), torch.full((tokens, n), 7.0, device="cuda", dtype=dtype)
                _lib.check(call(q, x, lhs, rhs, bias, scores, out, pairs, rows))
                d = _lib.GatherDescC(q.quant._c(), ops._CODE[dtype], 1, 0, 0, 1, n, k, pairs, rows, 5)
                y = torch.empty(tokens, choices, n, device="cuda", dtype=dtype)
                _lib.check(_lib.load().nvq_gather_qmm_expert_bias(C.byref(d), p(x), p(q.weight), p(q.scales), p(q.biases), p(q.global_scale), p(lhs), p(rhs),
                                                                  None, None, p(bias), p(y), None, ops._stream()))
                assert torch.equal(out, ops.weighted_sum(y, scores)), (tokens, choices, rows)


def test_what_the_two_kernels_keep():
    """More than four pairs a token, rows of the CPU's weights, short rows, float32, one output."""
    torch.manual_seed(1)
    for quant, n, k, choices, dtype in (((64, 4), 1024, 2880, 5, torch.bfloat16), ((64, 4), 512, 2880, 2, torch.bfloat16), ((64, 4), 1024, 1024, 2, torch.bfloat16),
                                        ((64, 4), 1024, 2880, 2, torch.float32), ((64, 4), 1, 2880, 2, torch.bfloat16)):
        q = nv.quantize(torch.randn(5, n, k, device="cuda").to(dtype), nv.Quant.affine(*quant))
        ids = torch.arange(choices, device="cuda", dtype=torch.int32)
        x, scores, out = torch.randn(choices, k, device="cuda").to(dtype), torch.rand(1, choices, device="cuda").to(dtype), torch.empty(1, n, device="cuda", dtype=dtype)
        assert call(q, x, ids, ids, None, scores, out, choices, choices) == _lib.UNSUPPORTED


def test_questions_about_nothing():
    """Descriptors that no launch would take."""
    ask = lambda **odd: [f(C.byref(_lib.GatherDescC(**{**dict(quant=nv.Quant.affine(64, 4)._c(), dtype=ops._CODE[torch.bfloat16], transpose=1, m=1, n=1024, k=2880, pairs=4,
                                                              x_batches=4, experts=8), **odd}))) for f in (_lib.load().nvq_gather_sorted_takes, lambda d: _lib.load().nvq_gather_qmm_sum_takes(d, 4))]
    nv.quantize(torch.zeros(1, 64, device="cuda"), nv.Quant.affine(64, 4))  # (the library has a device)
    assert ask() == [1, 1]
    for odd in (dict(pairs=0), dict(pairs=-4), dict(experts=0), dict(experts=-1), dict(x_batches=0), dict(n=0), dict(k=0), dict(k=2881), dict(transpose=0), dict(dtype=-1)):
        assert ask(**odd) == [0, 0], odd
    assert _lib.load().nvq_gather_sorted_takes(None) == 0 and _lib.load().nvq_gather_qmm_sum_takes(None, 1) == 0


def test_the_question_answers_as_the_call():
    """`nvq_gather_qmm_sum_takes`, by which a block asks before it launches."""
    torch.manual_seed(2)
    for quant, n, k, tokens, choices, dtype in (("MXFP4", 2880, 2880, 1, 4, torch.bfloat16), ("MXFP4", 2880, 2880, 1, 5, torch.bfloat16), ("NVFP4", 1024, 1024, 2, 2, torch.float16),
                                                ((64, 4), 1024, 2880, 3, 4, torch.bfloat16), ((64, 4), 1024, 2048, 1, 2, torch.bfloat16), ((64, 4), 512, 2880, 1, 2, torch.bfloat16),
                                                ((32, 8), 1030, 352, 1, 1, torch.float16), ((64, 6), 8192, 4096, 8, 4, torch.bfloat16), ((64, 4), 1024, 2880, 1, 2, torch.float32)):
        kind = nv.Quant.affine(*quant) if isinstance(quant, tuple) else nv.Quant.new(getattr(nv.QuantMode, quant))
        q, pairs = nv.quantize(torch.randn(5, n, k, device="cuda").to(dtype), kind), tokens * choices
        ids = torch.arange(pairs, device="cuda", dtype=torch.int32)
        x, scores, out = torch.randn(pairs, k, device="cuda").to(dtype), torch.rand(tokens, choices, device="cuda").to(dtype), torch.empty(tokens, n, device="cuda", dtype=dtype)
        d = _lib.GatherDescC(q.quant._c(), ops._CODE[dtype], 1, 0, 0, 1, n, k, pairs, pairs, 5)
        rc = call(q, x, ids, ids % 5, None, scores, out, pairs, pairs)
        assert rc in (0, _lib.UNSUPPORTED) and _lib.load().nvq_gather_qmm_sum_takes(C.byref(d), choices) == (rc == 0), (quant, n, k, choices)
