"""Biases of the decode kernel (`qmv4_lds_kernel`): requested with the weights where K is one step of it or the codes are affine, read at the
end elsewhere, and none.  Bit for bit the product followed by the addition (crates/nuvec-nn/src/layers.rs:155-162)."""
import pytest
import torch

import nuvec_amd as nv
from nuvec_amd import layers

pytestmark = pytest.mark.gpu

QUANTS = {"MXFP4": nv.Quant.new(nv.QuantMode.MXFP4), "MXFP8": nv.Quant.new(nv.QuantMode.MXFP8), "NVFP4": nv.Quant.new(nv.QuantMode.NVFP4), "4 bits": nv.Quant.affine(32, 4),
          "8 bits": nv.Quant.affine(32, 8), "6 bits": nv.Quant.affine(64, 6), "3 bits": nv.Quant.affine(64, 3)}


# K: a step of 4096 values and the ones beside it, and a part of a third; rows that end inside a block
@pytest.mark.parametrize("quant", list(QUANTS))
@pytest.mark.parametrize("k", [2240, 4032, 4096, 4160, 8384])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_linear(quant, k, dtype):
    torch.manual_seed(k)
    n, quant = 1029, QUANTS[quant]
    q = nv.quantize((torch.randn(n, k, device="cuda") * 0.05).to(dtype), quant)
    bias = torch.randn(n, device="cuda").to(dtype)
    for m in (1, 2, 3, 4):
        x = torch.randn(m, k, device="cuda").to(dtype)
        if nv.ops.quantized_matmul_kernel(m, n, k, quant, dtype) == "qmv4_lds_kernel":
            assert torch.equal(layers.QuantizedLinear(q.weight, q.scales, q.biases, bias, quant)(x), nv.quantized_matmul(x, q) + bias), m
        elif m == 1 and quant.bits != 4:
            pytest.fail("the decode kernel does not run a row that this is about")


@pytest.mark.parametrize("quant", ["MXFP4", "MXFP8", "NVFP4", "4 bits"])
@pytest.mark.parametrize("k", [4096, 4160, 8384])
def test_gated_pairs(quant, k):
    torch.manual_seed(k)
    experts, hidden, quant = 3, 1088, QUANTS[quant]
    gate, up = (nv.quantize((torch.randn(experts, hidden, k, device="cuda") * k ** -0.5).bfloat16(), quant) for _ in range(2))
    gb, ub = (torch.randn(experts, hidden, device="cuda").bfloat16() for _ in range(2))
    pair = lambda a, b: None if a is None else nv.pair_rows(a, b, 1)
    both = nv.Quantized(pair(gate.weight, up.weight), pair(gate.scales, up.scales), pair(gate.biases, up.biases), quant)
    x, ids = torch.randn(4, k, device="cuda").bfloat16(), torch.tensor([2, 0, 2, 1], dtype=torch.int32, device="cuda")
    rows = torch.arange(4, dtype=torch.int32, device="cuda")
    g, u = (nv.gather_qmm(x.unsqueeze(1), q, None, ids).squeeze(1) for q in (gate, up))
    for biased in (False, True):
        want = nv.glu(g, u, "swiglu_oai", **(dict(gate_bias=gb, up_bias=ub, ids=ids) if biased else {}))
        got = nv.gather_qmm_glu(x, both, rows, ids, None, "swiglu_oai", expert_bias=pair(gb, ub) if biased else None)
        assert torch.equal(got, want), biased
