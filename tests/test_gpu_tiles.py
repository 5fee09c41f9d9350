"""The tiles of the products that expand codes themselves (csrc/qmm_kernel.h, csrc/qmk_kernel.h): which of them a product runs on."""
import pytest
import torch

import nuvec_amd as nv
from nuvec_amd import ops

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
