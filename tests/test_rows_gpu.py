"""Row kernels on the GPU at widths their other tests leave out: the register
form of the ConvRot quantizer on K that is no multiple of 512, and the row
packers behind operands that are not read in place."""
import numpy as np
import pytest
import torch

from conftest import case
from oracle import convrot as cr
from oracle import int8 as oi
from test_convrot_gpu import _rows

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("g,shape", [(256, (37, 768)), (256, (5, 3328)), (512, (3, 4608)), (8, (9, 1000)),
                                     (16, (4, 48)), (32, (3, 8160)), (64, (6, 16320)), (128, (2, 640))])
def test_rot_quant_rows_ragged_widths(cuda, dtype, g, shape):
    from rdna2_ops.quantize import rotate_quantize_int8_rowwise
    case(f"rot quant ragged {dtype} g{g} {shape}")
    x = _rows(shape, g * 31 + shape[1]).to(dtype)
    q, step = rotate_quantize_int8_rowwise(x.to(cuda), g)
    qo, so = cr.rot_quant_rows(x.float().numpy(), g)
    assert np.array_equal(step.cpu().numpy().reshape(-1), so)
    assert np.array_equal(q.cpu().numpy(), qo)


@pytest.mark.parametrize("k", [1, 7, 15, 16, 17, 100, 127, 129, 1000, 3256])
@pytest.mark.parametrize("offset", [0, 1, 8])
def test_packed_rows(cuda, k, offset):
    """int8 operands whose rows are not 16-byte aligned or whose K is ragged
    are packed: unit K stride at any alignment, and K strided (a [K, N]
    row-major right operand)."""
    from rdna2_ops.int8_gemm import int8_matmul
    case(f"packed rows k{k} offset{offset}")
    g = torch.Generator().manual_seed(k + offset)
    m, n = 40, 70
    a = torch.randint(-128, 128, (m, k + offset + 3), generator=g, dtype=torch.int8)[:, offset:offset + k]
    w = torch.randint(-128, 128, (n, k + offset + 5), generator=g, dtype=torch.int8)[:, offset:offset + k]
    ref = oi.int8_matmul(a.numpy(), np.ascontiguousarray(w.numpy().T))
    store_a = torch.empty(m, k + offset + 3, dtype=torch.int8, device=cuda)[:, offset:offset + k]
    store_w = torch.empty(n, k + offset + 5, dtype=torch.int8, device=cuda)[:, offset:offset + k]
    store_a.copy_(a.to(cuda))
    store_w.copy_(w.to(cuda))
    assert np.array_equal(int8_matmul(store_a, store_w.T).cpu().numpy(), ref)
    assert np.array_equal(int8_matmul(store_a, store_w.T.contiguous()).cpu().numpy(), ref)


@pytest.mark.parametrize("k", [1000, 1027, 130])
@pytest.mark.parametrize("offset", [0, 1, 4])
def test_packed_half_rows(cuda, k, offset):
    """fp16 activations and fp8 weights with ragged K or unaligned rows."""
    from rdna2_ops.fp8_weight_gemm_v06 import fp8_weight_gemm
    case(f"packed half rows k{k} offset{offset}")
    g = torch.Generator().manual_seed(k + offset)
    a = torch.randn(40, k + 9, generator=g).half().to(cuda)[:, offset:offset + k]
    w = torch.randn(30, k + 9, generator=g).to(torch.float8_e4m3fn).to(cuda)[:, offset:offset + k]
    y = fp8_weight_gemm(a, w, method="fused_dot2").double()
    ref = a.double() @ w.double().T
    assert (y - ref).abs().max().item() <= 2.0 ** -11 * ref.abs().max().item() + 1e-4
