"""Row kernels on the GPU at widths their other tests leave out: the register
form of the ConvRot quantizer on K that is no multiple of 512."""
import numpy as np
import pytest
import torch

from conftest import case
from oracle import convrot as cr
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
