"""x on its way into LDS in the wave-per-row kernels: what a thread fetches ahead of the weights, and the rest of longer rows in batches."""
import pytest
import torch

from tests.test_gpu_decode_step import test_linear as check_linear
from tests.test_gpu_fp32_rows import _close, _data

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("B,K,dtype", [
    (1, 4104, torch.float16), (1, 12296, torch.bfloat16), (1, 65536, torch.float16), (2, 4096, torch.float16), (2, 8200, torch.bfloat16), (2, 32768, torch.float16),
    (1, 2052, torch.float32), (2, 4100, torch.float32), (3, 2052, torch.float32), (4, 8192, torch.float32), (7, 1000, torch.float32), (8, 4096, torch.float32),
    (5, 8184, torch.float16)])
@pytest.mark.parametrize("norm", [False, True])
def test_projections(B, K, dtype, norm):
    """One vector more than is fetched ahead, one batch and several, all the LDS that a call may take, batch rows that the kernel's rows exceed."""
    check_linear(B, K, 21, dtype, norm)


@pytest.mark.parametrize("H,I,B", [(512, 4096, 1), (512, 4100, 1), (264, 12288, 1), (264, 12292, 1), (100, 2052, 2), (516, 6148, 2), (8200, 400, 1), (4100, 404, 2),
                                   (512, 2048, 3), (520, 8196, 4), (6148, 300, 4)])
def test_hf_layout_calls(H, I, B):
    """The dense down product over intermediate rows up to and beyond four and twelve vectors a thread, and long rows of x."""
    import flash_gemv

    x, wg, wu, wd, t, a, z = _data(H, I, B)
    _close(flash_gemv.flag_gemv_gemv_inner_fp32(x, wg, wu, wd.t().contiguous(), t), z @ wd.double())
