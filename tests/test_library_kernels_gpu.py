"""Which of the library's kernels the large products run."""
import ctypes

import pytest
import torch

from mini_engine_amd.kernels import ops
from test_kernels_gpu import DEV, close, hip

pytestmark = pytest.mark.gpu


def _kernel(M, N, K, dtype):
    name = ctypes.create_string_buffer(512)
    rc = ops.core().cdll.me_gemm_library_kernel(ops._code(dtype), ctypes.c_size_t(ops.LIBRARY_WORKSPACE_BYTES), M, N, K, 1, name, 512)
    assert rc == 0
    return name.value.decode()


@pytest.mark.parametrize("M,N,K", [(8005, 4096, 1024), (8005, 6144, 1024), (3123, 4096, 1024), (4096, 4096, 4096), (2048, 24576, 4096)])
def test_the_kernel_that_is_wrong_now_and_then_is_not_taken(M, N, K):
    """The hand-scheduled kernel of 256 x 256 tiles is the heuristic's first choice for these shapes. What runs in its place adds
    up K in one piece: one rounding to bfloat16 (2^-9 at most, 2e-3 of the norm) on float32 sums of up to 4,096 terms."""
    g = torch.Generator(device=DEV).manual_seed(M)
    x, w = torch.randn(M, K, device=DEV, generator=g).to(torch.bfloat16), torch.randn(N, K, device=DEV, generator=g).to(torch.bfloat16)
    y = hip().linear(x, w)
    name = _kernel(M, N, K, torch.bfloat16)
    assert name and "Custom" not in name
    rows = torch.arange(0, M, 97, device=DEV)
    close(y[rows], x[rows].double() @ w.double().t(), 4e-3)
