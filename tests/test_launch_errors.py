"""A launch that fails is an error of the call that made it."""
import pytest
import torch
from ctypes import c_int, c_void_p

from transformer_amd import kernels


# of every kernel behind the call: few rows through LDS and straight from memory, along the columns, tiles, groups
@pytest.mark.parametrize("M,N,K,streams", [(4, 2048, 2048, True), (8, 1024, 8192, True), (1, 64, 1540, True), (4, 2048, 512, False),
                                           (4, 16384, 1024, False), (12, 16384, 2048, False), (2000, 2048, 64, False), (1021, 3072, 2048, False)])
def test_a_float32_product_without_a_device_fails(M, N, K, streams):
    if torch.cuda.is_available():
        pytest.skip("the operands are addresses of nothing: only where no kernel can be launched")
    lib = kernels.library()
    at = c_void_p(1 << 20)
    f32 = c_int(kernels.F32)
    rc = lib.ta_gemm_simple(None, f32, f32, f32, at, c_int(K), at, c_int(K), None, at, c_int(N), c_int(M), c_int(N), c_int(K))
    assert rc != 0
    # a product handed on returns what the one that took it returns: its check takes the error, a second one finds none
    assert lib.ta_last_error().startswith(b"ta_gemm_stream" if streams else b"ta_gemm_simple"), lib.ta_last_error()
