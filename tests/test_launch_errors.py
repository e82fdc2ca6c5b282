"""A launch that fails is an error of the call that made it."""
import pytest
import torch
from ctypes import c_float, c_int, c_void_p

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


def test_more_rows_than_a_launch_holds_are_refused():
    """Before anything is launched: rounding the rows up to whole tiles must not pass the largest number."""
    lib = kernels.library()
    at, zero = c_void_p(1 << 20), c_float(0.0)
    for rows in (2147483393, 2147483647):
        assert lib.ta_gemm_glu(None, at, c_int(64), at, c_int(64), None, at, c_int(8192), c_int(rows), c_int(8192), c_int(64), c_int(0), zero, zero, zero) != 0
        assert lib.ta_last_error().startswith(b"ta_gemm_glu: M=%d" % rows), lib.ta_last_error()
        assert lib.ta_gemm_plain(None, at, c_int(64), at, c_int(64), at, c_int(256), c_int(rows), c_int(256), c_int(64), c_int(0)) != 0
        assert lib.ta_last_error().startswith(b"ta_gemm_plain: M=%d" % rows), lib.ta_last_error()
        assert not lib.ta_gemm_split_glu_takes(c_int(rows), c_int(8192), c_int(2048), c_int(2048), c_int(2048))
        assert lib.ta_gemm_split_glu(None, at, c_int(2048), at, c_int(2048), None, at, c_int(8192), c_int(rows), c_int(8192), c_int(2048)) != 0
        assert lib.ta_last_error().startswith(b"ta_gemm_split_glu: M=%d" % rows), lib.ta_last_error()
