"""Which prompts' products go to the kernels for many bfloat16 rows, and which steps to the one for a token side input: not those at which the vendor
library, or the kernels one by one, were measured to be faster."""
import pytest

from ctypes import c_int

from transformer_amd import kernels


def _glu(m, n, k):
    return bool(kernels.library().ta_gemm_glu_pays(c_int(m), c_int(n), c_int(k)))


def _plain(m, n, k):
    return bool(kernels.library().ta_gemm_plain_pays(c_int(m), c_int(n), c_int(k)))


@pytest.mark.parametrize("m,n,k,takes", [
    (384, 14336, 4096, False), (385, 14336, 4096, True), (512, 14336, 4096, True), (513, 14336, 4096, False), (640, 14336, 4096, False), (641, 14336, 4096, True),
    (641, 8192, 4096, False), (768, 8192, 8192, False), (769, 8192, 4096, True), (700, 11008, 4096, True), (512, 8192, 4096, True),       # 192 tiles in three rows
    (1025, 8192, 2048, False), (1280, 8192, 2048, False), (1281, 8192, 2048, True), (1100, 8192, 4096, True), (1024, 8192, 2048, True),    # a quarter of a second round
    (1025, 14336, 2048, True), (8192, 16384, 2048, False), (8192, 16384, 4096, True), (1536, 16384, 2048, True), (7900, 16384, 2048, True),  # whole rounds only
    (2048, 16384, 2048, False), (2011, 14336, 4096, True), (5000, 7996, 4096, False), (5000, 8002, 4096, False), (5000, 8192, 1984, False), (5000, 8192, 4100, False)])
def test_gated(m, n, k, takes):
    assert _glu(m, n, k) == takes


@pytest.mark.parametrize("m,n,k,takes", [
    (1536, 4096, 12352, False), (3072, 2048, 8192, False), (2048, 3072, 12288, False), (2176, 3072, 12288, True), (1280, 5120, 13824, True),     # 96 tiles alone, 108, 100
    (5504, 4096, 14336, True), (2656, 8192, 14336, True), (2656, 8192, 28672, False), (5504, 4096, 28672, True),                                 # 352
    (2011, 4096, 14336, False), (2011, 4096, 12288, True), (1792, 4096, 28672, True), (3164, 4096, 4096, True), (8192, 4096, 4096, False),       # 128, 112, 208, two rounds
    (816, 16384, 4096, False), (816, 16384, 16384, True), (8193, 4096, 14336, False), (4096, 4096, 8192, True), (3000, 4096, 14336, False), (3072, 2000, 8192, False)])
def test_plain(m, n, k, takes):
    assert _plain(m, n, k) == takes


@pytest.mark.parametrize("tokens,d,dim,plain,routed", [
    (1, 4096, 32, True, True), (64, 512, 32, True, True), (65, 512, 32, False, False), (0, 512, 32, False, False), (4, 2048, 64, True, True), (4, 2560, 64, False, True),
    (4, 4096, 64, False, False), (17, 4096, 64, True, True), (1, 1024, 128, False, True), (16, 2048, 128, False, False), (32, 2048, 128, True, True),
    (32, 2560, 128, False, False), (64, 4096, 128, False, False), (4, 2048, 48, False, False), (4, 2000, 64, False, False), (4, 4608, 32, False, False)])
def test_side_steps(tokens, d, dim, plain, routed):
    pays = [bool(kernels.library().ta_side_step_pays(c_int(tokens), c_int(d), c_int(dim), c_int(r))) for r in (0, 1)]
    assert pays == [plain, routed]
