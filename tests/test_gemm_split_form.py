"""Which kernel a float32 product of many rows goes to."""
import pytest

from ctypes import c_int

from transformer_amd import kernels

FAR = 7                      # the first of the forms for rows far apart


def form(m, n, k, lda=None, ldw=None, batch=1, vec=None):
    """0: few rows; 1: 256 x 128; 2, 3: 128 x 96 and 128 x 64 by two groups; 4: 64 x 64 by four; 5, 6: 128 x 64 and 64 x 64 by one;
    7, 8: the fourth and the fifth, rows any distance apart."""
    vec = k % 4 == 0 if vec is None else vec
    return kernels.library().ta_gemm_split_form(*map(c_int, (m, n, k, lda or k, ldw or k, batch, int(vec))))


# the fastest of the forms, timed one by one (us of few rows, then forms 1 to 5)
@pytest.mark.parametrize("m,n,k,want", [
    (24, 6144, 256, 0),             # 6.9; 21.2 20.9 15.5 18.3 12.1
    (17, 16384, 512, 0),            # 12.4; 37.3 21.6 16.3 19.3 19.8
    (48, 6144, 256, 0),             # 9.4; 21.3 21.2 15.9 19.8 12.0
    (700, 4096, 1024, 5),           # 103; 69.6 74.4 56.7 65.2 50.9
    (257, 8192, 1024, 5),           # 86; 70.7 71.1 55.3 63.8 51.0
    (64, 6144, 8192, 4)])           # 147; 491 241 172 129 248
def test_the_costs_choose_the_fastest(m, n, k, want):
    assert form(m, n, k) == want


@pytest.mark.parametrize("m,n,k", [(1021, 16384, 2048), (1021, 2044, 2048), (300, 9000, 1292), (300, 9001, 1291), (300, 2048, 2048), (1100, 5570, 68)])
def test_rows_far_apart_go_by_tiles_too(m, n, k):
    assert 0 < form(m, n, k) < FAR
    for lda, ldw in ((4194304, None), (None, 4194304), (2147483644, 2147483644)):
        assert form(m, n, k, lda, ldw) >= FAR
    assert form(m, n, k, 4194300, 4194300) == form(m, n, k)
    if k > 128:
        assert form(12, n, k, 4194304) == form(12, n, k) == 0
