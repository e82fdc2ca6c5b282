"""The row counts in which the vendor library is given a product: no GPU is needed."""
import pytest

from transformer_amd.parts.linear import library_rows


@pytest.mark.parametrize("n,k", [(65792, 16384), (131072, 14336), (256, 16384), (5120, 13824), (6144, 14336), (4096, 28672),
                                 (12288, 14336), (4096, 8192), (4096, 10176)])
def test_widths_that_were_not_measured_stay_whole(n, k):
    for rows in (1, 257, 4097, 20000, 100003):
        assert library_rows(rows, n, k) == [rows]


@pytest.mark.parametrize("n,k", [(4096, 10240), (4096, 14336), (8192, 28672), (16384, 14336)])
def test_calls_hold_every_row_once(n, k):
    full = 65536 * 256 // n
    for rows in (1, full, full + 1, full + full // 8, 2 * full, 2 * full + 1, 5 * full - 3, 70001):
        calls = library_rows(rows, n, k)
        assert sum(calls) == rows and min(calls) > 0 and max(calls) <= 2 * full
        assert len(calls) == 1 or rows > full
