"""float32 products in three bfloat16 an operand: every form that many rows go to, at the edges of its tiles, segments and groups,
has the bits of rows by themselves; how far the sums are from 64 bits; operands and sums that are not finite."""
import pytest
import torch

from test_gemm_split_form import form
from transformer_amd import kernels

pytestmark = pytest.mark.gpu

# form: rows, columns, k. 1: 256 x 128; 2, 3: 128 x 96 and 128 x 64 by two groups; 4: 64 x 64 by four; 5: 128 x 64, 6: 64 x 64 by one (short k); 0: few rows. Of each form k of whole segments (which is code of its own), of whole blocks, ending inside a block, inside the segment of a later
# group, an odd number of blocks, and where a form takes them numbers of k that are no multiple of 4
SHAPES = [(1, 1021, 4100, 512), (1, 1021, 16384, 512), (1, 1021, 8192, 2048), (1, 513, 16387, 264), (2, 1000, 3070, 1024), (2, 1021, 3000, 2048), (2, 900, 2050, 1796),
          (3, 1021, 2044, 2048), (3, 200, 5000, 1536), (3, 1021, 2044, 2044), (3, 500, 4090, 1300), (4, 130, 4100, 2048), (4, 130, 4100, 2000), (4, 40, 16000, 1540),
          (4, 129, 3000, 1056), (5, 700, 5000, 1024), (5, 257, 9000, 1292), (5, 300, 9001, 1291), (5, 1100, 5570, 68), (5, 1100, 5570, 67), (5, 70, 12290, 36),
          (2, 65, 16400, 516), (6, 300, 12290, 128), (6, 300, 12290, 127), (4, 300, 2047, 772), (0, 3, 12300, 128), (0, 17, 33000, 2048)]


def _draw(m, n, k):
    g = torch.Generator(device="cuda").manual_seed(m + 7 * n + 31 * k)
    return torch.randn(m, k, generator=g, device="cuda"), torch.randn(n, k, generator=g, device="cuda")


def _alone(a, w):
    return torch.cat([kernels.gemm_simple(a[i:i + 1].contiguous(), w, torch.empty(1, w.shape[0], device="cuda")) for i in range(a.shape[0])])


@pytest.mark.parametrize("chosen,m,n,k", SHAPES)
def test_many_rows_have_the_bits_of_each_alone(chosen, m, n, k):
    assert form(m, n, k) == chosen             # what this shape is here for
    a, w = _draw(m, n, k)
    rows = sorted({0, min(15, m - 1), min(16, m - 1), m // 2, max(0, m - 17), m - 1})
    alone = _alone(a[rows], w)
    for shift, width in ((1, n + 3), (0, n), (4, (n + 11) // 4 * 4)):      # results stored one by one, and 16 bytes at a time where that fits
        out = torch.full((m + 1, width), 7.0, device="cuda")
        got = kernels.gemm_simple(a, w, out[:m, shift:shift + n])
        assert bool((out[:, :shift] == 7).all()) and bool((out[:, shift + n:] == 7).all()) and bool((out[m] == 7).all())
        assert torch.equal(got[rows], alone)
    exact = a[rows].double() @ w.double().t()
    # a block's chain of six instructions loses at most 2^-23 of what it reaches each, a sum of blocks or segments half that, what is
    # left out 2.9e-7 of every product
    blocks = -(-k // 32)
    bound = ((6 + min(blocks, 8) / 2 + blocks / 16) * 2.0 ** -23 + 2.9e-7) * (a[rows].double().abs() @ w.double().abs().t())
    off = (alone.double() - exact).abs()
    assert bool((off <= bound).all())
    # chains of fused multiply-adds over segments of 256 are 2.9e-7 away in the mean over normal entries
    assert float(off.norm() / exact.norm()) < 2e-7


@pytest.mark.parametrize("m,n,k", [(1021, 2044, 2048), (130, 4100, 2000), (70, 4000, 2048), (33, 300, 1000), (12, 5200, 2048), (12, 5200, 4096), (8, 4100, 2048), (3, 500, 8192)])
def test_what_is_not_finite(m, n, k):
    """Infinities, undefined numbers, numbers beyond bfloat16's largest and sums that overflow: what 64 bits give in 32."""
    a, w = _draw(m, n, k)
    w *= 0.01
    w[:, 100] *= 1e-3
    a[0, 7], a[1, 9], a[2, 100] = float("inf"), float("nan"), 3.4e38
    w[11, 7] = 0.0                               # infinity times zero
    w[17, 55] = -float("inf")
    w[19, 3] = 3e38                              # overflows where the row's number is above 1.13 (one product: two could cancel in 64 bits)
    exact = (a.double() @ w.double().t()).float()
    got = kernels.gemm_simple(a, w, torch.empty(m, n, device="cuda"))
    assert torch.equal(got.isnan(), exact.isnan()) and torch.equal(got.isinf(), exact.isinf())
    inf = exact.isinf()
    assert torch.equal(got[inf], exact[inf])
    ok = exact.isfinite()
    scale = torch.where(ok, a.double().abs() @ w.double().abs().t(), torch.zeros((), dtype=torch.float64, device="cuda"))
    assert bool(((got.double() - exact.double()).abs()[ok] <= 1e-5 * scale[ok]).all())
