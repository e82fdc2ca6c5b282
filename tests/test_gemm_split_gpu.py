"""float32 products in three bfloat16 an operand: every form that many rows go to, at the edges of its tiles, segments and groups,
has the bits of rows by themselves; how far the sums are from 64 bits; operands and sums that are not finite."""
import pytest
import torch

from transformer_amd import kernels

pytestmark = pytest.mark.gpu

# rows, columns, k: 256 x 128; 128 x 96 and 128 x 64 by two groups; 64 x 64 by four; 128 x 64 and 64 x 64 by one (short k). k of whole
# segments, of whole blocks, ending inside a block, inside the segment of a later group, an odd number of blocks
SHAPES = [(1021, 4100, 512), (513, 16387, 264), (1000, 3070, 1024), (257, 9000, 1292), (1021, 2044, 2048), (900, 2050, 1796), (130, 4100, 2000),
          (129, 3000, 1056), (40, 16000, 1540), (300, 2047, 772), (65, 16400, 516), (1100, 5570, 68), (3, 12300, 128), (70, 12290, 36), (17, 33000, 2048)]


def _draw(m, n, k):
    g = torch.Generator(device="cuda").manual_seed(m + 7 * n + 31 * k)
    return torch.randn(m, k, generator=g, device="cuda"), torch.randn(n, k, generator=g, device="cuda")


def _alone(a, w):
    return torch.cat([kernels.gemm_simple(a[i:i + 1].contiguous(), w, torch.empty(1, w.shape[0], device="cuda")) for i in range(a.shape[0])])


@pytest.mark.parametrize("m,n,k", SHAPES)
def test_many_rows_have_the_bits_of_each_alone(m, n, k):
    a, w = _draw(m, n, k)
    out = torch.full((m + 1, n + 3), 7.0, device="cuda")
    kernels.gemm_simple(a, w, out[:m, 1:n + 1])
    assert bool((out[:, 0] == 7).all()) and bool((out[:, n + 1:] == 7).all()) and bool((out[m] == 7).all())
    rows = sorted({0, min(15, m - 1), min(16, m - 1), m // 2, max(0, m - 17), m - 1})
    assert torch.equal(out[rows, 1:n + 1], _alone(a[rows], w))
    exact = a[rows].double() @ w.double().t()
    # a block's chain of six instructions loses at most 2^-23 of what it reaches each, a sum of blocks or segments half that, what is
    # left out 2^-24 of every product
    blocks = -(-k // 32)
    bound = (6 + min(blocks, 8) / 2 + blocks / 16 + 1) * 2.0 ** -23 * (a[rows].double().abs() @ w.double().abs().t())
    off = (out[rows, 1:n + 1].double() - exact).abs()
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
