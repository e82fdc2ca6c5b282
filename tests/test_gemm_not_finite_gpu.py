"""float32 products whose sums are not finite: what they cost, how exact they are where 32 bits hold them after all, and that a row's bits do
not depend on its neighbours."""
import pytest
import torch

from transformer_amd import kernels

pytestmark = pytest.mark.gpu

# tiles of 256 x 128, groups, 64 x 64, few rows, along the columns, whole lines through LDS at both lengths of k
SHAPES = [(1021, 16384, 512), (1021, 2044, 2048), (130, 4100, 2000), (70, 4000, 2048), (33, 300, 1000), (12, 5200, 2048), (12, 5200, 4096), (8, 4100, 2048), (3, 500, 8192)]


def _draw(m, n, k):
    g = torch.Generator(device="cuda").manual_seed(m + 7 * n + 31 * k)
    return torch.randn(m, k, generator=g, device="cuda"), torch.randn(n, k, generator=g, device="cuda")


def _run(a, w, bias=None):
    return kernels.gemm_simple(a, w, torch.empty(a.shape[0], w.shape[0], device="cuda"), bias)


def _us(f):
    best = 1e9
    for _ in range(5):
        a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
        a.record()
        for _ in range(4):
            f()
        b.record()
        torch.cuda.synchronize()
        best = min(best, a.elapsed_time(b) * 250)
    return best


@pytest.mark.parametrize("m,n,k", SHAPES)
def test_an_undefined_row_costs_its_neighbours_little(m, n, k):
    a, w = _draw(m, n, k)
    out = torch.empty(m, n, device="cuda")
    usual = _us(lambda: kernels.gemm_simple(a, w, out))
    want = out.clone()
    a[m // 2, k // 3] = float("nan")
    spoilt = _us(lambda: kernels.gemm_simple(a, w, out))
    want[m // 2] = float("nan")
    assert torch.equal(out.isnan(), want.isnan()) and torch.equal(out.nan_to_num(), want.nan_to_num())
    # one wave looks through a row once: some 10 us, where walks along k in series take milliseconds
    assert spoilt < 1.5 * usual + 25


@pytest.mark.parametrize("m,n,k", SHAPES)
def test_sums_past_the_split_keep_their_bits(m, n, k):
    """Numbers that round past bfloat16's largest: every sum is formed again, as exact as chains over segments are (3.3e-7 over normal entries)."""
    a, w = _draw(m, n, k)
    a[:, 5] = 3.4e38 * a[:, 5].sign()
    w[:, 5] *= 1e-38
    got, exact = _run(a, w), a.double() @ w.double().t()
    assert float((got.double() - exact).norm() / exact.norm()) < 3.3e-7
    rows = sorted({0, m // 2, m - 1})
    assert torch.equal(torch.cat([_run(a[i:i + 1].contiguous(), w) for i in rows]), got[rows])


@pytest.mark.parametrize("m,n,k", SHAPES)
def test_a_bias_that_overflows(m, n, k):
    """Sums that only their bias takes past 32 bits, beside sums that are not finite by themselves."""
    a, w = _draw(m, n, k)
    bias = torch.zeros(n, device="cuda")
    bias[::2] = 3.4028234e38
    a *= 2e31 / k ** .5                          # half an ulp of the bias is 1e31
    a[:, 1], a[:, k - 2], w[:, 1], w[:, k - 2] = 1e37, -1e37, 1.0, 1.0     # what another order of the sums would differ by is 1e30
    w[3::8, 3] = float("inf")
    got = _run(a, w, bias)
    rows = sorted({0, min(17, m - 1), m // 2, m - 1})
    alone = torch.cat([_run(a[i:i + 1].contiguous(), w, bias) for i in rows])
    assert torch.equal(got[rows].isnan(), alone.isnan()) and torch.equal(got[rows].nan_to_num(), alone.nan_to_num())
    plain = _run(a, w)
    want = plain + bias
    assert torch.equal(got.isnan(), want.isnan()) and torch.equal(got.nan_to_num(), want.nan_to_num())
    assert bool(got[:, ::2].isinf().any()) and bool(got[:, ::2].isfinite().any())
