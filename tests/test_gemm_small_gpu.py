"""float32 products of operands down to the smallest that float32 has: a power of two in front of either operand changes nothing but the result's
own, and subnormal entries count in full, in every kernel."""
import pytest
import torch

from transformer_amd import kernels

pytestmark = pytest.mark.gpu

# tiles of 256 x 128, groups, 64 x 64, few rows, along the columns, whole lines through LDS at both lengths of k, short k
SHAPES = [(1021, 8192, 512), (513, 8200, 264), (1021, 2044, 2048), (130, 4100, 2000), (70, 4000, 2048), (33, 300, 1000), (12, 5200, 2048), (12, 5200, 4096),
          (8, 4100, 2048), (3, 500, 8192), (5, 40, 300), (300, 6000, 100), (300, 900, 24)]


def _draw(m, n, k):
    """Entries of either sign in 24 bits, 1 to 16 in size."""
    g = torch.Generator(device="cuda").manual_seed(m + 7 * n + 31 * k)

    def one(rows):
        x = 1 + torch.rand(rows, k, generator=g, device="cuda")
        x = x * 2.0 ** torch.randint(0, 4, (rows, k), generator=g, device="cuda")
        return x * (torch.randint(0, 2, (rows, k), generator=g, device="cuda") * 2 - 1)

    return one(m), one(n)


def _run(a, w):
    return kernels.gemm_simple(a, w, torch.empty(a.shape[0], w.shape[0], device="cuda"))


@pytest.mark.parametrize("m,n,k", SHAPES)
def test_powers_of_two_pass_through(m, n, k):
    a, w = _draw(m, n, k)
    plain = _run(a, w)
    for ea, ew in ((-120, 90), (90, -120), (-126, 70), (-45, -45)):          # the last bits of a product stay above 2^-149: chains round alike
        assert torch.equal(_run(a * 2.0 ** ea, w * 2.0 ** ew), plain * 2.0 ** (ea + ew)), (ea, ew)


@pytest.mark.parametrize("m,n,k", SHAPES)
def test_subnormal_entries_count(m, n, k):
    a, w = _draw(m, n, k)
    tiny = (a * 2.0 ** 17).trunc() * 2.0 ** -149                # up to 21 bits, of which the smallest float32 is one
    for x, y in ((tiny, w * 2.0 ** 90), (tiny * 2.0 ** 4, w * 2.0 ** 123)):   # the second past what a split operand takes
        exact = x.double() @ y.double().t()
        size = x.double().abs() @ y.double().abs().t()
        # as for entries of ordinary size (or, past the split's range, chains of fused multiply-adds)
        assert bool(((_run(x, y).double() - exact).abs() <= 1e-5 * size).all())
        assert float((_run(x, y).double() - exact).norm() / exact.norm()) < 5e-7
    few = torch.zeros_like(a)
    few[:, 0] = tiny[:, 0]
    got = _run(few, w * 2.0 ** 90)
    exact = few.double()[:, :1] * (w.double()[:, :1].t() * 2.0 ** 90)
    assert bool(((got.double() - exact).abs() <= 2.0 ** -21 * exact.abs()).all())


@pytest.mark.parametrize("m,n,k", [(1021, 16384, 2048), (513, 16386, 520)])
def test_gated_products_of_small_entries(m, n, k):
    a, w = _draw(m, n, k)
    w = w * (k ** -0.5 / 64)
    small, large = a * 2.0 ** -123, w * 2.0 ** 110
    assert kernels.split_glu_takes(small, large)
    got = kernels.gemm_split_glu(small, large, torch.empty(m, n // 2, device="cuda"))
    assert torch.equal(got, kernels.gemm_split_glu(a, w * 2.0 ** -13, torch.empty(m, n // 2, device="cuda")))
    assert torch.equal(got, kernels.swiglu(_run(small, large), torch.empty(m, n // 2, device="cuda")))
