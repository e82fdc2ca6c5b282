"""float32 products of few rows over a short k, whose waves share a segment: the bits that the same rows have among so many that they go by tiles, at the
edges of its tiles of 8 to 64 rows, of blocks and segments, of what it takes, and side by side."""
import pytest
import torch

from test_gemm_split_form import form
from transformer_amd import kernels

pytestmark = pytest.mark.gpu

MANY, WIDE = 1100, 5570


def _draw(rows, k, seed):
    return torch.randn(rows, k, generator=torch.Generator(device="cuda").manual_seed(seed), device="cuda")


@pytest.mark.parametrize("k", [33, 36, 64, 65, 96, 128, 160, 255, 256, 257, 260, 384, 511, 512, 513, 516, 640, 641, 768, 772, 1000, 1024, 1028, 1280, 1284, 1500, 2048, 2500])
def test_the_bits_of_the_same_rows_among_many(k):
    a, w = _draw(MANY, k, 1), _draw(WIDE, k, 2)
    assert form(MANY, WIDE, k) > 0
    many = kernels.gemm_simple(a, w, torch.empty(MANY, WIDE, device="cuda"))
    for m in (1, 7, 8, 9, 16, 17, 31, 32, 33, 64, 65, 100):
        for n in (5, 64, 1027):                    # fewer and more columns of the same matrix: other numbers of workgroups
            room = torch.full((m + 1, n + 2), 7.0, device="cuda")
            got = kernels.gemm_simple(a[:m], w[:n], room[:m, 1:n + 1])
            assert torch.equal(got, many[:m, :n]), (m, n)
            assert bool((room[:, 0] == 7).all()) and bool((room[:, n + 1] == 7).all()) and bool((room[m] == 7).all())
    wide = kernels.gemm_simple(a[:33], w, torch.empty(33, WIDE, device="cuda"))
    assert torch.equal(wide, many[:33])
    exact = a[:33].double() @ w.double().t()
    assert float((wide.double() - exact).norm() / exact.norm()) < 2e-7


@pytest.mark.parametrize("k", [48, 200, 512, 700])
@pytest.mark.parametrize("m", [1, 12, 30, 50])
def test_side_by_side_and_with_a_bias(m, k):
    a, w = _draw(7 * m, k, 3).view(7, m, k), _draw(7 * 300, k, 4).view(7, 300, k)
    got = kernels.gemm_simple_batched(a, w, torch.empty(7, m, 300, device="cuda"))
    bias = _draw(1, 300, 5)[0]
    for i in range(7):
        alone = kernels.gemm_simple(a[i], w[i], torch.empty(m, 300, device="cuda"))
        assert torch.equal(got[i], alone)
        assert torch.equal(kernels.gemm_simple(a[i], w[i], torch.empty(m, 300, device="cuda"), bias), alone + bias)
