"""float32 products over a short k are chains of fused multiply-adds, each rounded once, and a row has the same bits alone."""
import pytest
import torch

from transformer_amd import kernels

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("k", [1, 2, 3, 4, 5, 8, 13, 16, 31, 32, 33])
@pytest.mark.parametrize("m,n", [(1, 16384), (5, 40), (70, 12290), (300, 900), (1100, 5570)])
def test_chains(m, n, k):
    g = torch.Generator(device="cuda").manual_seed(m + 7 * n + 31 * k)
    a, w = torch.randn(m, k, generator=g, device="cuda"), torch.randn(n, k, generator=g, device="cuda")
    room = torch.full((m + 1, n + 2), 7.0, device="cuda")
    got = kernels.gemm_simple(a, w, room[:m, 1:n + 1])
    assert bool((room[:, 0] == 7).all()) and bool((room[:, n + 1] == 7).all()) and bool((room[m] == 7).all())
    # each addition rounds by at most 2^-24 of what it gives; past k = 32 what the split leaves out and six sums of a block besides
    off = (got.double() - a.double() @ w.double().t()).abs()
    bound = k * 2.0 ** -24 if k <= 32 else 3e-7 + 8 * 2.0 ** -23
    assert bool((off <= bound * (1 + 1e-6) * (a.double().abs() @ w.double().abs().t())).all())
    rows = sorted({0, m // 2, m - 1})
    alone = torch.cat([kernels.gemm_simple(a[i:i + 1].contiguous(), w, torch.empty(1, n, device="cuda")) for i in rows])
    assert torch.equal(alone, got[rows])
