"""float32 products of rows that lie further apart than 32-bit offsets of a tile's rows reach."""
import pytest
import torch

from test_gemm_split_form import FAR, form
from transformer_amd import kernels

pytestmark = pytest.mark.gpu

STEP = 4194308


def _far(x, shift):
    room = torch.empty(x.shape[0] * STEP + 8, device="cuda")
    y = room.as_strided(x.shape, (STEP, 1), shift)
    y.copy_(x)
    return y


@pytest.mark.parametrize("m,n,k,which,shift", [(300, 9000, 1292, "a", 0), (300, 2044, 2044, "a", 0), (333, 4500, 1027, "a", 1), (1021, 900, 300, "w", 0), (1021, 900, 100, "w", 4), (20, 300, 2048, "a", 0)])
def test_the_same_bits(m, n, k, which, shift):
    g = torch.Generator(device="cuda").manual_seed(k)
    a, w = torch.randn(m, k, generator=g, device="cuda"), torch.randn(n, k, generator=g, device="cuda")
    want = kernels.gemm_simple(a, w, torch.empty(m, n, device="cuda"))
    assert form(m, n, k, STEP if which == "a" else None, STEP if which == "w" else None) >= FAR or m == 20
    x, y = (_far(a, shift), w) if which == "a" else (a, _far(w, shift))
    assert torch.equal(kernels.gemm_simple(x, y, torch.empty(m, n, device="cuda")), want)
    del x, y
    torch.cuda.empty_cache()
