"""The experts' products through LDS in steps of 64 k, rows one step ahead and columns two: the bits of the kernel without LDS
(the same instruction over the same ascending k)."""
import pytest
import torch

from transformer_amd import kernels

pytestmark = pytest.mark.gpu
BF = torch.bfloat16


# k of one to six whole steps, of a last step of 8, 32, 40 and 56; runs within, at and over a block of 16 tiles, short ones
# several to a workgroup
@pytest.mark.parametrize("K", [64, 128, 192, 384, 72, 160, 232, 312])
@pytest.mark.parametrize("runs,N", [((16, 1, 1, 1, 18), 512), ((5, 0, 33, 2, 2), 300)])
def test_steps_through_lds_equal_operands_from_memory(K, runs, N):
    g = torch.Generator(device="cuda").manual_seed(K + N)
    tiles = [e for e, n in enumerate(runs) for _ in range(n)]
    tile_expert = torch.tensor(tiles + [-1], dtype=torch.int32, device="cuda")
    rows = 16 * len(tile_expert)
    a = torch.randn(rows, K, generator=g, device="cuda").to(BF)
    w = (torch.randn(len(runs), N, K, generator=g, device="cuda") / K ** 0.5).to(BF)
    want = kernels.moe_gemm(a, w, tile_expert, torch.full((rows, N), 7.0, device="cuda"), form="direct")
    for _ in range(3):
        got = kernels.moe_gemm(a, w, tile_expert, torch.full((rows, N), 7.0, device="cuda"), form="lds")
        assert torch.equal(got, want)
