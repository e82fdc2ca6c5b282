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


# either side of the lines between the forms, by the size of the matrices: the form that is taken has its own bits, and the sums
# of the two differ by the order of K products
@pytest.mark.parametrize("tiles,N,K", [(1023, 256, 8), (1024, 256, 8), (511, 512, 10232), (512, 512, 10232), (699, 512, 10240), (700, 512, 10240)])
def test_line_between_the_forms(tiles, N, K):
    g = torch.Generator(device="cuda").manual_seed(tiles)
    tile_expert = torch.full((tiles,), -1, dtype=torch.int32, device="cuda")
    tile_expert[:3] = torch.tensor([0, 0, 1])
    a = torch.zeros(tiles * 16, K, device="cuda", dtype=BF)
    a[:48] = torch.randn(48, K, generator=g, device="cuda").to(BF)
    w = (torch.randn(2, N, K, generator=g, device="cuda") / K ** 0.5).to(BF)
    run = lambda form: kernels.moe_gemm(a, w, tile_expert, torch.full((tiles * 16, N), 7.0, device="cuda"), form=form)[:48]
    few, lds, taken = run("split_k"), run("lds"), run("auto")
    line = 1024 if N * K < 5 << 20 else 1400
    assert torch.equal(taken, few if tiles * ((N + 255) // 256) < line else lds)
    weight = torch.cat([w[:1], w[:1], w[1:]]).float().abs()
    slack = K * 2.0 ** -23 * torch.bmm(a[:48].float().abs().view(3, 16, K), weight.transpose(1, 2).contiguous()).view(48, N)
    assert bool(((few - lds).abs() <= slack + 1e-30).all())
