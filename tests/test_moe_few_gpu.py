"""The experts' products of few tokens by workgroups of 16, 32 and 64 rows of the matrix: against 64 bits, and with the bits
that every width gives (the waves divide k alike)."""
import pytest
import torch

from transformer_amd import kernels

pytestmark = pytest.mark.gpu
BF = torch.bfloat16


def _routing(nt, top, E, g):
    logits = torch.randn(nt, E, generator=g, device="cuda")
    i32 = lambda n: torch.empty(n, dtype=torch.int32, device="cuda")
    rows = kernels.moe_max_rows(nt * top, E)
    chosen, weight = torch.empty(nt, top, dtype=torch.int32, device="cuda"), torch.empty(nt, top, device="cuda")
    row_pair, tile_expert, pair_row = i32(rows), i32(rows // 16), i32(nt * top)
    kernels.moe_route_plan(logits, E, top, chosen, weight, E, row_pair, tile_expert, pair_row, "softmax", True)
    return chosen, weight, row_pair, tile_expert, pair_row


@pytest.mark.parametrize("pairs,E,rows", [(1, 32, 16), (4, 32, 64), (16, 32, 256), (40, 32, 528), (3, 1, 32), (17, 1, 32)])
def test_no_more_rows_than_the_chosen_experts_can_fill(pairs, E, rows):
    assert kernels.moe_max_rows(pairs, E) == rows


# (tokens, top, experts, columns, k): 16, 32 and 64 rows of the matrix a workgroup, at the lines between them and with a last
# workgroup of a few columns
@pytest.mark.parametrize("nt,top,E,N,K", [(1, 4, 32, 1024, 256), (4, 4, 32, 1024, 512), (4, 4, 32, 1025, 264), (4, 4, 32, 2048, 128),
                                          (4, 4, 32, 2049, 72), (16, 6, 20, 2000, 40), (1, 1, 3, 5, 8), (2, 2, 5, 17, 1000)])
def test_products_against_64_bits(nt, top, E, N, K):
    g = torch.Generator(device="cuda").manual_seed(N + K + nt)
    chosen, weight, row_pair, tile_expert, pair_row = _routing(nt, top, E, g)
    rows = row_pair.numel()
    h = torch.randn(nt, K, generator=g, device="cuda").to(BF)
    w = (torch.randn(E, N, K, generator=g, device="cuda") / K ** 0.5).to(BF)
    at, expert = pair_row.long(), chosen.view(-1).long()
    token = torch.arange(nt * top, device="cuda") // top
    x, m = h[token].double(), w[expert].double()
    want = (m @ x[:, :, None])[:, :, 0]
    # a float32 sum of K products, in another order
    slack = K * 2.0 ** -23 * (m.abs() @ x.abs()[:, :, None])[:, :, 0]
    a = torch.zeros(rows, K, device="cuda", dtype=BF)
    a[at] = h[token]
    plain = kernels.moe_gemm(a, w, tile_expert, torch.full((rows, N), 7.0, device="cuda"))
    assert bool(((plain[at].double() - want).abs() <= slack + 1e-30).all())
    got = kernels.moe_gemm_tokens(h, top, row_pair, None, w, tile_expert, torch.empty(rows, N, device="cuda", dtype=BF), None)
    assert torch.equal(got[at], plain[at].to(BF))
    if N % 2 == 0:
        got = kernels.moe_gemm_tokens(h, top, row_pair, None, w, tile_expert, torch.empty(rows, N // 2, device="cuda", dtype=BF), None, glu=True)
        both = plain[at].to(BF).float()
        gate, up = both[:, :N // 2], both[:, N // 2:]
        want = gate / (1.0 + torch.exp(-gate)) * up
        # the exponential and the division to a few units of 2^-22, one rounding to 8 bits
        assert bool(((got[at].float() - want).abs() <= 2.0 ** -8 * want.abs() + 1e-6).all())
