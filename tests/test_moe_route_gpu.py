"""Routing with the scores in registers (64 or 256 of them) against routing with the scores in LDS, which more than 256 take: columns
that can't be chosen are added until it does, and the choices and the weights' bits stay."""
import pytest
import torch

from transformer_amd import kernels

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("E,top", [(1, 1), (8, 3), (63, 6), (64, 64), (65, 4), (200, 17), (256, 8)])
@pytest.mark.parametrize("score,renormalize,corrected", [("softmax", False, False), ("softmax", True, True), ("sigmoid", True, True)])
def test_scores_in_registers_choose_as_scores_in_lds(E, top, score, renormalize, corrected):
    g = torch.Generator(device="cuda").manual_seed(E + top)
    nt, inf = 20, float("inf")
    logits = (torch.randn(nt, E, generator=g, device="cuda") * 4).round() / 2            # equals among them
    logits[1], logits[2, ::2], logits[3, : E // 2] = float("nan"), float("nan"), -inf
    logits[4], logits[5] = 0.0, -0.0
    correction = (torch.randn(E, generator=g, device="cuda") * 4).round() / 8 if corrected else None
    wide = torch.cat([logits, torch.full((nt, 300 - E), -inf, device="cuda")], 1)
    also = torch.cat([correction, torch.full((300 - E,), -inf, device="cuda")]) if corrected else None
    out = lambda n: (torch.zeros(n, top, dtype=torch.int32, device="cuda"), torch.zeros(n, top, device="cuda"))
    want, got = out(nt), out(nt)
    kernels.moe_route(wide, 300, top, *want, score, renormalize, correction=also, factor=1.5)
    kernels.moe_route(logits, E, top, *got, score, renormalize, correction=correction, factor=1.5)
    # a choice that neither the softmax's zeros nor -inf can take, which is nobody's in the wide form
    some = torch.isfinite(logits).sum(1) >= top if score == "softmax" and not corrected else torch.ones(nt, dtype=torch.bool, device="cuda")
    assert torch.equal(got[0][some], want[0][some])
    assert torch.equal(torch.nan_to_num(got[1][some], 7.0).view(torch.int32), torch.nan_to_num(want[1][some], 7.0).view(torch.int32))
    few = out(16)
    if top <= 32:
        i32 = lambda n: torch.empty(n, dtype=torch.int32, device="cuda")
        rows = kernels.moe_max_rows(16 * top, E)
        kernels.moe_route_plan(logits[:16], E, top, *few, E, i32(rows), i32(rows // 16), i32(16 * top), score, renormalize,
                               correction=correction, factor=1.5)
        assert torch.equal(few[0], got[0][:16])
        assert torch.equal(torch.nan_to_num(few[1], 7.0), torch.nan_to_num(got[1][:16], 7.0))
