"""Latent attention of few single tokens: four waves a share of the keys, the heads' maps riding on the rotation and on the
merge, against 64 bits and against the kernels that they stand for."""
import pytest
import torch

from transformer_amd import kernels

pytestmark = pytest.mark.gpu
BF = torch.bfloat16


def _step(lens, H, rank, rot, dn, dv, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    rnd = lambda *s: torch.randn(*s, generator=g, device="cuda")
    B, W = len(lens), kernels.latent_row_width(rank, rot, BF)
    pages = max(lens) // 64 + 1
    table = torch.randperm(B * pages, generator=torch.Generator().manual_seed(seed)).int().view(B, pages).cuda()
    kc = torch.zeros(B * pages, 1, 64, W, device="cuda", dtype=BF)
    kc[..., :rank + rot] = rnd(B * pages, 1, 64, rank + rot).to(BF)
    return dict(B=B, W=W, table=table, kc=kc, q=rnd(B, H * (dn + rot)).to(BF), ang=rnd(B, rot // 2, 2), gate=rnd(B, H).to(BF),
                sink=rnd(H), uk=(rnd(H, dn, rank) / dn ** 0.5).to(BF), uv=(rnd(H, rank, dv) / rank ** 0.5).to(BF),
                cu=torch.arange(B + 1, dtype=torch.int32, device="cuda"), pos=torch.tensor(lens, dtype=torch.int32, device="cuda"))


def _rows(s, qa, lens, rank, rot, window, gate, sink, scale):
    """The weighted rows in 64 bits, from the wide queries as they are stored."""
    H = qa.shape[1]
    out = torch.empty(s["B"], H, rank, dtype=torch.float64, device="cuda")
    for b, n in enumerate(lens):
        first = max(0, n + 1 - window) if window else 0
        rows = s["kc"][s["table"][b].long()].view(-1, s["W"])[first:n + 1].double()
        sc = qa[b].double()[:, :rank + rot] @ rows[:, :rank + rot].t() * scale
        top = sc.amax(1, keepdim=True)
        e = (sc - top).exp()
        den = e.sum(1, keepdim=True) + ((s["sink"].double()[:, None] - top).exp() if sink else 0)
        out[b] = e / den @ rows[:, :rank]
        if gate:
            out[b] *= torch.sigmoid(s["gate"][b].double())[:, None]
    return out


@pytest.mark.parametrize("lens", [[0], [31, 32, 700], [900] * 4 + [63], [5, 1030, 64, 200, 0, 333, 95, 96, 1, 640, 17, 88, 500, 31, 33, 257]])
@pytest.mark.parametrize("H,rank,rot,dn,dv", [(16, 256, 64, 128, 128), (3, 136, 62, 40, 72), (20, 200, 0, 256, 8), (1, 8, 192, 1, 64)])
@pytest.mark.parametrize("window,gate,sink,shares", [(None, True, False, 17), (300, False, True, 2), (64, True, True, 70)])
def test_maps_against_64_bits_and_separate_kernels(lens, H, rank, rot, dn, dv, window, gate, sink, shares):
    s = _step(lens, H, rank, rot, dn, dv, len(lens) + H)
    B, scale = s["B"], (rank + rot) ** -0.5
    assert kernels.latent_maps_take(B, H, dn, rank, dv, shares)
    qa = torch.full((B, H, s["W"]), 9.0, device="cuda", dtype=BF)
    rot_dims = rot // 2 * 2
    kernels.latent_query_map(s["q"], H, dn, rot, rot_dims, s["ang"], s["uk"], qa, rank)
    plain = torch.full_like(qa, 9.0)
    kernels.latent_query_rot(s["q"], H, dn, rot, rot_dims, s["ang"], plain, rank)
    assert torch.equal(qa[:, :, rank:], plain[:, :, rank:])
    x, w = s["q"].view(B, H, dn + rot)[:, :, :dn].double().transpose(0, 1), s["uk"].double()
    want = (x @ w).transpose(0, 1)
    # a float32 sum of dn products and one rounding to 8 bits
    bound = 2.0 ** -8 * want.abs() + dn * 2.0 ** -23 * (x.abs() @ w.abs()).transpose(0, 1) + 1e-30
    assert bool(((qa[:, :, :rank].double() - want).abs() <= bound).all())

    g, k = s["gate"] if gate else None, s["sink"] if sink else None
    args = (s["table"], s["cu"], s["pos"])
    ol = torch.empty(B, H, rank, device="cuda", dtype=BF)
    kernels.latent_attention(qa, ol, s["kc"], *args, 1, rank, rot, scale, window, gate=g, shares=shares, sink=k)
    rows = _rows(s, qa, lens, rank, rot, window, gate, sink, scale)
    # exponentials and their sums to a few units of 2^-22, one rounding to 8 bits
    assert bool(((ol.double() - rows).abs() <= 2.0 ** -8 * rows.abs() + 2e-5).all())
    out = torch.full((B, H, dv), 9.0, device="cuda", dtype=BF)
    kernels.latent_attention_map(qa, s["uv"], out, s["kc"], *args, rank, rot, scale, window, g, shares, k)
    x, w = ol.double().transpose(0, 1), s["uv"].double()
    want = (x @ w).transpose(0, 1)
    bound = 2.0 ** -8 * want.abs() + rank * 2.0 ** -23 * (x.abs() @ w.abs()).transpose(0, 1) + 1e-30
    assert bool(((out.double() - want).abs() <= bound).all())


@pytest.mark.parametrize("H,rank,rot", [(40, 256, 64), (5, 512, 64), (3, 264, 120), (2, 130, 60)])
@pytest.mark.parametrize("shares", [2, 9, 33])
def test_shares_of_wide_rows_against_64_bits(H, rank, rot, shares):
    """Several tiles a sequence, rows of both widths that four waves share, quarters that end before the row does."""
    lens = [0, 100, 1500, 63]
    s = _step(lens, H, rank, rot, 8, 8, H)
    qa = torch.zeros(4, H, s["W"], device="cuda", dtype=BF)
    qa[..., :rank + rot] = torch.randn(4, H, rank + rot, generator=torch.Generator(device="cuda").manual_seed(H), device="cuda").to(BF)
    ol = torch.empty(4, H, rank, device="cuda", dtype=BF)
    kernels.latent_attention(qa, ol, s["kc"], s["table"], s["cu"], s["pos"], 1, rank, rot, 0.05, None, shares=shares)
    rows = _rows(s, qa, lens, rank, rot, None, False, False, 0.05)
    assert bool(((ol.double() - rows).abs() <= 2.0 ** -8 * rows.abs() + 2e-5).all())


def test_what_the_maps_refuse():
    s = _step([10] * 17, 2, 64, 16, 16, 16, 1)
    qa = torch.empty(17, 2, s["W"], device="cuda", dtype=BF)
    assert not kernels.latent_maps_take(17, 2, 16, 64, 16, 4) and not kernels.latent_maps_take(4, 2, 16, 64, 16, 1)
    assert not kernels.latent_maps_take(4, 2, 257, 64, 16, 4) and not kernels.latent_maps_take(4, 2, 16, 60, 16, 4)
    with pytest.raises(kernels.KernelError):
        kernels.latent_query_map(s["q"], 2, 16, 16, 16, s["ang"], s["uk"], qa, 64)


@pytest.mark.parametrize("H,rank,rot,window", [(40, 256, 64, None), (5, 512, 64, 70), (3, 264, 120, None), (2, 130, 60, 1), (63, 200, 0, 600)])
def test_one_share_of_wide_rows_against_64_bits(H, rank, rot, window):
    """Four waves a tile without a merge: the gate and the sink in their own epilogue."""
    lens = [0, 100, 1500, 63, 31, 32]
    s = _step(lens, H, rank, rot, 8, 8, H)
    qa = torch.zeros(len(lens), H, s["W"], device="cuda", dtype=BF)
    qa[..., :rank + rot] = torch.randn(len(lens), H, rank + rot, generator=torch.Generator(device="cuda").manual_seed(H), device="cuda").to(BF)
    for gate, sink in ((False, False), (True, True)):
        ol = torch.empty(len(lens), H, rank, device="cuda", dtype=BF)
        kernels.latent_attention(qa, ol, s["kc"], s["table"], s["cu"], s["pos"], 1, rank, rot, 0.05, window,
                                 gate=s["gate"] if gate else None, shares=1, sink=s["sink"] if sink else None)
        rows = _rows(s, qa, lens, rank, rot, window, gate, sink, 0.05)
        assert bool(((ol.double() - rows).abs() <= 2.0 ** -8 * rows.abs() + 2e-5).all())


@pytest.mark.parametrize("B,H", [(257, 16), (129, 32), (86, 40)])
def test_one_more_sequence_does_not_leave_the_keys_to_one_wave(B, H):
    """Where the rule goes from two shares to one, one takes about as long as two: a wave that walks a tile's keys by itself
    took five times as long."""
    rank, rot, n = 256, 64, 900
    g = torch.Generator(device="cuda").manual_seed(B)
    W, pages = rank + rot, n // 64 + 1
    table = torch.arange(B * pages, dtype=torch.int32, device="cuda").view(B, pages)
    kc = torch.randn(B * pages, 1, 64, W, generator=g, device="cuda", dtype=BF)
    qa = torch.randn(B, H, W, generator=g, device="cuda", dtype=BF)
    out = torch.empty(B, H, rank, device="cuda", dtype=BF)
    cu, pos = torch.arange(B + 1, dtype=torch.int32, device="cuda"), torch.full((B,), n, dtype=torch.int32, device="cuda")
    assert kernels.latent_key_shares(B, 1, H, rank, W, n + 1, None) == 1 and kernels.latent_key_shares(B - 1, 1, H, rank, W, n + 1, None) == 2

    def us(shares):
        best = float("inf")
        for _ in range(5):
            a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            a.record()
            for _ in range(10):
                kernels.latent_attention(qa, out, kc, table, cu, pos, 1, rank, rot, 0.05, None, shares=shares)
            b.record()
            b.synchronize()
            best = min(best, a.elapsed_time(b))
        return best

    us(2)
    assert us(1) < 2 * us(2)
