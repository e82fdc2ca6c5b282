"""Kernels of steps of few tokens: gated linear attention in one kernel, the diagonal recurrence's gates."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _t(a, dtype=torch.float32):
    return torch.as_tensor(np.ascontiguousarray(a)).to(DEV, dtype)


@pytest.mark.parametrize("weights", ["float32", "bfloat16"])
@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
@pytest.mark.parametrize("bonus", [False, True])
@pytest.mark.parametrize("geom", [(3, 64, 64, 64), (2, 128, 128, 16), (2, 16, 64, 3), (5, 256, 16, 9), (1, 64, 256, 100), (2, 192, 32, 1)])
def test_a_step_in_one_kernel_equals_its_kernels(geom, bonus, dtype, weights):
    """Decays, recurrence and head norm as kernels of their own, against ``gla_step``. The decays' sums and the readout's are
    taken in another order: some 2e-7 of a result that is a sum of dk products, then one rounding to the output's type."""
    from transformer_amd import kernels as K
    H, dk, dv, rank = geom
    if weights == "bfloat16" and dtype == "float32":
        pytest.skip("float32 rows have float32 weights")
    if bonus and dk != dv:
        pytest.skip("heads of the bonus recurrence are square")
    assert K.gla_step_fits(dk, dv)
    td, tw = getattr(torch, dtype), getattr(torch, weights)
    rng, B, n = np.random.default_rng(dk + rank), 4, H * dk
    cu, slots = _t(np.arange(B + 1), torch.int32), _t([5, 0, 3, 1], torch.int32)
    first = _t(rng.standard_normal((6, H, dk, dv)))
    a2, a2b, w = _t(rng.standard_normal((n, rank)), tw), _t(rng.standard_normal(n)), _t(1 + 0.2 * rng.standard_normal(n if bonus else dv))
    s0, s1, alpha = first.clone(), first.clone(), torch.empty(B, n, device=DEV)
    o = torch.empty(K.gla_row_parts(dk), B, H, dv, device=DEV)
    want, got = torch.empty(B, H * dv, dtype=td, device=DEV), torch.empty(B, H * dv, dtype=td, device=DEV)
    if bonus:
        rkvg, low, u = _t(rng.standard_normal((4, B, n)), td), _t(rng.standard_normal((B, rank)), td), _t(rng.standard_normal((H, dk)))
        K.wkv_recurrent(rkvg, low, H, dk, dv, a2, a2b, u, s0, cu, slots, o, alpha)
        K.head_norm_gate(o, rkvg[3], H, dv, w, 1e-5, want)
        K.gla_step(rkvg[0], 0, B * n, 2 * B * n, low, a2, a2b, 1.0, 1.0, u, s1, slots, rkvg[3], w, 1e-5, got)
    else:
        proj = _t(rng.standard_normal((B, 2 * n + 2 * H * dv + rank)), td)
        K.gla_recurrent(proj, H, dk, dv, rank, a2, a2b, 4.0, s0, cu, slots, o, alpha)
        K.gla_out(o, proj, H, dk, dv, w, 1e-5, want)
        g = 2 * n + H * dv
        K.gla_step(proj, 0, n, 2 * n, proj[:, g + H * dv:], a2, a2b, 4.0, dk ** -0.5, None, s1, slots, proj[:, g:g + H * dv], w,
                   1e-5, got)
    np.testing.assert_allclose(s1.cpu(), s0.cpu(), atol=2e-6 * float(s0.abs().max()))
    one = 2e-5 if dtype == "float32" else 2 ** -7
    np.testing.assert_allclose(got.float().cpu(), want.float().cpu(), atol=one * float(want.float().abs().max()), rtol=one)
    assert torch.equal(s1[[2, 4]], first[[2, 4]])


@pytest.mark.parametrize("geom", [(32, 128, 128), (16, 64, 64), (8, 256, 64), (8, 192, 64)])
def test_a_step_in_one_kernel_is_no_further_off_than_its_kernels(geom):
    """Against 64 bits, whole rows in float32; a twentieth for chance (64 x H x dv numbers)."""
    from transformer_amd import kernels as K
    H, dk, dv = geom
    B, rank, n = 64, 16, H * dk
    g = torch.Generator(device=DEV).manual_seed(dk)
    r = lambda *s: torch.randn(*s, generator=g, device=DEV)
    proj, a2, a2b, w, first = r(B, 2 * n + 2 * H * dv + rank), r(n, rank) / 4, 0.3 * r(n), 1 + 0.1 * r(dv), 3 * r(B, H, dk, dv)
    cu, slots, at = _t(np.arange(B + 1), torch.int32), _t(np.arange(B), torch.int32), 2 * n + H * dv
    out, alone = torch.empty(B, H * dv, device=DEV), torch.empty(B, H * dv, device=DEV)
    o, alpha = torch.empty(K.gla_row_parts(dk), B, H, dv, device=DEV), torch.empty(B, n, device=DEV)
    K.gla_step(proj, 0, n, 2 * n, proj[:, at + H * dv:], a2, a2b, 16.0, dk ** -0.5, None, first.clone(), slots,
               proj[:, at:at + H * dv], w, 1e-5, out)
    K.gla_recurrent(proj, H, dk, dv, rank, a2, a2b, 16.0, first.clone(), cu, slots, o, alpha)
    K.gla_out(o, proj, H, dk, dv, w, 1e-5, alone)
    x = proj.double()
    q, k, v = (t.reshape(B, H, -1) for t in x[:, :at].split([n, n, H * dv], 1))
    a = (torch.sigmoid(x[:, at + H * dv:] @ a2.double().T + a2b.double()) ** (1 / 16)).view(B, H, dk, 1)
    y = ((a * first.double() + k[..., None] * v[:, :, None]) * q[..., None]).sum(2) * dk ** -0.5
    y = y * torch.rsqrt((y * y).mean(-1, keepdim=True) + 1e-5) * w.double()
    gate = x[:, at:at + H * dv]
    want = y.reshape(B, -1) * gate * torch.sigmoid(gate)
    off, walk = (float((t.double() - want).norm() / want.norm()) for t in (out, alone))
    assert off <= 1.05 * walk


def test_heads_that_a_step_takes_and_refuses():
    from transformer_amd import kernels as K
    takes = [(64, 64), (128, 128), (16, 64), (256, 64), (64, 256), (32, 32)]
    refuses = [(128, 256), (8, 128), (64, 48), (20, 64), (512, 32), (16, 16), (64, 512)]
    assert all(K.gla_step_fits(*g) for g in takes) and not any(K.gla_step_fits(*g) for g in refuses)


@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
@pytest.mark.parametrize("geom", [(2, 64, 4), (3, 128, 1), (1, 256, 4), (2, 320, 2), (4, 640, 2)])
@pytest.mark.parametrize("lens", [[1], [1, 1, 1, 1, 1], [2, 1, 5], [1] * 17, [3, 250], [2, 0], [0, 2, 1], [1] * 16 + [0, 2]])
def test_gates_of_few_tokens(lens, geom, dtype):
    """Blocks of whole 64 inputs, against the formulas in 64 bits: sums of ``size`` products of order 1 / sqrt(size). As many
    tokens as sequences, too, where a sequence brings none and another two, and blocks so wide that 253 tokens go by the tiles."""
    from transformer_amd import kernels as K
    nb, size, taps = geom
    C, nt, B = nb * size, sum(lens), len(lens)
    td = getattr(torch, dtype)
    rng = np.random.default_rng(size + nt)
    yx = torch.as_tensor(rng.standard_normal((nt, 2 * C))).to(td)
    gw = torch.as_tensor(rng.standard_normal((2 * nb, size, size)) / size ** 0.5).to(td)
    f = lambda *s: torch.as_tensor(rng.standard_normal(s), dtype=torch.float32)
    xb, cb, lam, gb, tp, mem = f(C), f(C), f(C), f(2 * nb, size), f(C, taps), f(B + 1, taps - 1, C)
    slots = list(range(B, 0, -1))
    cu = np.concatenate([[0], np.cumsum(lens)])
    a, b = torch.empty(nt, C, device=DEV), torch.empty(nt, C, device=DEV)
    d = [x.to(DEV) for x in (yx, xb, tp, cb, mem, gw, gb, lam)]
    K.rglru_gates(d[0], C, d[1], d[2], d[3], d[4], d[5], d[6], d[7], 8.0, _t(cu, torch.int32), _t(slots, torch.int32), a, b)
    x, w = yx[:, C:].double() + xb.double(), gw.double()
    for i in range(B):
        rows = torch.cat([mem[slots[i]].double(), x[cu[i]:cu[i + 1]]])
        if not lens[i]:
            continue
        u = torch.stack([cb.double() + (rows[t:t + taps] * tp.double().T).sum(0) for t in range(lens[i])])
        ub = u.view(-1, nb, size)
        r, g = (torch.sigmoid(torch.einsum("tbi,boi->tbo", ub, w[z * nb:(z + 1) * nb]) + gb[z * nb:(z + 1) * nb].double()).reshape(-1, C)
                for z in (0, 1))
        log = -8.0 * r * torch.nn.functional.softplus(lam.double())
        np.testing.assert_allclose(a[cu[i]:cu[i + 1]].cpu(), log.exp(), atol=1e-5)
        np.testing.assert_allclose(b[cu[i]:cu[i + 1]].cpu(), (-torch.expm1(2 * log)).sqrt() * g * u, atol=2e-5, rtol=2e-5)


@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
@pytest.mark.parametrize("taps", [1, 2, 4, 8])
@pytest.mark.parametrize("channels", [4, 260, 1028])
def test_convolution_of_four_channels_a_thread_has_the_bits_of_one(channels, taps, dtype):
    """Rows that start on whole pieces against the same rows a column further: sequences that end inside, at and behind a
    thread's sixteen tokens, biases, activation, and the memory that is left behind."""
    from transformer_amd import kernels as K
    td, lens = getattr(torch, dtype), [1, 2, 30, 16, 5, 40]
    nt, C = sum(lens), channels
    g = torch.Generator(device=DEV).manual_seed(C + taps)
    r = lambda *s: torch.randn(*s, generator=g, device=DEV)
    x, w, bi, bo, mem = r(nt, C).to(td), r(C, taps), r(C), r(C), r(8, taps - 1, C)
    cu, slots = _t(np.concatenate([[0], np.cumsum(lens)]), torch.int32), _t([7, 0, 3, 2, 5, 6], torch.int32)
    got = []
    for off in (4, 5):
        rows = torch.zeros(nt, C + 8, dtype=td, device=DEV)
        rows[:, off:off + C] = x
        state = mem.clone() if taps > 1 else None
        out = torch.full((nt, C + 4), 7.0, dtype=td, device=DEV)
        K.causal_conv(rows, off, C, w, out[:, :C], state, cu, slots, max(lens), bias_in=bi, bias_out=bo, activation="silu")
        assert (out[:, C:] == 7).all()
        got.append((out[:, :C], state))
    assert torch.equal(got[0][0], got[1][0]) and torch.isfinite(got[0][0]).all()
    if taps > 1:
        assert torch.equal(got[0][1], got[1][1])


@pytest.mark.parametrize("dtype,last", [("bfloat16", 640), ("float32", 1340)])
@pytest.mark.parametrize("taps", [1, 2, 4, 8])
def test_large_convolutions_have_the_bits_of_one_channel_a_thread(taps, dtype, last):
    """As above with as many numbers as it takes four channels a thread (8 million, 16 million in float32), the last workgroup of
    a row part of one."""
    from transformer_amd import kernels as K
    td, lens, C = getattr(torch, dtype), [1, 2, 30, 16, last, 5], 12292
    nt, most = sum(lens), (16 if dtype == "float32" else 8) << 20
    assert nt * C >= most
    g = torch.Generator(device=DEV).manual_seed(taps)
    r = lambda *s: torch.randn(*s, generator=g, device=DEV)
    x, w, bi, bo, mem = r(nt, C).to(td), r(C, taps), r(C), r(C), r(8, taps - 1, C)
    cu, slots = _t(np.concatenate([[0], np.cumsum(lens)]), torch.int32), _t([7, 0, 3, 2, 5, 6], torch.int32)
    got = []
    for off in (4, 5):
        rows = torch.zeros(nt, C + 8, dtype=td, device=DEV)
        rows[:, off:off + C] = x
        state = mem.clone() if taps > 1 else None
        out = torch.full((nt, C + 4), 7.0, dtype=td, device=DEV)
        K.causal_conv(rows, off, C, w, out[:, :C], state, cu, slots, max(lens), bias_in=bi, bias_out=bo, activation="silu")
        assert (out[:, C:] == 7).all()
        got.append((out[:, :C], state))
    assert torch.equal(got[0][0], got[1][0]) and torch.isfinite(got[0][0]).all()
    if taps > 1:
        assert torch.equal(got[0][1], got[1][1])
