"""Matrix states of long steps, 16 tokens at a time, against the walk token by token in 64 bits."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _t(a, dtype=torch.float32):
    return torch.as_tensor(np.ascontiguousarray(a)).to(DEV, dtype)


def _walk(q, k, v, a, S, bonus=None):
    """q, k, a [n, H, dk], v [n, H, dv], S [H, dk, dv], 64 bits: readouts and the last state."""
    out = []
    for t in range(len(q)):
        kv = k[t][:, :, None] * v[t][:, None, :]
        if bonus is not None:
            out.append(np.einsum("hkv,hk->hv", S + bonus[:, :, None] * kv, q[t]))
        S = a[t][:, :, None] * S + kv
        if bonus is None:
            out.append(np.einsum("hkv,hk->hv", S, q[t]))
    return np.array(out), S


def _case(rng, kind, H, dk, dv, lens, dtype, planes):
    """Runs one step of the kind's entry point; (readouts, states, 64-bit readouts, 64-bit states)."""
    from transformer_amd import kernels as K
    td = getattr(torch, dtype)
    nt, batch, dv = sum(lens), len(lens), dk if kind == "bonus" else dv
    pad = 3 if dk % 4 else 0                                     # rows that start off whole pieces
    cu = np.concatenate([[0], np.cumsum(lens)])
    slots = list(rng.permutation(batch + 2)[:batch])
    state = _t(rng.standard_normal((batch + 2, H, dk, dv)))
    first = state.double().cpu().numpy()
    draw = lambda n: torch.as_tensor(rng.standard_normal((nt, n + pad))).to(td)
    f64 = lambda x, h=H: x.double().numpy().reshape(nt, h, -1)
    args = (_t(cu, torch.int32), _t(slots, torch.int32))
    scalar = kind in ("ssm", "fixed")
    rows = 1 if planes == "least" else K.gla_row_parts(dk)
    assert K.recurrence_planes(dk, nt, batch, scalar, kind == "bonus") == 1
    o = torch.full((rows, nt, H, dv), float("nan"), device=DEV)
    bonus = None
    if kind == "channel":
        rank = 5
        a2, a2b = rng.standard_normal((H * dk, rank)), rng.standard_normal(H * dk) - 1.0
        proj = torch.as_tensor(rng.standard_normal((nt, 2 * H * dk + 2 * H * dv + rank))).to(td)
        alpha = torch.empty(nt, H * dk, device=DEV)
        K.gla_recurrent(proj.to(DEV), H, dk, dv, rank, _t(a2, td), _t(a2b), 1.5, state, *args, o, alpha)
        q, k, v = (f64(x) for x in proj.split([H * dk, H * dk, H * dv, H * dv + rank], 1)[:3])
        q, a = q * dk ** -0.5, alpha.double().cpu().numpy().reshape(nt, H, dk)
    elif kind == "bonus":
        rank, n = 4, H * dk
        rkvg = torch.as_tensor(rng.standard_normal((3, nt, n))).to(td)
        u = rng.standard_normal((H, dk)).astype(np.float32)
        decay = torch.empty(nt, n, device=DEV)
        K.wkv_recurrent(rkvg.to(DEV), _t(rng.standard_normal((nt, rank)), td), H, dk, dv, _t(rng.standard_normal((n, rank)), td),
                        _t(rng.standard_normal(n)), _t(u), state, *args, o, decay)
        q, k, v = (f64(x) for x in rkvg)
        a, bonus = decay.double().cpu().numpy().reshape(nt, H, dk), u.astype(np.float64)
    elif kind == "fixed":
        proj, d = draw(2 * H * dk + H * dv), rng.uniform(0, 1, H).astype(np.float32)
        d[0] = 0.0
        K.decay_recurrent(proj.to(DEV), 0, H * dk, 2 * H * dk, H, dk, dv, _t(d), 0.5, state, *args, o)
        q, k, v = (f64(x) for x in proj[:, :2 * H * dk + H * dv].split([H * dk, H * dk, H * dv], 1))
        q, a = 0.5 * q, np.broadcast_to(d.astype(np.float64)[None, :, None], (nt, H, dk))
    else:                                                        # two heads read the same B and C
        G = H // 2
        xbc, decay, dt = draw(H * dv + 2 * G * dk), _t(rng.uniform(0, 1, (nt, H))), _t(rng.uniform(0, 1, (nt, H)))
        decay[::5] = 0.0
        K.ssm_recurrent(xbc.to(DEV), 0, H * dv, H * dv + G * dk, H, G, dk, dv, decay, dt, state, *args, o)
        v, k, q = (x.double().numpy() for x in xbc[:, :H * dv + 2 * G * dk].split([H * dv, G * dk, G * dk], 1))
        v, k, q = v.reshape(nt, H, dv), *(np.repeat(x.reshape(nt, G, dk), 2, 1) for x in (k, q))
        k = k * dt.double().cpu().numpy()[:, :, None]
        a = np.broadcast_to(decay.double().cpu().numpy()[:, :, None], (nt, H, dk))
    want = [_walk(*(x[cu[i]:cu[i + 1]] for x in (q, k, v, a)), first[slots[i]], bonus) for i in range(batch)]
    ends = first.copy()
    for s, w in zip(slots, want):
        ends[s] = w[1]
    return o.double().sum(0).cpu().numpy(), state.double().cpu().numpy(), np.concatenate([w[0] for w in want]), ends


@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
@pytest.mark.parametrize("kind", ["channel", "bonus", "fixed", "ssm"])
@pytest.mark.parametrize("geom", [(2, 3, 5), (2, 64, 32), (2, 50, 33), (4, 128, 128), (2, 65, 129), (200, 100, 70), (100, 128, 130), (2, 250, 40)])
def test_chunks_match_the_walk(geom, kind, dtype):
    """Sequences that end inside, at and behind a chunk's edge; heads narrower and wider than a tile; workgroups of 32, 64
    and 128 columns (200 and 100 heads). A sum of n products of order 1 in 32 bits is off by about sqrt(n) 6e-8 of its
    terms' size: n is 16 + dk within a chunk, and every chunk passes the state on once."""
    H, dk, dv = geom
    if dk > 128 and kind in ("channel", "bonus"):
        pytest.skip("walked token by token")
    lens = [70, 1, 16, 17, 33] if H < 100 else [40, 9]
    got, state, want, ends = _case(np.random.default_rng(H + dk), kind, H, dk, dv, lens, dtype, "least" if dv % 2 else "all")
    for a, b in ((got, want), (state, ends)):
        assert np.linalg.norm(a - b) <= 2e-6 * np.linalg.norm(b)
        np.testing.assert_allclose(a, b, atol=6e-8 * 16 * (16 + dk) ** 0.5 * np.abs(b).max())


@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
@pytest.mark.parametrize("geom", [(8, 250, 530), (64, 64, 130), (9, 256, 512), (128, 30, 140)])
def test_matrix_memory_in_chunks_matches_its_walk(geom, dtype):
    """A million numbers of state: chunks, against the kernel that walks the same tokens (``lanes``). Either is a chain of
    32-bit products of order 1; denominators and normalisers come out of the chunks' own sums."""
    from transformer_amd import kernels as K
    H, dk, dv = geom
    rng, lens = np.random.default_rng(dk), [70, 33]
    nt, off = sum(lens), dk % 4
    rows = _t(rng.standard_normal((nt, off + 2 * H * dk + H * dv)), getattr(torch, dtype))
    keep, write = rng.uniform(0.5, 1.0, (nt, H)), rng.uniform(0, 1, (nt, H))
    keep[::3], keep[::5], write[::4] = 1.0, 0.0, 0.0
    first, norm = _t(rng.standard_normal((3, H, dk, dv))), _t(rng.standard_normal((3, H, dk)))
    got = []
    for lanes in (0, 16):
        state, n = first.clone(), norm.clone()
        o, den = torch.full((nt, H, dv), float("nan"), device=DEV), torch.full((nt, H), float("nan"), device=DEV)
        K.memory_recurrent(rows, off, off + H * dk, off + 2 * H * dk, dk ** -0.5, _t(keep), _t(write), state, n,
                           _t([0, 70, 103], torch.int32), _t([2, 0], torch.int32), o, den, lanes=lanes)
        got.append((o, den, state, n))
    for a, b in zip(*got):
        assert float((a - b).norm()) <= 3e-6 * float(b.norm())
        assert float((a - b).abs().max()) <= 6e-8 * 16 * (16 + dk) ** 0.5 * float(b.abs().max())
    assert torch.equal(got[0][2][1], first[1]) and torch.equal(got[0][3][1], norm[1])


@pytest.mark.parametrize("bad", [float("inf"), float("nan")])
def test_a_later_tokens_values_reach_no_earlier_one(bad):
    from transformer_amd import kernels as K
    H, dk, dv, n, at = 2, 64, 48, 60, 21
    g = torch.Generator().manual_seed(3)
    proj = torch.randn(n, 2 * H * dk + H * dv, generator=g).to(DEV)
    args = (_t([0, n], torch.int32), _t([0], torch.int32))

    def run(p):
        state, o = torch.zeros(1, H, dk, dv, device=DEV), torch.empty(1, n, H, dv, device=DEV)
        return K.decay_recurrent(p, 0, H * dk, 2 * H * dk, H, dk, dv, _t([0.9, 0.5]), 1.0, state, *args, o)[0]

    clean = run(proj)
    for column in (2 * H * dk + 7, H * dk + 5, 3):               # a value, a key, a query
        p = proj.clone()
        p[at, column] = bad
        o = run(p)
        assert torch.allclose(o[:at], clean[:at], rtol=1e-5, atol=1e-5)
        assert not torch.isfinite(o[at, 0]).all()
        assert torch.allclose(o[:, 1], clean[:, 1], rtol=1e-5, atol=1e-5)


def _f32_walk(q, k, v, a, S, bonus=None):
    """The walk token by token in float32 (one sequence): readouts and the last state."""
    out = torch.empty(q.shape[0], q.shape[1], v.shape[2], device=DEV)
    for t in range(q.shape[0]):
        kv = k[t, :, :, None] * v[t, :, None]
        before, S = S, torch.addcmul(kv, a[t, :, :, None], S)
        out[t] = ((S if bonus is None else torch.addcmul(before, bonus[:, :, None], kv)) * q[t, :, :, None]).sum(1)
    return out, S


def _off(got, want):
    return float((got.double() - want).norm() / want.norm())


@pytest.mark.parametrize("fade", [0.02, 0.5, 3.0])
@pytest.mark.parametrize("kind", ["channel", "bonus"])
def test_chunks_are_no_further_off_than_a_walk_in_32_bits(kind, fade):
    """Decays that last for hundreds of tokens, for tens and for a few. The products of a chunk's decays must not add up their
    roundings, nor may a readout be one chain over its channels: either doubles the error. What a chunk adds is one rounding
    of every decayed key, 2.5e-8 of it on average (2^-24 / sqrt(6)), which the walk of a state that soon forgets has not. A
    tenth is left for chance (the readout has 500 x 8 x 128 numbers)."""
    from transformer_amd import kernels as K
    H, d, n, rank = 8, 128, 500, 4
    g = torch.Generator(device=DEV).manual_seed(int(100 * fade))
    r = lambda *s: torch.randn(*s, generator=g, device=DEV)
    state, decay, o = r(1, H, d, d), torch.empty(n, H * d, device=DEV), torch.empty(1, n, H, d, device=DEV)
    first, args = state[0].clone(), (_t([0, n], torch.int32), _t([0], torch.int32))
    if kind == "channel":                        # log sigmoid(z) / 1: about -fade
        proj = r(n, 4 * H * d + rank).bfloat16()
        z = 0.3 * r(H * d) - np.log(np.expm1(fade))
        K.gla_recurrent(proj, H, d, d, rank, 0.1 * r(H * d, rank).bfloat16(), z, 1.0, state, *args, o, decay)
        q, k, v = (x.float().view(n, H, d) for x in proj[:, :3 * H * d].split(H * d, 1))
        q, u = q * d ** -0.5, None
    else:
        rkv, u = r(3, n, H * d).bfloat16(), 0.5 * r(H, d)
        K.wkv_recurrent(rkv, r(n, rank).bfloat16(), H, d, d, 0.1 * r(H * d, rank).bfloat16(), 0.3 * r(H * d) + np.log(fade), u,
                        state, *args, o, decay)
        q, k, v = (x.float().view(n, H, d) for x in rkv)
    a = decay.view(n, H, d)
    walked, last = _f32_walk(q, k, v, a, first, u)
    want, end = _walk(*(x.double().cpu().numpy() for x in (q, k, v, a, first)), None if u is None else u.double().cpu().numpy())
    want, end = _t(want, torch.float64), _t(end, torch.float64)
    for got, walk, exact in ((o[0], walked, want), (state[0], last, end)):
        assert _off(got, exact) <= 1.1 * (_off(walk, exact) ** 2 + 2.5e-8 ** 2) ** 0.5


@pytest.mark.parametrize("geom", [(8, 256, 512), (128, 64, 130), (256, 30, 140), (20, 250, 212)])
def test_matrix_memory_in_chunks_is_no_further_off_than_its_walk(geom):
    """A million numbers of state and more, 400 tokens: readouts, denominators, states and normalisers against 64 bits. What a
    chunk adds is one rounding of every decayed key, as above."""
    from transformer_amd import kernels as K
    (H, dk, dv), n = geom, 400
    g = torch.Generator(device=DEV).manual_seed(7)
    rows = torch.randn(n, 2 * H * dk + H * dv, generator=g, device=DEV).bfloat16()
    keep, write = 1 - 0.1 * torch.rand(n, H, generator=g, device=DEV), torch.rand(n, H, generator=g, device=DEV)
    q, k, v = (x.double().cpu().numpy().reshape(n, H, -1) for x in rows.split([H * dk, H * dk, H * dv], 1))
    k = k * write.double().cpu().numpy()[:, :, None]
    v = np.concatenate([v, np.ones((n, H, 1))], 2)                # the normaliser is a column of ones
    want, end = _walk(q * dk ** -0.5, k, v, np.broadcast_to(keep.double().cpu().numpy()[:, :, None], (n, H, dk)), np.zeros((H, dk, dv + 1)))
    want, end = _t(want, torch.float64), _t(end, torch.float64)
    off = []
    for lanes in (0, 16):
        state, norm = torch.zeros(1, H, dk, dv, device=DEV), torch.zeros(1, H, dk, device=DEV)
        o, den = torch.empty(n, H, dv, device=DEV), torch.empty(n, H, device=DEV)
        K.memory_recurrent(rows, 0, H * dk, 2 * H * dk, dk ** -0.5, keep, write, state, norm, _t([0, n], torch.int32),
                           _t([0], torch.int32), o, den, lanes=lanes)
        off.append([_off(o, want[..., :dv]), _off(den, want[..., dv]), _off(state[0], end[..., :dv]), _off(norm[0], end[..., dv])])
    assert all(a <= 1.1 * (b ** 2 + 2.5e-8 ** 2) ** 0.5 for a, b in zip(*off)), off


@pytest.mark.parametrize("column", ["key", "query"])
def test_an_infinite_number_stays_infinite(column):
    """Everything positive: sums that an infinite term enters are infinite, as the walk's are, and not undefined."""
    from transformer_amd import kernels as K
    H, d, n, rank, at = 2, 64, 60, 4, 21
    g = torch.Generator(device=DEV).manual_seed(3)
    proj = torch.rand(n, 4 * H * d + rank, generator=g, device=DEV) + 0.1
    proj[at, (H * d if column == "key" else 0) + 5] = float("inf")
    o, decay = torch.empty(2, n, H, d, device=DEV), torch.empty(n, H * d, device=DEV)
    K.gla_recurrent(proj.bfloat16(), H, d, d, rank, torch.zeros(H * d, rank, device=DEV).bfloat16(), torch.ones(H * d, device=DEV), 2.0,
                    torch.ones(1, H, d, d, device=DEV), _t([0, n], torch.int32), _t([0], torch.int32), o, decay)
    inf = torch.zeros(n, H, dtype=torch.bool, device=DEV)
    inf[at:, 0] = True if column == "key" else inf[at:, 0]
    inf[at, 0] = True
    got = o.sum(0)
    assert (got[inf] == float("inf")).all() and torch.isfinite(got[~inf]).all()


@pytest.mark.parametrize("geom,lens,chunks", [((2, 64, 32), [23, 23, 24], False), ((2, 64, 32), [24, 24, 24], True), ((3, 128, 64), [190, 193], False),
                                              ((3, 128, 64), [191, 193], True), ((3, 192, 64), [300], False), ((64, 192, 64), [40, 35], True),
                                              ((95, 128, 64), [30, 29], False), ((96, 128, 64), [30, 29], True)])
def test_both_sides_of_the_line_between_walk_and_chunks(geom, lens, chunks):
    """Few long sequences and many heads: the planes say which it is; readouts and states against 64 bits either way."""
    from transformer_amd import kernels as K
    H, dk, dv = geom
    nt, B = sum(lens), len(lens)
    ask = dict(scalar_decay=True, dtype=torch.bfloat16, heads=H, value_dim=dv)
    planes = K.recurrence_planes(dk, nt, B, **ask)
    assert planes == (1 if chunks else K.gla_row_parts(dk)) and K.gla_row_parts(dk) > 1
    assert K.recurrence_planes(dk, nt, B, **{**ask, "dtype": torch.float32}) == K.gla_row_parts(dk)
    g = torch.Generator(device=DEV).manual_seed(H + dk)
    rows = torch.randn(nt, 2 * H * dk + H * dv, generator=g, device=DEV).bfloat16()
    first, d = torch.randn(B, H, dk, dv, generator=g, device=DEV), torch.rand(H, generator=g, device=DEV)
    cu = np.concatenate([[0], np.cumsum(lens)])
    args, state, o = (_t(cu, torch.int32), _t(np.arange(B), torch.int32)), first.clone(), torch.full((planes, nt, H, dv), float("nan"), device=DEV)
    K.decay_recurrent(rows, 0, H * dk, 2 * H * dk, H, dk, dv, d, 0.5, state, *args, o)
    q, k, v = (x.double().cpu().numpy().reshape(nt, H, -1) for x in rows.split([H * dk, H * dk, H * dv], 1))
    a = np.broadcast_to(d.double().cpu().numpy()[None, :, None], (nt, H, dk))
    want = [_walk(*(x[cu[i]:cu[i + 1]] for x in (0.5 * q, k, v, a)), first[i].double().cpu().numpy()) for i in range(B)]
    assert _off(o.sum(0), _t(np.concatenate([w[0] for w in want]), torch.float64)) <= 2e-6
    assert _off(state, _t(np.array([w[1] for w in want]), torch.float64)) <= 2e-6


def test_the_entry_without_planes_keeps_its_arguments():
    """``ta_decay_recurrent`` takes the walk's planes and no number of them."""
    from ctypes import c_float, c_int, c_void_p
    from transformer_amd import kernels as K
    H, d, n = 3, 64, 50
    g = torch.Generator(device=DEV).manual_seed(1)
    rows, decays = torch.randn(n, 3 * H * d, generator=g, device=DEV).bfloat16(), torch.rand(H, generator=g, device=DEV)
    cu, slots = _t([0, n], torch.int32), _t([0], torch.int32)
    state, other = torch.zeros(1, H, d, d, device=DEV), torch.zeros(1, H, d, d, device=DEV)
    o, want = torch.empty(2, n, H, d, device=DEV), torch.empty(2, n, H, d, device=DEV)
    K.decay_recurrent(rows, 0, H * d, 2 * H * d, H, d, d, decays, 0.5, state, cu, slots, want)
    p = lambda t: c_void_p(t.data_ptr())
    rc = K.library().ta_decay_recurrent(K._stream(), c_int(K._code(rows.dtype)), p(rows), c_int(3 * H * d), c_int(0), c_int(H * d),
                                        c_int(2 * H * d), p(decays), c_float(0.5), p(other), p(cu), p(slots), c_int(1), c_int(n),
                                        c_int(H), c_int(d), c_int(d), p(o))
    torch.cuda.synchronize()
    assert rc == 0 and torch.equal(o, want) and torch.equal(state, other)
