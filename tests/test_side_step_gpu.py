"""The end of a block with a token side input in one kernel: against its kernels one by one and against 64 bits, for a plain result in planes and for experts' rows,
at the widths, side columns and numbers of tokens that it takes."""
import pytest
import torch

from transformer_amd import kernels

pytestmark = pytest.mark.gpu


def _g(*shape, seed=0, scale=1.0, dtype=torch.float32):
    gen = torch.Generator(device="cuda").manual_seed(seed)
    return (torch.randn(*shape, generator=gen, device="cuda") * scale).to(dtype)


def _one_by_one(x, delta, w, eps, gate, side, proj, v, eps_side, w_next, eps_next):
    cast = torch.empty(x.shape, device="cuda", dtype=torch.bfloat16)
    kernels.postnorm_add(x, delta, w, eps, xcast=cast)
    g = kernels.activation(kernels.gemm_simple(cast, gate, torch.empty(x.shape[0], gate.shape[0], device="cuda", dtype=torch.float32)),
                           torch.empty(x.shape[0], gate.shape[0], device="cuda"), "gelu_tanh", side=side).bfloat16()
    y = kernels.gemm_simple(g, proj, torch.empty_like(x))
    before = x.clone()
    out = torch.empty(x.shape, device="cuda", dtype=torch.bfloat16)
    kernels.postnorm_add(x, y, v, eps_side, next_weight=w_next, next_eps=eps_next, out=out)
    return before, x, out


def _exact(x, given, w, eps, gate, side, proj, v, eps_side, w_next, eps_next):
    """In 64 bits from the operands on, nothing rounded: what the result's own add gives, the stream behind both, the next norm."""
    norm = lambda t, gain, e: t * (t.square().mean(1, keepdim=True) + e).rsqrt() * gain.double()
    if isinstance(given, kernels.RoutedRows):
        g = given
        pairs = g.pair_row.view(x.shape[0], g.top).long()
        parts = torch.where((pairs >= 0)[..., None], g.rows.double()[pairs.clamp_min(0)], 0.0)
        delta = (parts if g.weight is None else parts * g.weight.double()[..., None]).sum(1)
        if g.shared is not None:
            shared = g.shared.double() if g.shared.dim() == 2 else g.shared.double().sum(0)
            delta = delta + (shared if g.shared_gate is None else shared * torch.sigmoid(g.shared_gate.double()))
    else:
        delta = given.double() if given.dim() == 2 else given.double().sum(0)
    before = x.double() + norm(delta, w, eps)
    g = torch.nn.functional.gelu(before @ gate.double().t(), approximate="tanh") * side.double()
    after = before + norm(g @ proj.double().t(), v, eps_side)
    return before, after, norm(after, w_next, eps_next)


@pytest.mark.parametrize("nt,d,dim,kind", [(1, 512, 32, "plain"), (4, 2048, 64, "routed"), (64, 1024, 128, "routed"), (7, 4096, 64, "planes"),
                                           (3, 1536, 32, "gated"), (5, 2560, 128, "weighted"), (16, 2048, 64, "planes"), (2, 4096, 128, "gated")])
def test_side_step(nt, d, dim, kind):
    x0, w, v, w_next = _g(nt, d, seed=1), 1 + _g(d, seed=2, scale=.1), 1 + _g(d, seed=3, scale=.1), 1 + _g(d, seed=4, scale=.1)
    gate, proj = _g(dim, d, seed=5, scale=d ** -.5, dtype=torch.bfloat16), _g(d, dim, seed=6, scale=dim ** -.5, dtype=torch.bfloat16)
    side = _g(nt, 3 * dim, seed=7)[:, dim:2 * dim]
    if kind in ("plain", "planes"):
        delta = given = _g(nt, d, seed=8) if kind == "plain" else _g(3, nt, d, seed=8)
    else:
        top = 6 if kind == "weighted" else 4
        rows, pair_row = _g(nt * top + 5, d, seed=9), torch.randperm(nt * top + 5, device="cuda")[:nt * top].int()
        pair_row[::5] = -1                       # a pair without a row adds nothing
        pw = _g(nt, top, seed=10).abs() if kind == "weighted" else None
        shared = _g(2, nt, d, seed=11) if kind == "gated" else _g(nt, d, seed=11) if kind == "routed" else None
        shared_gate = _g(nt, 9, seed=12)[:, 8:] if kind == "gated" else None
        given = kernels.RoutedRows(rows, top, pair_row, pw, shared, shared_gate)
        delta = kernels.moe_combine(rows, top, pair_row, pw, shared, shared_gate, torch.empty(nt, d, device="cuda"))
    args = (w, 1e-5, gate, side, proj, v, 1e-6, w_next, 1e-5)
    before, want, want_out = _one_by_one(x0.clone(), delta, *args)
    out = torch.empty(nt, d, device="cuda", dtype=torch.bfloat16)
    got = kernels.side_step(x0.clone(), given, *args, out=out)
    # sums in another order may move a row's bfloat16 copy or a gated column by one rounding, 2^-8 of it, and what the side input adds by as much
    added = (want - before).norm(dim=1)
    assert bool(((got - want).norm(dim=1) <= 2.0 ** -8 * added + 1e-5 * want.norm(dim=1)).all())
    assert bool(((out.float() - want_out.float()).norm(dim=1) <= 2.0 ** -7 * want_out.float().norm(dim=1)).all())
    assert torch.equal(kernels.side_step(x0.clone(), given, *args[:-2]), got)          # without a norm behind it
    # against 64 bits: the rows' and the gated columns' bfloat16 copies are 2^-9 off at the most each, and so is what the side input adds, in the
    # norm over a row; the rest is 32 bits, and the next norm's rows are rounded once more
    exact_before, exact, exact_out = _exact(x0, given, *args)
    added = (exact - exact_before).norm(dim=1)
    bound = 2.0 ** -8 * added + 1e-6 * exact.norm(dim=1)
    assert bool(((got.double() - exact).norm(dim=1) <= bound).all())
    assert bool(((out.double() - exact_out).norm(dim=1) <= (2.0 ** -9 + bound / exact.norm(dim=1)) * 1.01 * exact_out.norm(dim=1)).all())
    # and no further from them than the kernels one by one, but for the closeness of two roundings
    assert float((got.double() - exact).norm()) <= 1.5 * float((want.double() - exact).norm())


def test_who_takes_it_and_what_it_refuses():
    gate, proj = _g(64, 2048, dtype=torch.bfloat16), _g(2048, 64, dtype=torch.bfloat16)
    assert kernels.side_step_takes(4, 2048, gate, proj) and not kernels.side_step_takes(65, 2048, gate, proj)
    assert not kernels.side_step_takes(4, 2048, gate.float(), proj) and not kernels.side_step_takes(4, 2048, gate[:48].contiguous(), proj[:, :48].contiguous())
    x, w = _g(2, 2048), _g(2048)
    with pytest.raises(kernels.KernelError):
        kernels.side_step(x, _g(2, 2047), w, 1e-5, gate, _g(2, 64), proj, w, 1e-5)
    with pytest.raises(kernels.KernelError):
        kernels.side_step(x, _g(2, 2048), w, 1e-5, gate, _g(2, 64), proj, w, 1e-5, next_weight=w)
