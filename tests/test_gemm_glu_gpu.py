"""The gated feed-forward of many bfloat16 rows in one kernel: at the edges of its tiles of 256 and 128 rows and 128 channels, for odd and even
numbers of steps of 64 k, against float32; a row has the same bits in either tile."""
import pytest
import torch

from transformer_amd import kernels

pytestmark = pytest.mark.gpu


def _draw(m, n, k, seed=0):
    g = torch.Generator(device="cuda").manual_seed(m + 7 * n + 31 * k + seed)
    a = torch.randn(m, k, generator=g, device="cuda").bfloat16()
    w = (torch.randn(2 * n, k, generator=g, device="cuda") / k ** 0.5).bfloat16()
    return a, w, torch.randn(2 * n, generator=g, device="cuda")


def _want(a, w, act, bias=None, limits=None):
    gu = a.double() @ w.double().t()
    if bias is not None:
        gu = gu + bias.double()
    g, u = gu.chunk(2, 1)
    if limits is not None:
        limit, slope, shift = limits
        g, u = g.clamp(max=limit), u.clamp(-limit, limit)
        return g * torch.sigmoid(slope * g) * (u + shift)
    return (torch.nn.functional.silu(g) if act == "silu" else torch.nn.functional.gelu(g, approximate="tanh")) * u


def _close(got, want):
    # one rounding to 8 bits, and float32 sums of k products: far below it where the result is not near zero
    assert bool(((got.double() - want).abs() <= 2.0 ** -8 * want.abs() + 1e-5).all())


# a single row; one row over and under a half and a whole tile; channels that end inside a tile; whole rounds and a last round of up to half as
# many tiles as CUs, of more, and one of tiles that begin behind the last row
@pytest.mark.parametrize("m,n,k", [(1, 4, 64), (127, 128, 128), (128, 132, 192), (129, 4, 320), (255, 260, 64), (257, 124, 192), (384, 128, 256), (385, 516, 128),
                                   (513, 8192, 128), (640, 11008, 192), (769, 16384, 64), (2011, 4100, 448), (1025, 14336, 128), (4400, 1028, 64)])
def test_tiles_and_steps(m, n, k):
    a, w, _ = _draw(m, n, k)
    room = torch.full((m + 1, n + 8), 7.0, device="cuda", dtype=torch.bfloat16)
    got = kernels.gemm_glu(a, w, room[:m, 4:n + 4])
    assert bool((room[:, :4] == 7).all()) and bool((room[:, n + 4:] == 7).all()) and bool((room[m] == 7).all())
    _close(got, _want(a, w, "silu"))
    rows = sorted({0, m // 2, max(0, m - 130), m - 1})       # another number of rows: other tiles, the same bits
    again = kernels.gemm_glu(a[rows].contiguous(), w, torch.empty(len(rows), n, device="cuda", dtype=torch.bfloat16))
    assert torch.equal(again, got[rows])


@pytest.mark.parametrize("act,limits", [("silu", None), ("gelu_tanh", None), ("silu", (1.5, 1.702, 1.0))])
def test_activations_biases_and_wider_rows(act, limits):
    m, n, k = 300, 500, 320
    a, w, bias = _draw(m, n, k, 1)
    wide = torch.zeros(m, k + 64, device="cuda", dtype=torch.bfloat16)
    wide[:, 8:k + 8] = a
    for b in (None, bias):
        got = kernels.gemm_glu(wide[:, 8:k + 8], w, torch.empty(m, n, device="cuda", dtype=torch.bfloat16), act, b, limits)
        _close(got, _want(a, w, act, b, limits))


def test_who_takes_it_and_what_it_refuses():
    a, w, _ = _draw(512, 8192, 2112)
    out = torch.empty(512, 8192, device="cuda", dtype=torch.bfloat16)
    assert kernels.glu_pays(a, w) and not kernels.glu_pays(a[:64], w) and not kernels.glu_pays(a[:, 4:2052], w[:, 4:2052]) \
        and not kernels.glu_pays(a[:, :2080], w[:, :2080]) and not kernels.glu_pays(a.float(), w)
    for args in ((a[:, :1000], w[:, :1000], out), (a[:, 4:964], w[:, :960], out), (a, w, out[:, :8000]), (a[:500], w, out)):
        with pytest.raises(kernels.KernelError):
            kernels.gemm_glu(*args)
    with pytest.raises(kernels.KernelError):
        kernels.gemm_glu(a, w, out, "relu2")
