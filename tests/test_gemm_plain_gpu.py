"""The float32 product of many bfloat16 rows: at the edges of its tiles of 256 and 128 rows and 256 columns, for odd and even numbers of steps of
64 k, stored and added, against 64 bits; and through ``linear`` and ``linear_delta`` where its rule takes it."""
import pytest
import torch

from transformer_amd import kernels
from transformer_amd.parts.linear import Workspace, linear, linear_delta

pytestmark = pytest.mark.gpu


def _g(*shape, seed=0, scale=1.0, dtype=torch.bfloat16):
    gen = torch.Generator(device="cuda").manual_seed(seed)
    return (torch.randn(*shape, generator=gen, device="cuda") * scale).to(dtype)


def _close(got, a, w, x=None):
    # exact products; a chain of at most k additions, each rounded to 24 bits of a partial sum below sum |a w|, and one to the stream
    want, size = a.double() @ w.double().t(), a.double().abs() @ w.double().abs().t()
    if x is not None:
        want, size = want + x.double(), size + x.double().abs()
    assert bool(((got.double() - want).abs() <= a.shape[1] * 2.0 ** -24 * size).all())


# a single row; one over and under a half and a whole tile; whole rounds of the CUs, a last round of up to half as many tiles, and of more
@pytest.mark.parametrize("m,n,k", [(1, 256, 64), (127, 512, 128), (129, 256, 192), (256, 256, 320), (257, 768, 64), (385, 256, 448), (1025, 8192, 128),
                                   (1281, 16384, 64), (2011, 4096, 192), (4097, 4096, 64)])
def test_tiles_and_steps(m, n, k):
    a, w, x = _g(m, k, seed=1), _g(n, k, seed=2), _g(m, n, seed=3, dtype=torch.float32)
    room = torch.full((m + 1, n + 8), 7.0, device="cuda")
    got = kernels.gemm_plain(a, w, room[:m, 4:n + 4])
    assert bool((room[:, :4] == 7).all()) and bool((room[:, n + 4:] == 7).all()) and bool((room[m] == 7).all())
    _close(got, a, w)
    added = kernels.gemm_plain(a, w, x.clone(), add=True)
    assert torch.equal(added, x + got)
    rows = sorted({0, m // 2, max(0, m - 130), m - 1})       # another number of rows: other tiles, the same bits
    assert torch.equal(kernels.gemm_plain(a[rows].contiguous(), w, torch.empty(len(rows), n, device="cuda")), got[rows])


@pytest.mark.parametrize("m,n,k", [(1600, 4096, 14336), (3164, 4096, 4096)])
def test_where_the_rule_takes_it(m, n, k):
    a, w, x = _g(m, k, seed=1), _g(n, k, seed=2, scale=k ** -.5), _g(m, n, seed=3, dtype=torch.float32)
    got = linear(a, w, torch.empty(m, n, device="cuda"))
    assert kernels.plain_pays(a, w, got)
    _close(got, a, w)
    into = x.clone()
    linear_delta(a, w, Workspace("cuda"), "delta", into=into)
    assert torch.equal(into, x + got)


def test_who_takes_it_and_what_it_refuses():
    a, w, out = _g(3164, 4096), _g(4096, 4096), torch.empty(3164, 4096, device="cuda")
    assert kernels.plain_pays(a, w, out) and not kernels.plain_pays(a, w, out.bfloat16()) and not kernels.plain_pays(a[:500], w, out[:500]) \
        and not kernels.plain_pays(a[:2300], w, out[:2300]) and not kernels.plain_pays(a.float(), w, out) and not kernels.plain_pays(a, w[:4000], out[:, :4000])
    for args in ((a[:, :1000], w[:, :1000], out), (a, w[:4000], out[:, :4000]), (a, w, out[:, :4090]), (a[:3000], w, out)):
        with pytest.raises(kernels.KernelError):
            kernels.gemm_plain(*args)
