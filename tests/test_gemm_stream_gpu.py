"""float32 products of up to 8 rows whose weight streams through LDS: the bits of the product, the norm and the
activation that they stand for, at the edges of segments, tiles and rounds."""
import pytest
import torch

from transformer_amd import kernels

pytestmark = pytest.mark.gpu

# (n, k): whole segments and k that ends inside a segment, a block or a round; fewer tiles than workgroups, one more
# than a round of them, a last tile of 1 to 7 columns
SHAPES = [(2048, 2048), (8, 1536), (1, 1540), (4097, 2048), (4101, 1996), (2050, 2052), (259, 4096), (2300, 4092), (2056, 3000),
          (16, 4100), (2048, 8192), (2057, 8196), (65, 6164), (2, 12292), (40, 16384)]


def _draw(m, n, k, seed=0):
    g = torch.Generator(device="cuda").manual_seed(seed + 31 * m + n + 7 * k)
    a = torch.randn(m, k, generator=g, device="cuda")
    w = torch.randn(n, k, generator=g, device="cuda") / k ** 0.5
    return a, w, g


def _plain(a, w):
    """Rows of one more than the kernel takes: another kernel, with the bits that every row has by itself."""
    more = torch.cat([a, a.new_zeros(9, a.shape[1])])
    return kernels.gemm_simple(more, w, torch.empty(more.shape[0], w.shape[0], device="cuda"))[:a.shape[0]]


@pytest.mark.parametrize("n,k", SHAPES)
@pytest.mark.parametrize("m", [1, 2, 3, 4, 5, 8])
def test_rows_have_the_bits_of_the_other_kernels(m, n, k):
    a, w, g = _draw(m, n, k)
    want = _plain(a, w)
    room = torch.full((m + 1, n), 7.0, device="cuda")
    got = kernels._gemm_stream("test", a, w, room[:m])
    assert torch.equal(got, want) and bool((room[m] == 7.0).all())
    bias = torch.randn(n, generator=g, device="cuda")
    assert torch.equal(kernels._gemm_stream("test", a, w, torch.empty_like(want), bias), want + bias)
    x = torch.randn(m, n, generator=g, device="cuda")
    assert torch.equal(kernels._gemm_stream("test", a, w, x.clone(), add=True), x + want)
    exact = a.double() @ w.double().t()
    # a chain of at most 256 fused multiply-adds and k / 256 additions, each half an ulp of what it reaches
    bound = (256 + k / 256) * 2.0 ** -24 * (a.double().abs() @ w.double().abs().t())
    assert bool(((got.double() - exact).abs() <= bound).all())


@pytest.mark.parametrize("n,k", [s for s in SHAPES if s[1] <= 4096])
@pytest.mark.parametrize("m", [1, 3, 8])
def test_norm_and_gates_have_the_bits_of_their_kernels(m, n, k):
    x, w, g = _draw(m, 2 * n, k, 5)
    gain = torch.randn(k, generator=g, device="cuda")
    h = kernels.add_rmsnorm(x.clone(), gain, 1e-5, torch.empty_like(x))
    norm = kernels.RowNorm(x, gain, 1e-5)
    gu = _plain(h, w)
    assert torch.equal(kernels.gemm_normed(norm, w, torch.empty_like(gu)), gu)
    bias = torch.randn(2 * n, generator=g, device="cuda")
    want = kernels.swiglu(gu + bias, torch.empty(m, n, device="cuda"))
    assert torch.equal(kernels.gemm_normed(norm, w, torch.empty_like(want), bias, glu=True), want)
    assert torch.equal(kernels._gemm_stream("test", h, w, torch.empty_like(want), bias, glu=True), want)


def test_rows_of_wider_buffers_and_what_it_refuses():
    a, w, _ = _draw(4, 300, 2048)
    wide = torch.zeros(4, 4096, device="cuda")
    wide[:, 4:2052] = a
    out = torch.full((4, 512), 3.0, device="cuda")
    kernels._gemm_stream("test", wide[:, 4:2052], w, out[:, 8:308])
    assert torch.equal(out[:, 8:308], _plain(a, w)) and bool((out[:, :8] == 3.0).all()) and bool((out[:, 308:] == 3.0).all())
    with pytest.raises(kernels.KernelError):       # rows that do not start on 16 bytes
        kernels._gemm_stream("test", wide[:, 1:2049], w, torch.empty(4, 300, device="cuda"))
    with pytest.raises(kernels.KernelError):       # nine rows
        kernels._gemm_stream("test", torch.zeros(9, 2048, device="cuda"), w, torch.empty(9, 300, device="cuda"))
    assert not kernels.add_takes(9, w) and not kernels.normed_takes(9, w) and not kernels.normed_takes(4, w[:, 1:])
