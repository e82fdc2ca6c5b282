"""The float32 gated feed-forward of many rows in one kernel: the bits of product and activation in turn, at the edges of its tiles of 256 rows and
64 channels, for k of whole segments and not, where rows and results do not start on 16 bytes, and for sums that are not finite."""
import pytest
import torch

from transformer_amd import kernels

pytestmark = pytest.mark.gpu


def _draw(m, n, k):
    g = torch.Generator(device="cuda").manual_seed(m + 7 * n + 31 * k)
    return torch.randn(m, k, generator=g, device="cuda"), torch.randn(2 * n, k, generator=g, device="cuda") * k ** -.5, \
        torch.randn(2 * n, generator=g, device="cuda")


def _in_turn(a, w, bias):
    gu = kernels.gemm_simple(a, w, torch.empty(a.shape[0], w.shape[0], device="cuda"))
    return kernels.swiglu(gu, torch.empty(a.shape[0], w.shape[0] // 2, device="cuda"), bias)


@pytest.mark.parametrize("m,n,k", [(1021, 8192, 2048), (513, 8193, 520), (769, 8190, 1292), (1021, 8188, 512), (500, 16383, 264), (3000, 8192, 256)])
def test_the_bits_of_product_and_activation(m, n, k):
    a, w, bias = _draw(m, n, k)
    assert kernels.split_glu_takes(a, w)
    for b in (None, bias):
        want = _in_turn(a, w, b)
        for shift, width in ((0, n), (1, n + 3), (4, (n + 11) // 4 * 4)):
            room = torch.full((m + 1, width + 4), 7.0, device="cuda")
            got = kernels.gemm_split_glu(a, w, room[:m, shift:shift + n], b)
            assert torch.equal(got, want)
            assert bool((room[:, :shift] == 7).all()) and bool((room[:, shift + n:] == 7).all()) and bool((room[m] == 7).all())


def test_what_is_not_finite():
    a, w, bias = _draw(1021, 8192, 512)
    a[0, 7], a[1, 9], a[2, 100], a[700] = float("inf"), float("nan"), 3.4e38, 0.0
    w[11, 7], w[8192 + 12, 7] = 0.0, 0.0         # infinity times zero, in a gate and in an up
    w[17, 55], w[8192 + 18, 55] = -float("inf"), float("inf")
    w[19, 3], w[8192 + 20, 3] = 3e38, 3e38
    for b in (None, bias):
        want, got = _in_turn(a, w, b), kernels.gemm_split_glu(a, w, torch.empty(1021, 8192, device="cuda"), b)
        assert bool(want.isnan().any()) and bool(want.isinf().any())
        assert torch.equal(got.isnan(), want.isnan()) and torch.equal(got.nan_to_num(nan=0.0), want.nan_to_num(nan=0.0))


def test_who_takes_it_and_what_it_refuses():
    a, w, _ = _draw(1021, 8192, 512)
    out = torch.empty(1021, 8192, device="cuda")
    assert not kernels.split_glu_takes(a[:16], w) and not kernels.split_glu_takes(a[:, 1:], w[:, 1:]) and not kernels.split_glu_takes(a[:, :130], w[:, :130]) \
        and not kernels.split_glu_takes(a.bfloat16(), w.bfloat16())
    for args in ((a[:16], w, out[:16]), (a, w, out[:, :8000]), (a[:1000], w, out), (a[:, 2:], w[:, 2:], out)):
        with pytest.raises(kernels.KernelError):
            kernels.gemm_split_glu(*args)
