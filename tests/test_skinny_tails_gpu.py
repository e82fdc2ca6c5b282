"""What the few-rows product does behind its sums: activations, and several products in one launch."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _randn(seed, *shape):
    g = torch.Generator(device=DEV).manual_seed(seed)
    return torch.randn(*shape, generator=g, device=DEV).bfloat16()


@pytest.mark.parametrize("kind", ["gelu", "gelu_tanh", "relu2", "silu"])
@pytest.mark.parametrize("m,n,k", [(1, 24, 64), (4, 64, 2048), (16, 1000, 136), (3, 10256, 256), (16, 10240, 4096)])
def test_activation_in_the_product_has_the_bits_of_its_kernel(m, n, k, kind):
    """One tile and many, k that ends inside a chunk, the kernel that holds its rows (640 tiles and more), side rows that
    are part of a wider table."""
    from transformer_amd import kernels as K
    a, w = _randn(1, m, k), _randn(2, n, k)
    table = _randn(3, m, n + 40).float()
    for side in (None, table[:, 8:8 + n]):
        for dtype in (torch.bfloat16, torch.float32):
            want = K.gemm_skinny(a, w, torch.empty(m, n, dtype=dtype, device=DEV))
            K.activation(want, want, kind, side=side)
            got = K.gemm_skinny_act(a, w, torch.full((m, n), float("nan"), dtype=dtype, device=DEV), kind, side)
            assert torch.equal(got, want)


@pytest.mark.parametrize("kind", ["gelu_tanh", "silu"])
@pytest.mark.parametrize("m,n,k", [(1, 24, 64), (8, 1000, 136), (16, 14336, 4096)])
def test_gated_activation_in_the_product_has_the_bits_of_its_kernel(m, n, k, kind):
    from transformer_amd import kernels as K
    a, w = _randn(4, m, k), _randn(5, 2 * n, k)
    parts = [K.gemm_skinny(a, w[i * n:(i + 1) * n], torch.empty(m, n, dtype=torch.bfloat16, device=DEV)) for i in range(2)]
    want = K.glu(torch.cat(parts, 1), torch.empty(m, n, dtype=torch.bfloat16, device=DEV), kind)
    got = K.gemm_skinny_act(a, w, torch.empty(m, n, dtype=torch.bfloat16, device=DEV), kind, glu=True)
    # the halves' sums are cut among as many waves as their own shape says: a rounding apart at most
    assert float((got.float() - want.float()).abs().max()) <= 2 ** -7 * float(want.float().abs().max())
    assert float((got.float() - want.float()).norm()) <= 2 ** -8 * float(want.float().norm())


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("count,m,n,k", [(1, 1, 16, 8), (4, 4, 2048, 2048), (3, 16, 40, 200), (5, 7, 100, 1000)])
def test_products_in_one_launch_have_the_bits_of_their_own(count, m, n, k, dtype):
    from transformer_amd import kernels as K
    a, w = _randn(6, count + 1, m, k)[:count], _randn(7, count, n, k)
    out = torch.full((count, m, n), float("nan"), dtype=dtype, device=DEV)
    K.gemm_skinny_many(a, w, out)
    for i in range(count):
        assert torch.equal(out[i], K.gemm_skinny(a[i], w[i], torch.empty(m, n, dtype=dtype, device=DEV)))


def test_shapes_that_do_not_fit_are_refused():
    from transformer_amd import kernels as K
    a, w = _randn(8, 4, 64), _randn(9, 32, 64)
    out = torch.empty(4, 32, dtype=torch.bfloat16, device=DEV)
    for call in (lambda: K.gemm_skinny_act(a, w, out[:, :31], "silu"), lambda: K.gemm_skinny_act(a, w, out, "tanh"),
                 lambda: K.gemm_skinny_act(a, w, out, "relu2", glu=True),
                 lambda: K.gemm_skinny_act(a, w, out, "silu", side=torch.zeros(4, 31, device=DEV)),
                 lambda: K.gemm_skinny_many(a.view(1, 4, 64), w.view(2, 16, 64), out.view(1, 4, 32)),
                 lambda: K.gemm_skinny_many(_randn(1, 1, 17, 64), w.view(1, 32, 64), torch.empty(1, 17, 32, device=DEV))):
        with pytest.raises(K.KernelError):
            call()


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("n", [4096, 4097, 5120, 5121, 6143, 6144, 7168, 7169])
@pytest.mark.parametrize("m,k", [(1, 128), (16, 4096), (5, 1000)])
def test_a_workgroup_a_cu_has_the_bits_of_tiles_of_16(m, k, n, dtype):
    """20, 24 and 28 columns a workgroup, the last one part of one; with a bias, behind a norm, with an activation."""
    from transformer_amd import kernels as K
    a, w, bias = _randn(10, m, k), _randn(11, n, k), _randn(12, n).float()
    parts = torch.rand(-(-k // 16), 16, generator=torch.Generator(device=DEV).manual_seed(13), device=DEV)
    scale = K.RowScale(parts, 1e-5, k)
    for more in ({}, {"bias": bias}, {"scale": scale}, {"bias": bias, "scale": scale}):
        want = K.gemm_skinny(a, w, torch.empty(m, n, dtype=dtype, device=DEV), waves=4, **more)
        got = torch.full((m, n + 8), 7.0, dtype=dtype, device=DEV)
        K.gemm_skinny(a, w, got[:, :n], **more)
        assert torch.equal(got[:, :n], want) and (got[:, n:] == 7).all()
    want = K.activation(K.gemm_skinny(a, w, torch.empty(m, n, dtype=dtype, device=DEV), waves=4), want, "relu2")
    assert torch.equal(K.gemm_skinny_act(a, w, torch.empty(m, n, dtype=dtype, device=DEV), "relu2"), want)


@pytest.mark.parametrize("count,m,n,k", [(2, 16, 10240, 256), (3, 4, 10250, 2048), (2, 1, 10233, 4096), (2, 9, 10240, 4104)])
def test_wide_products_in_one_call_have_the_bits_of_their_own(count, m, n, k):
    """640 tiles of columns and more: each goes to the kernel that holds its rows, as it would alone; a k that it does not hold."""
    from transformer_amd import kernels as K
    a, w = _randn(14, count + 1, m, k)[:count], _randn(15, count, n, k)
    out = torch.full((count, m, n + 8), 7.0, dtype=torch.bfloat16, device=DEV)
    K.gemm_skinny_many(a, w, out[:, :, :n])
    for i in range(count):
        assert torch.equal(out[i, :, :n], K.gemm_skinny(a[i], w[i], torch.empty(m, n, dtype=torch.bfloat16, device=DEV)))
    assert (out[:, :, n:] == 7).all()
