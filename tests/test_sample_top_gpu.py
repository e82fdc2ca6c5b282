"""Cuts at few tokens in two kernels: the tokens that the kernel that walks a row token by token chooses."""
import numpy as np
import pytest
import torch

from transformer_amd import kernels

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _rows(vocab):
    """Rows whose threshold falls on the edges: of steps of logit / T, of a part's tokens handed on, of the interval in which
    the row's mass is known before it is added up."""
    g = np.random.default_rng(vocab)
    l = (g.normal(size=(20, vocab)) * 2.5).astype(np.float32)
    l[1] = np.round(l[1] * 16) / 16                            # equal logits on the steps' edges
    l[2, ::7] = 9.0                                            # equals in every part, more than a part hands on
    l[3] = -3.0
    l[4, :4000] = -np.inf                                      # parts of nothing, or nearly
    l[5] = -np.inf
    l[5, vocab - 1] = 1.5
    l[6] *= 40                                                 # few tokens within 16 units of a part's largest
    l[7] *= 0.01
    l[8] += 1e4
    l[9, -3:] = 20.0
    l[10] = -np.inf
    l[10, 5:vocab:vocab // 8] = 2.0                            # eight or nine equals and nothing else: shares of exactly 1/8
    l[11] = -np.inf
    l[11, :64] = np.log(0.5) * np.arange(64)                   # running sums that meet 1/2, 3/4, ... of the row's mass
    l[12, g.permutation(vocab)[:300]] = 7.0                    # ties across parts, ranked by index
    l[13, :4096] += 30.0                                       # one part holds all
    return l


@pytest.mark.parametrize("vocab", [200, 4095, 4097, 8192, 40963, 65536])
@pytest.mark.parametrize("k", [1, 7, 31, 128])
def test_the_same_tokens_as_by_walking(vocab, k):
    l = _rows(vocab)
    n = len(l)
    ld = (vocab + 11) // 4 * 4
    aligned = torch.zeros(n, ld, device=DEV)[:, 4:4 + vocab]
    shifted = torch.zeros(n, ld, device=DEV)[:, 1:1 + vocab]
    for t in (aligned, shifted):
        t.copy_(torch.from_numpy(l))
    need = kernels.sample_scratch(n, vocab, k, 0.9)
    assert need > 0
    scratch = torch.full((need,), 255, dtype=torch.uint8, device=DEV)
    a, b = (torch.empty(n, dtype=torch.int32, device=DEV) for _ in range(2))
    for i, (T, p) in enumerate(((1.0, 1.0), (0.8, 0.95), (1.0, 0.5), (1.0, 0.875), (0.05, 0.99), (30.0, 0.3), (2.0, 0.9999), (1.0, 0.0))):
        u = torch.rand(n, generator=torch.Generator().manual_seed(i)).to(DEV)
        u[:2] = torch.tensor([0.0, 1.0 - 2.0 ** -24])
        kernels.sample(aligned, u, a, T, k, p, scratch)
        kernels.sample(shifted, u, b, T, k, p)
        assert torch.equal(a, b), (T, p, (a != b).nonzero().flatten().tolist())


@pytest.mark.parametrize("n,vocab,k", [(64, 200000, 40), (3, 209000, 40), (2, 300000, 6), (1, 1048576, 8)])
def test_many_parts(n, vocab, k):
    """More parts than a wave has lanes, rows in turns, and as many handed-on tokens as there is room for."""
    g = torch.Generator(device=DEV).manual_seed(n)
    logits = torch.randn(n, vocab + 4, generator=g, device=DEV) * 2.0
    u = torch.rand(n, generator=g, device=DEV)
    a, b = (torch.empty(n, dtype=torch.int32, device=DEV) for _ in range(2))
    scratch = torch.empty(kernels.sample_scratch(n, vocab, k, 0.9), dtype=torch.uint8, device=DEV)
    kernels.sample(logits[:, :vocab], u, a, 0.9, k, 0.9, scratch)
    shifted = torch.empty(n, vocab + 4, device=DEV)[:, 1:1 + vocab]
    shifted.copy_(logits[:, :vocab])
    kernels.sample(shifted, u, b, 0.9, k, 0.9)
    assert torch.equal(a, b)


def _flat(vocab):
    """Rows whose tokens lie within a few steps of each other, down to the pieces that a step is cut into."""
    g = np.random.default_rng(vocab)
    z = g.normal(size=(16, vocab))
    l = np.empty((16, vocab), np.float32)
    for i, sd in enumerate((0.1, 0.07, 0.05, 0.03, 0.01, 0.003, 0.001, 0.0003, 1e-4, 1e-7)):
        l[i] = z[i] * sd + 0.3 * (i - 4)
    l[10] = np.round(z[10] * 40) / 4096                        # equals on the pieces' edges
    l[11] = 1000 + z[11] * 0.05                                # few values to a piece
    l[12] = 3e5 + z[12] * 0.05                                 # a value a step: no pieces
    l[13] = z[13] * 0.05
    l[13, :4096] *= 100                                        # one part's tokens spread, the others' not
    l[14] = z[14] * 0.05
    l[14, ::2] = -np.inf
    l[15] = z[15] * 0.05
    l[15, g.permutation(vocab)[:20]] += 18.0                   # the threshold 16 units below the largest
    return l


@pytest.mark.parametrize("vocab,k", [(200, 7), (4097, 128), (32000, 50), (32000, 128), (65536, 128), (128256, 40), (128256, 64), (300000, 6)])
def test_flat_rows(vocab, k):
    l = _flat(vocab)
    n, ld = len(l), (vocab + 11) // 4 * 4
    aligned = torch.zeros(n, ld, device=DEV)[:, 4:4 + vocab]
    shifted = torch.zeros(n, ld, device=DEV)[:, 1:1 + vocab]
    for t in (aligned, shifted):
        t.copy_(torch.from_numpy(l))
    scratch = torch.full((kernels.sample_scratch(n, vocab, k, 0.9),), 255, dtype=torch.uint8, device=DEV)
    a, b = (torch.empty(n, dtype=torch.int32, device=DEV) for _ in range(2))
    for i, (T, p) in enumerate(((1.0, 1.0), (1.0, 0.95), (0.7, 0.5), (8.0, 0.9), (0.05, 0.99), (1.0, 1e-4))):
        u = torch.rand(n, generator=torch.Generator().manual_seed(i)).to(DEV)
        kernels.sample(aligned, u, a, T, k, p, scratch)
        kernels.sample(shifted, u, b, T, k, p)
        assert torch.equal(a, b), (T, p, (a != b).nonzero().flatten().tolist())


@pytest.mark.parametrize("sd", [0.08, 0.05, 0.03])
def test_flat_rows_stay_in_parts(sd):
    """Rows that are given back to one workgroup each take eight times as long as others (216 us and 26)."""
    n, vocab, k = 8, 128256, 64
    g = torch.Generator(device=DEV).manual_seed(3)
    z = torch.randn(n, vocab, generator=g, device=DEV)
    u, out = torch.rand(n, generator=g, device=DEV), torch.empty(n, dtype=torch.int32, device=DEV)
    scratch = torch.empty(kernels.sample_scratch(n, vocab, k, 0.95), dtype=torch.uint8, device=DEV)

    def us(logits):
        best = float("inf")
        for _ in range(6):
            a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            a.record()
            for _ in range(10):
                kernels.sample(logits, u, out, 1.0, k, 0.95, scratch)
            b.record()
            b.synchronize()
            best = min(best, a.elapsed_time(b))
        return best

    assert us(z * sd) < 3 * us(z * 2.5)
