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
