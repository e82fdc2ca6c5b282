"""Choices whose random numbers travel in the launch's arguments and whose tokens the kernel writes to the host."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("n,vocab,k,p", [(1, 32000, 40, 0.95), (8, 128256, 40, 0.95), (64, 50000, 50, 1.0), (3, 30004, 7, 0.5),
                                         (5, 128256, 128256, 1.0), (2, 600000, 128, 0.9), (7, 40000, 40000, 0.8)])
def test_given_numbers_choose_as_copied_ones(n, vocab, k, p):
    """One part and many (of up to 64 and beyond), with and without cuts; a row whose threshold the parts do not enclose
    (all logits equal) goes through the whole row's walk."""
    from transformer_amd import kernels as K
    g = torch.Generator(device=DEV).manual_seed(vocab + n)
    logits = torch.randn(n, vocab, generator=g, device=DEV) * 2.5
    if n > 2:
        logits[1] = 0.25
    u = torch.rand(n, generator=torch.Generator().manual_seed(n))
    need = K.sample_scratch(n, vocab, k, p)
    assert need > 0
    scratch = torch.empty(need, dtype=torch.uint8, device=DEV)
    want = K.sample(logits, u.to(DEV), torch.empty(n, dtype=torch.int32, device=DEV), 0.8, k, p, scratch)
    out, host = torch.full((n,), -1, dtype=torch.int32, device=DEV), torch.full((n,), -1, dtype=torch.int32).pin_memory()
    K.sample_given(logits, u.tolist(), torch.empty(n, device=DEV), out, host, 0.8, k, p, scratch)
    torch.cuda.synchronize()
    assert torch.equal(out, want) and host.tolist() == want.tolist()


def test_what_given_numbers_refuse():
    from transformer_amd import kernels as K
    logits = torch.zeros(65, 32000, device=DEV)
    scratch = torch.empty(K.sample_scratch(65, 32000, 40, 0.9), dtype=torch.uint8, device=DEV)
    out, dev = torch.empty(65, dtype=torch.int32, device=DEV), torch.empty(65, device=DEV)
    pinned = torch.empty(65, dtype=torch.int32).pin_memory()
    calls = [lambda: K.sample_given(logits, [0.5] * 65, dev, out, pinned, 1.0, 40, 0.9, scratch),
             lambda: K.sample_given(logits[:4], [0.5] * 3, dev[:4], out[:4], pinned[:4], 1.0, 40, 0.9, scratch),
             lambda: K.sample_given(logits[:4], [0.5] * 4, dev[:4], out[:4], torch.empty(4, dtype=torch.int32), 1.0, 40, 0.9, scratch),
             lambda: K.sample_given(logits[:4, 1:], [0.5] * 4, dev[:4], out[:4], pinned[:4], 1.0, 40, 0.9, scratch),
             lambda: K.sample_given(logits[:4], [0.5] * 4, dev[:4], out[:4], pinned[:4], 1.0, 40, 0.9, scratch[:8])]
    for call in calls:
        with pytest.raises(K.KernelError):
            call()


@pytest.mark.parametrize("n", [1, 8, 64, 65])
def test_the_sampler_returns_the_same_tokens_on_both_sides(n):
    """64 rows go without copies, 65 with them; more choices in turn than there are buffers."""
    import transformer_amd as ta
    from transformer_amd import kernels as K
    from transformer_amd.sampling.sampler import Sampler, uniform
    g = torch.Generator(device=DEV).manual_seed(n)
    s = Sampler(ta.SampleArgs(0.7, 0.9, 30), seed=5, device=DEV)
    for turn in range(6):
        logits = torch.randn(n, 32000, generator=g, device=DEV) * 2
        got = s.choose_async(logits, range(n), [turn] * n)
        u = torch.tensor([uniform(5, i, turn) for i in range(n)], device=DEV)
        want = K.sample(logits, u, torch.empty(n, dtype=torch.int32, device=DEV), 0.7, 30, 0.9)
        assert got.result() == want.tolist() == got.device.tolist()


def test_host_tokens_stay_until_they_are_written():
    """A choice behind a few milliseconds of other work, dropped unread with its sampler: the pinned block that its kernel
    writes to may be anyone's only behind that kernel."""
    import transformer_amd as ta
    from transformer_amd.sampling.sampler import Sampler
    s = Sampler(ta.SampleArgs(0.7, 0.9, 30), seed=5, device=DEV)
    logits, big = torch.randn(8, 32000, device=DEV), torch.randn(4096, 4096, device=DEV)
    s.choose(logits, range(8), [0] * 8)
    for _ in range(3):
        s.choose_async(logits, range(8), [0] * 8)
    for _ in range(20):
        big = torch.mm(big, big).clamp_(-1, 1)
    c, done = s.choose_async(logits, range(8), [0] * 8), torch.cuda.Event()
    done.record()
    at = c._host.data_ptr()
    del s, c
    taken = [torch.empty(64, dtype=torch.int32, pin_memory=True) for _ in range(16)]
    assert done.query() or at not in [t.data_ptr() for t in taken]
    torch.cuda.synchronize()
