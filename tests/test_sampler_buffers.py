"""How long a choice's host memory lives: the kernel that draws the tokens stores them there, and torch's pool of pinned
memory does not know. No GPU: kernels, events and streams are stand-ins that note what happens in which order."""
import gc
import weakref

import pytest
import torch

import transformer_amd as ta
from transformer_amd.sampling import sampler as sampling


class Event:
    def __init__(self):
        self.passed = False

    def record(self, stream=None):
        pass

    def synchronize(self):
        self.passed = True


@pytest.fixture
def world(monkeypatch):
    """Sampler's surroundings; ``freed``: for every pinned block that has gone, whether each event had passed by then."""
    events, freed, real = [], [], torch.empty

    class Stream:
        cuda_stream = 0

    def make_event(*a, **k):
        events.append(Event())
        return events[-1]

    def empty(*shape, pin_memory=False, device=None, **k):
        t = real(*shape, **k)
        if pin_memory:
            weakref.finalize(t, lambda: freed.append([e.passed for e in events]))
        return t

    monkeypatch.setattr(torch, "empty", empty)
    monkeypatch.setattr(torch.cuda, "Event", make_event)
    monkeypatch.setattr(torch.cuda, "current_stream", lambda *a: Stream())
    monkeypatch.setattr(sampling.kernels, "sample_scratch", lambda *a: 16)
    monkeypatch.setattr(sampling.kernels, "sample_given", lambda *a: None)
    monkeypatch.setattr(sampling.kernels, "sample", lambda *a: None)
    return events, freed


def _sampler():
    return sampling.Sampler(ta.SampleArgs(0.8, 0.95, 40), device="cpu")


@pytest.mark.parametrize("first", ["sampler", "choice"])
def test_a_choice_that_nobody_reads_is_waited_for(world, first):
    events, freed = world
    s = _sampler()
    c = s.choose_async(torch.zeros(4, 512), range(4), [0] * 4)
    assert not events[-1].passed
    if first == "sampler":
        del s, c
    else:
        del c
        del s
    gc.collect()
    assert len(freed) == 2 and all(all(passed) for passed in freed)


def test_a_buffer_replaced_by_a_larger_one_is_waited_for(world):
    events, freed = world
    s = _sampler()
    for _ in range(s.RING):
        s.choose_async(torch.zeros(4, 512), range(4), [0] * 4)
    assert not any(e.passed for e in events)
    first = events[0]
    s.choose_async(torch.zeros(65, 512), range(65), [0] * 65)
    gc.collect()
    assert first.passed and len(freed) == 2 and all(passed[0] for passed in freed)
    assert not any(e.passed for e in events[1:])                 # the others are not waited for


def test_a_choice_keeps_its_buffer_when_the_sampler_goes(world):
    events, freed = world
    s = _sampler()
    c = s.choose_async(torch.zeros(4, 512), range(4), [0] * 4)
    del s
    gc.collect()
    assert not freed and not events[0].passed
    assert len(c.result()) == 4 and events[0].passed
