"""Chooses next tokens on the GPU from float32 logits.

The reference draws one unseeded random number per logits row and hands it to
its sampling operator together with (temperature, top_p, top_k)
(tensor/src/operators/random_sample.rs:64-75). Here the number
comes from a counter-based generator keyed by (seed, sequence number, tokens
generated so far), so a sequence draws the same numbers whatever batch it is in
and a run can be repeated.
"""
from __future__ import annotations

from typing import Sequence

import numpy as np
import torch

from .. import kernels
from .args import SampleArgs

_M64 = (1 << 64) - 1


def uniform(seed: int, sequence: int, drawn: int) -> float:
    """u in [0, 1) with 24 random bits: a splitmix64 finaliser over the three keys."""
    z = (seed * 0x9E3779B97F4A7C15 + sequence * 0xBF58476D1CE4E5B9
         + drawn * 0x94D049BB133111EB + 0x2545F4914F6CDD1D) & _M64
    z = ((z ^ (z >> 30)) * 0xBF58476D1CE4E5B9) & _M64
    z = ((z ^ (z >> 27)) * 0x94D049BB133111EB) & _M64
    z ^= z >> 31
    return (z >> 40) / float(1 << 24)


class _Buffers:
    """What a choice works in. The kernel that draws the tokens stores them straight into ``host``, which torch's pool of
    pinned memory does not hear of: the block may go back to it, for anyone to take, only behind that kernel."""

    def __init__(self, rows: int, device):
        self.rows = rows
        self.device = torch.empty(rows, dtype=torch.int32, device=device)
        self.uniform = torch.empty(rows, dtype=torch.float32, device=device)
        self.uniform_host = torch.empty(rows, dtype=torch.float32, pin_memory=True)
        self.host = torch.empty(rows, dtype=torch.int32, pin_memory=True)
        self.scratch = None
        self._views = (0, None)
        self._last = {}             # the last use on each stream

    def first(self, n: int):
        """The first n places of device, uniform and host; three slices cost 2.7 us, so the last n's are at hand."""
        if self._views[0] != n:
            self._views = (n, (self.device[:n], self.uniform[:n], self.host[:n]))
        return self._views[1]

    def used(self):
        """Marks the work that the current stream has been given so far as the last to touch these buffers."""
        # with the device's number a stream object costs 1 us less than without
        here = torch._C._cuda_getDevice() if torch.cuda.is_initialized() else None
        stream, event = torch.cuda.current_stream(here), torch.cuda.Event()
        event.record(stream)
        self._last[stream.cuda_stream] = event
        return event

    def __del__(self):
        for event in getattr(self, "_last", {}).values():
            event.synchronize()


class Chosen:
    """Tokens that the GPU has been asked to choose: ``device`` holds them (int32) as soon as
    the stream gets there; ``result()`` waits for their copy to the host."""

    def __init__(self, device: torch.Tensor, host: torch.Tensor, buffers: _Buffers):
        self.device, self._host, self._buffers, self._event = device, host, buffers, buffers.used()

    def result(self):
        self._event.synchronize()
        return self._host.tolist()


class Sampler:
    RING = 4        # choices that may be outstanding before a buffer is used again

    def __init__(self, args: SampleArgs = SampleArgs(), seed: int = 0, device="cuda:0"):
        self.args, self.seed, self.device = args, int(seed), torch.device(device)
        self._ring = [None] * self.RING
        self._turn = 0

    def _buffers(self, n: int) -> _Buffers:
        i = self._turn
        self._turn = (i + 1) % self.RING
        b = self._ring[i]
        if b is None or b.rows < n:
            b = self._ring[i] = _Buffers(max(64, n), self.device)
        return b

    def choose_async(self, logits: torch.Tensor, sequences: Sequence[int], drawn: Sequence[int]) -> Chosen:
        """logits: float32 [n, vocab] on the GPU. sequences[i], drawn[i]: the keys of
        row i's random number. Nothing here waits for the GPU, but for a choice of more rows than a buffer has
        room for while the one that it replaces is still in flight."""
        n = logits.shape[0]
        b = self._buffers(n)
        out, u_dev, out_host = b.first(n)
        if self.args.greedy:
            kernels.argmax(logits, out)
            out_host.copy_(out, non_blocking=True)
        else:
            u = [uniform(self.seed, s, d) for s, d in zip(sequences, drawn)]
            k = self.args.top_k if self.args.top_k is not None else logits.shape[1]
            need = kernels.sample_scratch(n, logits.shape[1], int(k), float(self.args.top_p))
            if need and (b.scratch is None or b.scratch.numel() < need):
                b.scratch = torch.empty(need, dtype=torch.uint8, device=self.device)
            if need and len(u) == n <= kernels.SAMPLE_GIVEN_ROWS and logits.data_ptr() % 16 == 0 \
                    and logits.stride(0) % 4 == 0:
                # the numbers go with the launch, the tokens come back from the kernel that draws them
                kernels.sample_given(logits, u, u_dev, out, out_host, float(self.args.temperature), int(k),
                                     float(self.args.top_p), b.scratch)
            else:
                u_host = b.uniform_host[:n]
                u_host.numpy()[:] = np.asarray(u, dtype=np.float32)
                u_dev.copy_(u_host, non_blocking=True)
                kernels.sample(logits, u_dev, out, float(self.args.temperature), int(k),
                               float(self.args.top_p), b.scratch if need else None)
                out_host.copy_(out, non_blocking=True)
        return Chosen(out, out_host, b)

    def choose(self, logits: torch.Tensor, sequences: Sequence[int], drawn: Sequence[int]):
        """As ``choose_async``, returning the chosen tokens as a list of ints."""
        return self.choose_async(logits, sequences, drawn).result()
