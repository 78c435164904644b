"""Sampling one token per row of logits on the GPU.

Strategy per row as in pico_vllm/sampler.py:40-88 (greedy / temperature /
temperature with top-p), but in one call with per-row parameters for the whole
batch (a short chain of launches, several workgroups a row) instead of torch
calls per group of equal parameters.  Randomness comes from
a counter-based generator on the host (``uniform`` here; the launch makes the same numbers in
native code): the uniform number of a draw depends
only on (seed, index of the token in its request), so a request samples the
same tokens whatever else is in the batch.
"""
from __future__ import annotations

import weakref
from typing import List, Sequence

import torch

from ..ops import kernels

_MASK = (1 << 64) - 1
POLL_US = 2000


def _splitmix64(x: int) -> int:
    x = (x + 0x9E3779B97F4A7C15) & _MASK
    z = x
    z = ((z ^ (z >> 30)) * 0xBF58476D1CE4E5B9) & _MASK
    z = ((z ^ (z >> 27)) * 0x94D049BB133111EB) & _MASK
    return z ^ (z >> 31)


def uniform(seed: int, index: int) -> float:
    """A number in [0, 1) with 24 random bits, a pure function of (seed, index): the generator in its plain form, which launches make
    natively (``kernels.sample_uniforms``) and tests hold them to."""
    z = _splitmix64(_splitmix64(seed & _MASK) ^ ((index * 0xD6E8FEB86659FD93) & _MASK))
    return (z >> 40) / float(1 << 24)


def _outlive(landing, landed) -> None:
    """The host memory ``landing`` is held until what writes there is done."""
    for event in landed:
        if event is not None:
            event.synchronize()


class Sampler:
    def __init__(self, device: torch.device, max_rows: int):
        self.device = device
        self.max_rows = max_rows
        self._options = kernels.SampleOptions(max_rows)
        self._dev = torch.zeros(3, max_rows, dtype=torch.float32, device=device)
        self._out = torch.zeros(max_rows, dtype=torch.int32, device=device)
        self._argmax_work = kernels.argmax_workspace(max_rows, device) if torch.cuda.is_available() else None
        # of calls without top_p; what its search needs (as much as the logits of 256 rows) waits for the first call that has it
        self._sample_work = kernels.sample_workspace(max_rows, device, top_p_rows=False) if torch.cuda.is_available() else None
        self._top_p_work = None
        # two sets, used in turn: a step's tokens may be read after the next step was launched.  The last launch writes them there itself,
        # a word a row: the launch's stamp above the token, so that words of a launch that nobody read are not taken for another's
        self._landing = [torch.zeros(max_rows, dtype=torch.int64, pin_memory=torch.cuda.is_available()) for _ in range(2)]
        self._stamps, self._stamp = [0, 0], 1
        self._tokens = [torch.zeros(max_rows, dtype=torch.int32) for _ in range(2)]
        self._landing_at = [kernels.host_on_device(t) if torch.cuda.is_available() and max_rows else 0 for t in self._landing]
        self._landed = [torch.cuda.Event() if torch.cuda.is_available() else None for _ in range(2)]
        self._turn = 0
        # a launch that is never read still writes there
        weakref.finalize(self, _outlive, self._landing, self._landed).atexit = False

    def _work(self, vocab: int) -> torch.Tensor:
        """The workspace of a search, kept: all rows that the sampler was made for, of as many logits as have been seen."""
        if self._top_p_work is None or vocab > self._top_p_work[0]:
            self._top_p_work = None                          # (the smaller one goes first)
            self._top_p_work = (vocab, kernels.sample_workspace(self.max_rows, self.device, vocab))
        return self._top_p_work[1]

    def sample(self, logits: torch.Tensor, temperatures: Sequence[float], top_ps: Sequence[float],
               seeds: Sequence[int], indices: Sequence[int]) -> List[int]:
        """logits: float32 [R, V]; one (temperature, top_p, seed, token index) per row."""
        return self.read(self.launch(logits, temperatures, top_ps, seeds, indices))

    @property
    def device_tokens(self) -> torch.Tensor:
        """int32 [max_rows] on the device: row r holds the token of row r of the last launch."""
        return self._out

    def read(self, ticket) -> List[int]:
        """The tokens of the launch that returned ``ticket``; waits for that launch only."""
        turn, R = ticket
        if R == 0:
            return []
        if not self._landing_at[turn]:
            self._landed[turn].synchronize()
            return self._landing[turn][:R].tolist()
        # the host sees a word some 6 us before it would see the event behind it (8 rows: 48 us from call to tokens, 54 so); of a wait so
        # long that this does not count the rest is the event's
        tokens = self._tokens[turn]
        if not kernels.landed(self._landing[turn], R, self._stamps[turn], tokens, POLL_US):
            self._landed[turn].synchronize()
            if not kernels.landed(self._landing[turn], R, self._stamps[turn], tokens, POLL_US):
                raise RuntimeError("the step's tokens did not arrive")
        return tokens[:R].tolist()

    def launch(self, logits: torch.Tensor, temperatures: Sequence[float], top_ps: Sequence[float],
               seeds: Sequence[int], indices: Sequence[int]):
        """Start sampling and the copy of the tokens to the host; returns a ticket for ``read``.
        At most two launches may be unread at a time."""
        R = logits.shape[0]
        if not (len(temperatures) == len(top_ps) == len(seeds) == len(indices) == R):
            raise ValueError("one set of sampling parameters per row of logits is needed")
        if R > self.max_rows:
            raise ValueError(f"{R} rows to sample, the sampler was made for {self.max_rows}")
        if R == 0:
            return (0, 0)
        turn = self._turn
        landing, stamp = self._landing_at[turn], self._stamp
        self._stamp = stamp % 0xffffffff + 1
        self._stamps[turn] = stamp
        if not any(temperatures):
            # all rows greedy: no options, and the argmax alone spreads a row over several workgroups
            kernels.argmax(logits, self._out, self._argmax_work, landing, stamp)
        else:
            self._options.fill(temperatures, top_ps, seeds, indices)
            searched = any(t > 0 and p < 1 for t, p in zip(temperatures, top_ps))
            work = self._work(logits.shape[1]) if searched else self._sample_work
            kernels.sample_rows(logits, self._options, self._dev, self._out, work, searched, landing, stamp)
        self._turn ^= 1
        if not landing:
            self._landing[turn][:R].copy_(self._out[:R], non_blocking=True)
        self._landed[turn].record()
        return (turn, R)
