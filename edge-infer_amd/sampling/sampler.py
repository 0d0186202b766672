"""Draws tokens from float32 logits on the GPU (see csrc/sampling.hip).

A request's draws depend only on (seed, its stream number, its step counter), so it
samples the same tokens alone or in any batch.
"""
from __future__ import annotations

from array import array
from typing import List, Sequence

import torch

from ..csrc import lib
from .params import SamplingParams


class Sampler:
    def __init__(self, device):
        self.device = torch.device(device)
        self._tokens = torch.empty(1024, dtype=torch.int32, device=self.device)
        self._probabilities = torch.empty(1024, dtype=torch.float32, device=self.device)
        self._meta = torch.empty(2048, dtype=torch.int32, device=self.device)
        # stream numbers and counters travel through pinned memory; two buffers in turn, so
        # that filling one does not disturb a copy of the other that is still queued
        self._meta_host = [torch.empty(2048, dtype=torch.int32, pin_memory=True) for _ in range(2)]
        self._meta_turn = 0
        # tokens that go to the host are written there by the kernel that chose them
        self._tokens_host = torch.empty(1024, dtype=torch.int32, pin_memory=True)
        self._partial = None          # scratch of the greedy search over a wide vocabulary
        self._scratch = None          # zeroed scratch of sampling from a wide vocabulary
        self._last_rows = 0

    def _reserve(self, rows: int) -> None:
        if self._tokens.numel() < rows:
            self._tokens = torch.empty(rows, dtype=torch.int32, device=self.device)
            self._probabilities = torch.empty(rows, dtype=torch.float32, device=self.device)
            self._meta = torch.empty(2 * rows, dtype=torch.int32, device=self.device)
            self._meta_host = [torch.empty(2 * rows, dtype=torch.int32, pin_memory=True)
                               for _ in range(2)]
            self._tokens_host = torch.empty(rows, dtype=torch.int32, pin_memory=True)

    @staticmethod
    def _given(streams, counters):
        """The two as arrays that go with the launch; None for many rows, or where their values
        have to be looked at one by one (as a tensor of them does)."""
        if len(streams) > lib.SAMPLE_GIVEN_ROWS:
            return None
        try:
            return array("i", list(streams)), array("i", list(counters))
        except (TypeError, OverflowError):
            return None

    def sample_device(self, logits: torch.Tensor, params: SamplingParams, streams: Sequence[int],
                      counters: Sequence[int]) -> torch.Tensor:
        """int32 tokens [rows] on the device (a view that the next call overwrites)."""
        rows = logits.shape[0]
        self._reserve(rows)
        tokens = self._tokens[:rows]
        self._choose(logits, params, streams, counters, tokens)
        return tokens

    def _choose(self, logits, params, streams, counters, tokens) -> None:
        rows, vocab = logits.shape
        params.validate(vocab)
        probabilities = self._probabilities[:rows]
        if params.is_greedy(vocab):
            need = lib.argmax_partial_size(rows, vocab)
            if need and (self._partial is None or self._partial.numel() < need):
                self._partial = torch.empty(need, dtype=torch.float32, device=self.device)
            lib.argmax(logits, tokens, probabilities, self._partial if need else None)
            return
        if len(streams) != rows or len(counters) != rows:
            raise ValueError("one stream number and one counter per row are needed")
        keys = self._given(streams, counters)
        if keys is None:
            host = self._meta_host[self._meta_turn]
            self._meta_turn ^= 1
            host[:2 * rows] = torch.tensor(list(streams) + list(counters), dtype=torch.int32)
            self._meta[:2 * rows].copy_(host[:2 * rows], non_blocking=True)
            keys = self._meta[:rows], self._meta[rows:2 * rows]
        need = lib.sample_scratch_size(rows, vocab)
        if need and (self._scratch is None or self._scratch.numel() < need):
            self._scratch = torch.zeros(need, dtype=torch.int32, device=self.device)
        lib.sample(logits, params.temperature, params.top_p, params.top_k, params.seed,
                   *keys, tokens, probabilities, self._scratch if need else None)

    def __call__(self, logits, params, streams, counters) -> List[int]:
        """Tokens as Python ints (waits for the step)."""
        rows = logits.shape[0]
        self._reserve(rows)
        tokens = self._tokens_host[:rows]
        self._choose(logits, params, streams, counters, tokens)
        torch.cuda.current_stream().synchronize()
        self._last_rows = rows
        return tokens.tolist()

    def probabilities(self) -> List[float]:
        """Probability of each token of the last call within its filtered distribution."""
        return self._probabilities[:self._last_rows].tolist()
