"""The 32-bit Mersenne Twister of C++'s std::mt19937 (Matsumoto and Nishimura,
ACM TOMACS 8 (1998); parameters of [rand.predef] in the C++ standard), and the
two draws the samplers make from it.

The reference's samplers share one std::mt19937 seeded with the user's seed
(samplingHelperFunctions.cpp:56-75): a uniform double rng() / rng.max() and an
index rng() % n.  Reproducing the generator bit for bit reproduces their
seeded samples.
"""

from __future__ import annotations

import numpy as np

MAX = 0xFFFFFFFF
_BLOCK = 624  # outputs taken from the generator at a time


class MT19937:
    """The generator itself is numpy's: RandomState(seed) fills its state as
    std::mt19937::seed does (x_i = 1812433253 (x_{i-1} ^ (x_{i-1} >> 30)) + i), and integers
    over the whole 32-bit range are its raw outputs.  (The same in Python statements took
    0.1 ms to seed and 0.2 ms per 624 outputs, several times a sampling run's GPU work.)"""

    def __init__(self, seed: int = 5489):
        self._state = np.random.RandomState()
        self.seed(seed)

    def seed(self, value: int) -> None:
        self._state.seed(int(value) & MAX)  # taken modulo 2^32
        self._block: list[int] = []
        self._idx = 0

    def __call__(self) -> int:
        if self._idx >= len(self._block):
            self._refill()
        y = self._block[self._idx]
        self._idx += 1
        return y

    def _refill(self) -> None:
        self._block = self._state.randint(0, MAX + 1, size=_BLOCK, dtype=np.uint32).tolist()
        self._idx = 0

    def take(self, count: int) -> list[int]:
        """The next `count` outputs."""
        out: list[int] = []
        while len(out) < count:
            if self._idx >= len(self._block):
                self._refill()
            part = self._block[self._idx : self._idx + count - len(out)]
            self._idx += len(part)
            out += part
        return out

    def random_double_0_1(self) -> float:
        """samplingHelperFunctions.cpp:62-64"""
        return float(self()) / float(MAX)

    def random_index(self, upper_bound_exclusive: int) -> int:
        """samplingHelperFunctions.cpp:66-72"""
        if upper_bound_exclusive == 0:
            return 0
        return self() % upper_bound_exclusive
