"""The exact integer sweep on the FP64 pipe (perm_exact.hip): products of groups of
ceil(n / 3) column sums must stay within 46 bits, else the 64-bit integer sweep runs.
Results are whole numbers and compared for equality."""

import math

import numpy as np
import pytest

import oracle
from piquassoboost_amd import _capi as C

pytestmark = pytest.mark.gpu


def _column_sum_matrix(rng, n, cmax):
    """n x n integers of both signs whose first group of columns has abs sums of cmax, the
    others the largest that keep the whole inside the exact bound."""
    g = (n + 2) // 3
    rest = min(cmax, int(2.0 ** ((125 - (n - 1) - g * math.log2(cmax)) / (n - g))))
    A = np.zeros((n, n), dtype=np.int64)
    for j in range(n):
        total = cmax if j < g else rest
        A[:, j] = rng.multinomial(total, np.full(n, 1.0 / n)) * np.where(rng.random(n) < 0.5, -1, 1)
    assert np.abs(A).sum(axis=0).max() == cmax
    return A


# cmax^ceil(n/3) <= 2^46 on the FP64 pipe: the last that fits and the first that does not;
# and 2^44, 2^45, 2^46, where the digits are flushed every 256, 32 and 4 steps
@pytest.mark.parametrize("n,cmax", [(9, 41285), (9, 41286), (12, 2048), (12, 2435), (12, 2896), (12, 2897),
                                    (14, 588), (18, 203), (20, 95), (20, 96), (22, 53), (22, 54)])
def test_group_bound(n, cmax):
    rng = np.random.default_rng(9700 + n * 10 + cmax)
    A = _column_sum_matrix(rng, n, cmax)
    ok, lb = C.exact_bound(A.astype(float))
    print(f"exact fp64: n={n} cmax={cmax} group {cmax ** ((n + 2) // 3) / 2 ** 46:.4f} x 2^46, log2 bound {lb:.1f}",
          flush=True)
    assert ok
    assert C.permanent_exact(A.astype(float))[0] == oracle.int_permanent(A.astype(np.int64))


@pytest.mark.parametrize("n", list(range(1, 21)) + [23])
def test_small_entries_every_size(n):
    """Walks from none (n = 1) past one flush, lanes from one to a full wave, one wave to many."""
    rng = np.random.default_rng(9800 + n)
    print(f"exact fp64: n={n}", flush=True)
    for lo, hi in ((0, 1), (-1, 1), (-3, 3)):
        A = rng.integers(lo, hi + 1, size=(n, n))
        if not C.exact_bound(A.astype(float))[0]:  # -3 .. 3 at n = 23: beyond the 128-bit range
            continue
        assert C.permanent_exact(A.astype(float))[0] == oracle.int_permanent(A.astype(np.int64))


@pytest.mark.parametrize("n", [24, 26, 27, 28, 29])
def test_all_ones(n):
    """perm(J) = n!: 42 and 43 bits a group at 26 and 27 columns, the integer sweep from 28 on."""
    print(f"exact fp64: J_{n}", flush=True)
    ok, lb = C.exact_bound(np.ones((n, n)))
    if not ok:
        pytest.skip(f"outside the exact bound (log2 {lb:.1f})")
    assert C.permanent_exact(np.ones((n, n)))[0] == math.factorial(n)
