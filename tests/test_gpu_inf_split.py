"""The double-double sweep over split rows against the one that keeps every column sum
normalised, which takes matrices whose entries' range is too wide to split: with a further
row and column that hold 2^-50 where they cross and zeros elsewhere, every term is the other
matrix's times 2^-50 exactly.  Slot counts at the edges of the lanes' shares; entries at the
edge of the range; zeros."""

import numpy as np
import pytest

import oracle
from conftest import random_complex

pytestmark = pytest.mark.gpu


def wide(A):
    W = np.pad(A, ((0, 1), (0, 1)))
    W[-1, -1] = 2.0 ** -50
    return W


@pytest.mark.parametrize("n", [2, 3, 7, 8, 9, 13, 15, 16, 17, 18, 20])
def test_plain(n):
    from piquassoboost_amd import _capi as C

    rng = np.random.default_rng(1300 + n)
    A = random_complex(rng, n, n)
    A[rng.random((n, n)) < 0.1] = 0.0
    np.fill_diagonal(A, 0.7 - 0.2j)
    split = C.permanent(A, C.ALGO_GLYNN, C.PREC_INF)
    assert split == C.permanent(wide(A), C.ALGO_GLYNN, C.PREC_INF) * 2.0 ** 50
    if n <= 13:
        ref = oracle.bbfg(A, "dd")
        assert abs(split - ref) <= 2.0 ** -51 * abs(ref)


@pytest.mark.parametrize("rows,cols", [
    ([8, 7, 8, 1], [12, 12]),          # 24 slots
    ([9, 9, 7], [10, 5, 10]),          # 25
    ([10, 12, 10], [16, 16]),          # 32
    ([10, 12, 11], [11, 11, 11]),      # 33
    ([13, 13, 13], [20, 19]),          # 39
])
def test_repeated(rows, cols):
    from piquassoboost_amd import _capi as C

    rng = np.random.default_rng(sum(rows) + 7)
    A = random_complex(rng, len(rows), len(cols))
    r, c = np.array(rows, np.int64), np.array(cols, np.int64)
    split = C.permanent_repeated(A, r, c, precision=C.PREC_INF)
    ref = C.permanent_repeated(wide(A), np.append(r, 1), np.append(c, 1), precision=C.PREC_INF)
    assert split == ref * 2.0 ** 50


@pytest.mark.parametrize("low", [-38, -39, -40, -41, -45, -70])
def test_entries_at_the_edge_of_the_range(low):
    """Entries from 2^low to 1: the sums are exact in either form."""
    from piquassoboost_amd import _capi as C

    rng = np.random.default_rng(-low)
    n = 9
    A = random_complex(rng, n, n) * 2.0 ** rng.integers(low, 1, (n, n))
    got, ref = C.permanent(A, C.ALGO_GLYNN, C.PREC_INF), oracle.bbfg(A, "dd")
    assert abs(got - ref) <= 2.0 ** -50 * abs(ref)


@pytest.mark.parametrize("v", [np.inf, np.nan])
def test_non_finite(v):
    from piquassoboost_amd import _capi as C

    A = np.ones((5, 5), np.complex128)
    A[2, 3] = v
    assert not np.isfinite(C.permanent(A, C.ALGO_GLYNN, C.PREC_INF))
