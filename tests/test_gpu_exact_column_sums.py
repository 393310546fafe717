"""Integer matrices whose column sums are so large that a power of theirs is small modulo
2^64 (2^22, 2^23, 2642246): inside the exact bound, beyond the products of 46 bits that the
sweep on the FP64 pipe takes.  The values are whole numbers, formed in Python's integers."""

import numpy as np
import pytest

from piquassoboost_amd import _capi as C

pytestmark = pytest.mark.gpu


def _whole_permanent(A):
    """Expansion along the rows: the permanents of the first rows over column subsets."""
    n = len(A)
    F = {0: 1}
    for row in A.tolist():
        G = {}
        for S, f in F.items():
            for j in range(n):
                if not S >> j & 1 and row[j]:
                    G[S | 1 << j] = G.get(S | 1 << j, 0) + f * row[j]
        F = G
    return F.get((1 << n) - 1, 0)


def _signed(rng, n, total):
    """n whole numbers of both signs whose absolute values add up to `total`."""
    return rng.multinomial(total, np.full(n, 1.0 / n)) * np.where(rng.random(n) < 0.5, -1, 1)


@pytest.mark.parametrize("cmax", [1 << 22, 1 << 23, 2642246])
@pytest.mark.parametrize("n", [7, 9, 10, 12])
def test_large_column_sums(n, cmax):
    rng = np.random.default_rng(9650 + n * 3 + cmax)
    mats = []
    for wide in (1, 3):  # columns of that sum, small ones beside them
        A = rng.integers(0, 3, size=(n, n))
        A[:, :wide] = np.stack([_signed(rng, n, cmax) for _ in range(wide)], axis=1)
        mats.append(A)
    A = rng.integers(0, 2, size=(n, n))  # a row of large entries: every column's sum is large
    A[0] = rng.integers(cmax - cmax // 16, cmax - n, size=n)
    A[0, 2] = cmax - A[1:, 2].sum()
    mats.append(A)
    for k, A in enumerate(mats):
        assert np.abs(A).sum(axis=0).max() == cmax
        ok, lb = C.exact_bound(A.astype(float))
        print(f"exact column sums: n={n} cmax={cmax} form {k}, log2 bound {lb:.1f}", flush=True)
        assert ok
        want = _whole_permanent(A)
        assert C.permanent_exact(A.astype(float))[0] == want
        assert C.permanent(A.astype(float)) == complex(float(want))
        assert C.permanent_list([A.astype(float)]) == [complex(float(want))]
