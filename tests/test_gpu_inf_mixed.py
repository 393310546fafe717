"""Double-double sweeps of lists and batches that hold matrices whose rows can be split on a
grid and ones whose entries are too far apart for that, together where the first are little
work and each kind by itself else (22 columns here): every value is its own call's and the
oracle's."""

import numpy as np
import pytest

import oracle
from conftest import random_complex
from piquassoboost_amd import _capi as C

pytestmark = pytest.mark.gpu


def _wide(A):
    A = A.copy()
    A[0, -1] *= 2.0 ** -60
    return A


@pytest.mark.parametrize("sizes", [(3, 3), (8, 9, 8), (13, 13, 12, 12, 13), tuple(range(2, 14)) * 6,
                                   (22, 3, 22, 9)])
def test_lists_and_batches(sizes):
    rng = np.random.default_rng(1400 + len(sizes))
    mats = [random_complex(rng, n, n) for n in sizes]
    mats = [_wide(A) if k % 2 else A for k, A in enumerate(mats)]
    print(f"inf mixed: {len(mats)} matrices", flush=True)
    ones = [np.ones(len(A), np.int64) for A in mats]
    got = C.permanent_list(mats, C.ALGO_GLYNN, C.PREC_INF)
    batch = C.permanent_batch([(A, o, o) for A, o in zip(mats, ones)], precision=C.PREC_INF)
    for A, v, b in zip(mats, got, batch):
        ref = oracle.bbfg(A, "dd")
        assert v == C.permanent(A, C.ALGO_GLYNN, C.PREC_INF)
        assert abs(v - ref) <= 2.0 ** -51 * abs(ref)
        assert abs(b - ref) <= 2.0 ** -51 * abs(ref)


def test_repeated_rows():
    rng = np.random.default_rng(1450)
    tasks = []
    for k, (rows, cols) in enumerate([([3, 2, 4], [5, 4]), ([8, 7, 8, 1], [12, 12]), ([1], [1]), ([2, 2, 2], [3, 3]),
                                      ([10, 12, 11], [11, 11, 11]), ([6, 6], [4, 4, 4])]):
        A = random_complex(rng, len(rows), len(cols))
        tasks.append((_wide(A) if k % 2 else A, np.array(rows, np.int64), np.array(cols, np.int64)))
    tasks.append((np.zeros((0, 0)), np.zeros(0, np.int64), np.zeros(0, np.int64)))  # decided without a sweep
    print("inf mixed: repeated", flush=True)
    got = C.permanent_batch(tasks, precision=C.PREC_INF)
    assert got[-1] == 1.0
    for v, (A, r, c) in list(zip(got, tasks))[:-1]:
        ref = oracle.bbfg_repeated(A, c, r, "dd")
        assert abs(v - ref) <= 2.0 ** -50 * abs(ref)
        one = C.permanent_repeated(A, r, c, precision=C.PREC_INF)
        assert abs(one - ref) <= 2.0 ** -50 * abs(ref)
