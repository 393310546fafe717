"""Large batches on one matrix, whose rows are formed on the GPU, against the same tasks
with a copy of the matrix each, whose rows the host lays out: the same bits."""

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def tasks(rows, cols, lo, hi, count, seed):
    rng = np.random.default_rng(seed)
    outs, ins = np.zeros((count, rows), np.int64), np.zeros((count, cols), np.int64)
    for i in range(count):
        n = int(rng.integers(lo, hi + 1))
        np.add.at(outs[i], rng.integers(0, rows, n), 1)
        np.add.at(ins[i], rng.integers(0, cols, n), 1)
    return outs, ins


@pytest.mark.parametrize("rows,cols,lo,hi,count,precision", [
    (5, 4, 0, 6, 65, "PREC_DOUBLE"),     # few modes, no photons among them: bunched, transposed
    (9, 30, 8, 15, 70, "PREC_DOUBLE"),   # rows and columns of different number
    (40, 21, 12, 17, 130, "PREC_DOUBLE"),  # expanded rows of all multiplicities
    (24, 24, 30, 36, 66, "PREC_DOUBLE"),   # more than 32 slots: two launches
    (12, 12, 3, 9, 80, "PREC_INF"),
])
def test_rows_formed_on_the_gpu(rows, cols, lo, hi, count, precision):
    from piquassoboost_amd import _capi as C

    rng = np.random.default_rng(rows)
    whole = rng.standard_normal((rows + 2, cols + 3)) + 1j * rng.standard_normal((rows + 2, cols + 3))
    U = whole[1 : rows + 1, 2 : cols + 2] / np.sqrt(2 * cols)
    U = np.ascontiguousarray(np.pad(U, ((0, 0), (0, 3))))[:, :cols]  # row stride cols + 3
    if hi > 30:  # few distinct rows keep the number of terms small
        outs, ins = tasks(4, 4, lo, hi, count, rows)
        outs, ins = np.pad(outs, ((0, 0), (0, rows - 4))), np.pad(ins, ((0, 0), (cols - 4, 0)))
    else:
        outs, ins = tasks(rows, cols, lo, hi, count, rows)
    prec = getattr(C, precision)
    got = C.permanent_batch_states(U, ins, outs, precision=prec)
    ref = C.permanent_batch([(np.ascontiguousarray(U), o, i) for o, i in zip(outs, ins)], precision=prec)
    assert np.array_equal(got, np.asarray(ref))
