"""Lists of more small shapes than one launch takes, and of shapes on either side of the
limits up to which they share one: every value is its own call's, bit for bit."""

import numpy as np
import pytest

from conftest import random_complex

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shapes", [
    [(r, c) for r in range(1, 12) for c in (r - 1, r, r + 1, r + 2) if c >= 1],   # a block per matrix
    [(c + d, c) for c in range(11, 23) for d in (-1, 0, 1)],                      # two launches of 16 and rest
    [(5, 5)] * 256 + [(6, 6)] * 257 + [(12, 12)] * 3 + [(4, 4)],
    [(14, 14)] * 129 + [(21, 21)] * 9 + [(17, 17), (22, 22)],
    [(13, 13)],
])
def test_equals_per_call(shapes):
    from piquassoboost_amd import _capi as C

    rng = np.random.default_rng(len(shapes))
    mats = [random_complex(rng, r, c) for r, c in shapes]
    order = rng.permutation(len(mats))
    got = C.permanent_list([mats[i] for i in order], C.ALGO_BBFG, C.PREC_FP64)
    for v, i in zip(got, order):
        if i % max(1, len(mats) // 60) == 0:
            assert v == C.permanent(mats[i], C.ALGO_BBFG, C.PREC_FP64), shapes[i]
