"""Permanents of up to 2048 signed terms in one block (perm_tiny.hip): plain ones of up to
12 rows (host, list and device entries) and single repeated-row calls of few steps."""

import numpy as np
import pytest

import oracle
from conftest import random_complex, rel_err
from piquassoboost_amd import _capi as C

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu
DEV = torch.device("cuda:0")
TOL = 1e-12


# one column to the most (24, then the general sweep), one row to the most (12, then 13),
# terms below a wave, of exactly one, past a block's threads
@pytest.mark.parametrize("shape", [(1, 1), (2, 1), (1, 24), (2, 24), (6, 6), (7, 7), (7, 12), (8, 7), (11, 11),
                                   (11, 24), (12, 11), (12, 12), (12, 24), (12, 25), (13, 12), (13, 13)])
def test_plain_shapes(shape):
    r, c = shape
    rng = np.random.default_rng(9900 + 40 * r + c)
    B = np.stack([random_complex(rng, r, c) for _ in range(5)])
    print(f"tiny: {r} x {c}", flush=True)
    one = [C.permanent(A, C.ALGO_BBFG, C.PREC_FP64) for A in B]
    assert C.permanent_list(list(B), C.ALGO_BBFG, C.PREC_FP64) == one
    dA = torch.from_numpy(B).to(DEV)
    out = torch.full((6, 6), float("nan"), dtype=torch.float64, device=DEV)
    wb = C.batch_device_workspace_bytes(5, r, c)
    work = torch.zeros(wb, dtype=torch.uint8, device=DEV)
    st = torch.cuda.current_stream(DEV).cuda_stream
    C.permanent_batch_device(dA.data_ptr(), 5, r, c, out.data_ptr(), work.data_ptr(), wb, st)
    C.permanent_device_noalloc(dA.data_ptr(), r, c, out[5].data_ptr(), st)
    o = out.cpu().numpy()
    for b in range(6):
        ref = oracle.bbfg(B[b % 5], "dd")
        scale = abs(ref) if r == c else max(abs(ref), np.prod(np.abs(B[b % 5]).sum(axis=0)) * 1e-3)
        assert abs(complex(o[b, 0], o[b, 1]) - ref) <= TOL * scale
        assert abs(one[b % 5] - ref) <= TOL * scale


# (row multiplicities, column multiplicities): steps 1, 2, a wave, 1023 .. 2048 and past,
# digits of radix 2 to 13, one row only, 24 photons and past
REPEATED = [([1], [1]), ([5], [5]), ([2, 1], [1, 1, 1]), ([1] * 7, [1] * 7), ([1] * 6 + [2], [1] * 8),
            ([3, 3, 3, 3, 3], [1] * 15), ([7, 7, 7], [3] * 7), ([12, 12], [8, 8, 8]),
            ([12, 13], [5] * 5), ([1] * 12, [1] * 12), ([1] * 13, [1] * 13), ([2] * 7, [1] * 14),
            ([4, 4, 4, 4, 4, 4], [2] * 12)]


@pytest.mark.parametrize("case", range(len(REPEATED)))
def test_repeated(case):
    rm, cm = (np.array(v, dtype=np.int64) for v in REPEATED[case])
    rng = np.random.default_rng(9990 + case)
    A = random_complex(rng, len(rm), len(cm))
    print(f"tiny: repeated {rm} {cm}", flush=True)
    ref = oracle.bbfg_repeated(A, cm, rm, "dd")
    got = C.permanent_repeated(A, rm, cm)
    assert rel_err(got, ref) < TOL
    C.permanent(random_complex(rng, 9, 9))  # another call on the context's staging buffer
    assert C.batch_replay_ms(3) > 0.0       # the call just made can be replayed, as any batch
    assert C.permanent_repeated(A, rm, cm) == got
    assert rel_err(C.permanent_batch([(A, rm, cm)] * 3)[1], ref) < TOL


def test_non_finite_entries_stay_non_finite():
    rng = np.random.default_rng(9995)
    for bad in (np.nan, np.inf):
        A = random_complex(rng, 9, 9)
        A[3, 7] = bad
        for v in (C.permanent(A, C.ALGO_BBFG, C.PREC_FP64), C.permanent_repeated(A, [1] * 9, [1] * 9)):
            assert not (np.isfinite(v.real) and np.isfinite(v.imag))
