"""The expanded plain sweep (perm_expand.hip): square matrices from 2^24 sign vectors on
are expanded along one row where their entries allow it.  Checked against the oracle over
the forms a matrix can have -- expanded or kept, mixed in one batch -- and against the
double-double sweep at sizes beyond the oracle."""

import numpy as np
import pytest

import oracle
from conftest import random_complex, rel_err
from piquassoboost_amd import _capi as C

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu
DEV = torch.device("cuda:0")
TOL = 1e-12  # the bar of the plain FP64 sweep


def device_batch(B):
    count, n, _ = B.shape
    dA = torch.from_numpy(np.ascontiguousarray(B)).to(DEV)
    out = torch.full((count, 6), float("nan"), dtype=torch.float64, device=DEV)
    wb = C.batch_device_workspace_bytes(count, n, n)
    work = torch.zeros(wb, dtype=torch.uint8, device=DEV)
    st = torch.cuda.current_stream(DEV).cuda_stream
    res = []
    for _ in range(2):  # the counters are left at zero
        C.permanent_batch_device(dA.data_ptr(), count, n, n, out.data_ptr(), work.data_ptr(), wb, st)
        torch.cuda.synchronize()
        res.append(out.cpu().numpy().copy())
    assert np.array_equal(res[0], res[1], equal_nan=True)
    assert int(work[: 4 * count].sum()) == 0
    return res[0][:, 0] + 1j * res[0][:, 1]


def forms(rng, n):
    """Matrices by the form the table may take: name -> matrix."""
    A = random_complex(rng, n, n)
    f = {"dense": A, "real": A.real + 0j, "scaled": A * (1e-5 * np.exp(rng.uniform(-3, 3, (1, n))))}
    f["one full row"] = np.where(rng.random((n, n)) < 0.3, 0, A)
    f["one full row"][n - 2] = A[n - 2]
    f["sparse"] = np.where(rng.random((n, n)) < 0.3, 0, A)  # kept
    f["sparse"][np.arange(n), (np.arange(n) + 1) % n] = 0
    f["spread"] = A.copy()  # kept: every row has an entry 2^-17 of the largest
    f["spread"][np.arange(n), np.arange(n)] *= 2.0**-20
    f["integers"] = rng.integers(1, 3, (n, n)) + 1j * rng.integers(-1, 2, (n, n))  # kept
    f["large"] = A * 2.0**21  # kept
    return f


@pytest.mark.parametrize("n", [14, 15, 17, 20])
def test_forms_in_one_batch(n):
    """The device batch decides per matrix, so one launch holds both."""
    rng = np.random.default_rng(9100 + n)
    f = forms(rng, n)
    count = max(len(f), 1 << (25 - n))
    B = np.stack([random_complex(rng, n, n) for _ in range(count)])
    at = rng.choice(count, size=len(f), replace=False)
    for i, m in zip(at, f.values()):
        B[i] = m
    print(f"expand: batch {count} x n={n}", flush=True)
    got = device_batch(B)
    for i, (name, m) in zip(at, f.items()):
        assert rel_err(got[i], oracle.bbfg(m, "dd")) < TOL, name
    for i in rng.choice(count, size=3, replace=False):
        assert rel_err(got[i], oracle.bbfg(B[i], "dd")) < TOL


@pytest.mark.parametrize("n", [25, 26])
def test_single_entries_agree(n):
    """Host call, list, device and no-allocation entries: the same bits; one oracle value."""
    rng = np.random.default_rng(9200 + n)
    for name, m in forms(rng, n).items():
        print(f"expand: n={n} {name}", flush=True)
        one = C.permanent(m, C.ALGO_BBFG, C.PREC_FP64)
        assert C.permanent_list([m, m[:3, :3], m], C.ALGO_BBFG, C.PREC_FP64)[::2] == [one, one]
        dA = torch.from_numpy(np.ascontiguousarray(m, dtype=np.complex128)).to(DEV)
        out = torch.zeros(12, dtype=torch.float64, device=DEV)
        wb = C.device_workspace_bytes(n, n)
        work = torch.zeros(wb, dtype=torch.uint8, device=DEV)
        st = torch.cuda.current_stream(DEV).cuda_stream
        C.permanent_device(dA.data_ptr(), n, n, out.data_ptr(), work.data_ptr(), wb, st)
        C.permanent_device_noalloc(dA.data_ptr(), n, n, out[6:].data_ptr(), st)
        o = out.cpu().numpy()
        assert complex(o[0], o[1]) == one and np.array_equal(o[:6], o[6:])
        if n == 25 and name in ("dense", "one full row", "spread"):
            assert rel_err(one, oracle.bbfg(m, "dd")) < TOL, name


@pytest.mark.parametrize("n", [27, 29, 31, 32, 33, 34])
def test_beyond_the_oracle_against_the_double_double_sweep(n):
    """The register and occupancy edges of the kernel (32 and 33 columns), odd sizes."""
    rng = np.random.default_rng(9300 + n)
    m = random_complex(rng, n, n)
    want = C.permanent(m, C.ALGO_BBFG, C.PREC_INF)
    got = C.permanent(m, C.ALGO_BBFG, C.PREC_FP64)
    print(f"expand: n={n} rel_err {rel_err(got, want):.1e}", flush=True)
    assert rel_err(got, want) < 1e-10  # the bar of the plain sweep at n = 28 .. 36


def test_non_finite_entries_stay_non_finite():
    rng = np.random.default_rng(9400)
    for bad in (np.nan, np.inf):
        A = random_complex(rng, 25, 25)
        A[3, 7] = bad
        v = C.permanent(A, C.ALGO_BBFG, C.PREC_FP64)
        assert not (np.isfinite(v.real) and np.isfinite(v.imag))


def _spread_over_rows(rng, photons, rows, only=None):
    """Multiplicities of `rows` rows with `photons` photons; only: every one that value."""
    if only:
        return np.full(photons // only, only, dtype=np.int64)
    return (1 + rng.multinomial(photons - rows, np.full(rows, 1.0 / rows))).astype(np.int64)


@pytest.mark.parametrize("photons,rows,only", [(13, 13, 0), (14, 13, 0), (16, 0, 2), (18, 0, 3), (21, 12, 0),
                                               (26, 16, 0), (20, 0, 4)])
@pytest.mark.parametrize("transposed", [False, True])
def test_repeated_rows(photons, rows, only, transposed):
    """Degrees 1, 2, 3 and none (every multiplicity 4), from the smallest expanded slot
    count on, both orientations, over the forms the rows can have; alone, in a batch with
    the others, and with no digit walked."""
    rng = np.random.default_rng(9500 + photons * 2 + transposed)
    mult = _spread_over_rows(rng, photons, rows, only)
    R = len(mult)
    one = np.ones(photons, np.int64)
    base = random_complex(rng, R, photons)
    mats = {"dense": base, "zeros in the single rows": np.where((mult == 1)[:, None] & (rng.random(base.shape) < 0.2),
                                                                0, base),
            "zeros in all rows": np.where(rng.random(base.shape) < 0.15, 0, base),
            "small": base * 1e-5, "integers": rng.integers(1, 4, base.shape) + 1j}
    tasks, want = [], []
    for name, m in mats.items():
        A, r, c = (np.ascontiguousarray(m.T), one, mult) if transposed else (m, mult, one)
        tasks.append((A, r, c))
        want.append(oracle.bbfg_repeated(np.ascontiguousarray(A, dtype=np.complex128), c, r, "dd"))
        print(f"expand: repeated {photons}/{R} {name} transposed={transposed}", flush=True)
        assert rel_err(C.permanent_repeated(A, r, c), want[-1]) < TOL, name
    for walk in (0, 1, 16):
        got = C.permanent_batch(tasks, walk_length=walk)
        for v, w in zip(got, want):
            assert rel_err(v, w) < TOL, walk


def test_repeated_rows_and_columns():
    """Multiplicities on both sides, up to the largest slot count (past 32 slots the batch
    is split), against the double-double sweep."""
    rng = np.random.default_rng(9600)
    tasks = []
    for photons, rows, cols in ((24, 14, 20), (31, 12, 26), (33, 13, 13), (36, 14, 12), (40, 14, 11)):
        tasks.append((random_complex(rng, rows, cols), _spread_over_rows(rng, photons, rows),
                      _spread_over_rows(rng, photons, cols)))
    print("expand: repeated rows and columns", flush=True)
    got = C.permanent_batch(tasks)
    want = C.permanent_batch(tasks, precision=C.PREC_INF)
    for v, w, (A, r, c) in zip(got, want, tasks):
        assert rel_err(v, w) < 1e-10, int(r.sum())
        assert rel_err(C.permanent_repeated(A, r, c), w) < 1e-10
