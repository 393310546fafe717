"""Matrices of small whole numbers times a power of two: the sum over all rows does not round
and they keep it, so a power of two taken out of the matrix comes out of the permanent, bit for
bit.  And matrices at the limits of the rule by which a row is expanded, which the host and the
table kernel apply apart: their sweeps must be the same."""

import numpy as np
import pytest

from conftest import random_complex
from piquassoboost_amd import _capi as C

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu
DEV = torch.device("cuda:0")


def _odd(rng, shape):
    """+-1 and +-3, a row of +-3: its quotients round, so an expansion along it would."""
    A = rng.choice([-1.0, 1.0, 3.0, -3.0], size=shape, p=(0.4, 0.4, 0.1, 0.1)) + 0j
    A[..., 3, :] = rng.choice([-3.0, 3.0], size=shape[:-2] + shape[-1:])
    return A


def _device(B):
    count, n, _ = B.shape
    dA = torch.from_numpy(np.ascontiguousarray(B)).to(DEV)
    out = torch.zeros((count, 6), dtype=torch.float64, device=DEV)
    wb = C.batch_device_workspace_bytes(count, n, n)
    work = torch.zeros(wb, dtype=torch.uint8, device=DEV)
    C.permanent_batch_device(dA.data_ptr(), count, n, n, out.data_ptr(), work.data_ptr(), wb,
                             torch.cuda.current_stream(DEV).cuda_stream)
    o = out.cpu().numpy()
    return o[:, 0] + 1j * o[:, 1]


@pytest.mark.parametrize("shift", [1, 7, -3])
@pytest.mark.parametrize("n", [14, 16])
def test_device_batch(n, shift):
    rng = np.random.default_rng(9420 + n)
    A = _odd(rng, (1 << (25 - n), n, n))
    A[::2] += 1j * rng.integers(-1, 2, size=A[::2].shape)
    print(f"expand grid: batch n={n} shift={shift}", flush=True)
    assert np.array_equal(_device(A * 2.0 ** -shift) * 2.0 ** (n * shift), _device(A))


def test_host_call():
    n = 25
    A = _odd(np.random.default_rng(9430), (n, n))
    print("expand grid: host n=25", flush=True)
    whole = C.permanent(A, C.ALGO_BBFG, C.PREC_FP64)
    assert C.permanent(A / 8, C.ALGO_BBFG, C.PREC_FP64) * 2.0 ** (3 * n) == whole
    assert C.permanent_list([A / 2, A], C.ALGO_BBFG, C.PREC_FP64) == [whole * 2.0 ** -n, whole]


@pytest.mark.parametrize("mult", [[1] * 14, [2] * 8, [3] * 7])
def test_repeated_rows(mult):
    n = sum(mult)
    A = _odd(np.random.default_rng(9440 + n), (len(mult), n))
    r, c = np.array(mult, np.int64), np.ones(n, np.int64)
    print(f"expand grid: repeated {mult}", flush=True)
    whole = C.permanent_repeated(A, r, c)
    assert C.permanent_repeated(A / 2, r, c) * 2.0 ** n == whole
    T = np.ascontiguousarray(A.T)
    assert C.permanent_repeated(T / 2, c, r) * 2.0 ** n == C.permanent_repeated(T, c, r)


def _limits(rng, n):
    A = random_complex(rng, n, n)
    A[np.maximum(np.abs(A.real), np.abs(A.imag)) < 2.0 ** -5] = 0.3 - 0.2j
    f = {}
    for name, least in (("least entry on the limit", 1.0), ("least entry below it", 1.0 - 2.0 ** -52)):
        f[name] = A.copy()
        f[name][0, 0] = 4.0
        f[name][:, 1] = (4.0 * 2.0 ** -16 * least) * (1.0 - 0.5j)  # every row's smallest
    f["largest on the limit"] = A.copy()
    f["largest on the limit"][2] = 2.0 ** 19 + 1j * rng.uniform(1.0, 2.0, n)
    f["largest on the limit"][2, 4] = 2.0 ** 20
    f["largest past it"] = f["largest on the limit"].copy()
    f["largest past it"][2, 4] = 2.0 ** 20 * (1.0 + 2.0 ** -52)
    for bits in (20, 21):  # whole numbers of 21 bits and of 22, times a power of two
        g = rng.integers(1, 8, (n, n)) + 1j * rng.integers(0, 8, (n, n))
        g[1, 2] = 2.0 ** bits + 1.0
        g[3] = (2.0 ** bits - 8.0) + rng.integers(0, 7, n)
        f[f"{bits + 1} bits"] = g * 2.0 ** -15
    return f


def test_limits_agree():
    n = 25
    for name, m in _limits(np.random.default_rng(9450), n).items():
        print(f"expand grid: {name}", flush=True)
        one = C.permanent(m, C.ALGO_BBFG, C.PREC_FP64)
        dA = torch.from_numpy(np.ascontiguousarray(m)).to(DEV)
        out = torch.zeros(6, dtype=torch.float64, device=DEV)
        C.permanent_device_noalloc(dA.data_ptr(), n, n, out.data_ptr(), torch.cuda.current_stream(DEV).cuda_stream)
        o = out.cpu().numpy()
        assert complex(o[0], o[1]) == one, name
