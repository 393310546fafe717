"""Both sides of the limits of the one-block kernel (perm_tiny.hip): 11 rows and 12, 24
columns and 25, device batches of 256 matrices and of 257."""

import numpy as np
import pytest

import oracle
from conftest import random_complex
from piquassoboost_amd import _capi as C

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu
DEV = torch.device("cuda:0")


def _device_batch(B):
    count, r, c = B.shape
    dA = torch.from_numpy(B).to(DEV)
    out = torch.full((count, 6), float("nan"), dtype=torch.float64, device=DEV)
    wb = C.batch_device_workspace_bytes(count, r, c)
    work = torch.zeros(wb, dtype=torch.uint8, device=DEV)
    C.permanent_batch_device(dA.data_ptr(), count, r, c, out.data_ptr(), work.data_ptr(), wb,
                             torch.cuda.current_stream(DEV).cuda_stream)
    o = out.cpu().numpy()
    return o[:, 0] + 1j * o[:, 1]


def _close(got, A):
    ref = oracle.bbfg(A, "dd")
    scale = abs(ref) if A.shape[0] == A.shape[1] else np.prod(np.abs(A).sum(axis=0)) * 1e-3
    return abs(got - ref) <= 1e-12 * max(abs(ref), scale)


@pytest.mark.parametrize("shape", [(11, 10), (11, 12), (11, 24), (11, 25), (12, 11), (12, 12), (12, 24), (12, 25)])
def test_rows_and_columns(shape):
    B = np.stack([random_complex(np.random.default_rng(9960 + k), *shape) for k in range(3)])
    print(f"tiny limits: {shape}", flush=True)
    one = [C.permanent(A, C.ALGO_BBFG, C.PREC_FP64) for A in B]
    assert C.permanent_list(list(B), C.ALGO_BBFG, C.PREC_FP64) == one
    for A, v, d in zip(B, one, _device_batch(B)):
        assert _close(v, A) and _close(d, A)


@pytest.mark.parametrize("count", [256, 257])
@pytest.mark.parametrize("shape", [(1, 1), (5, 5), (11, 11)])
def test_device_batches(shape, count):
    rng = np.random.default_rng(9970 + count)
    B = np.stack([random_complex(rng, *shape) for _ in range(count)])
    print(f"tiny limits: {count} x {shape}", flush=True)
    got = _device_batch(B)
    assert np.isfinite(got).all()
    for k in (0, 1, 17, 128, 255, count - 1):
        assert _close(got[k], B[k])
