"""The engine's host side without a GPU, on the stand-in for the HIP runtime
(host_runtime.cpp), which writes the launched kernels down and can be told to fail.  Each
test runs in a process of its own."""

import shutil
import subprocess
import sys
from pathlib import Path

import pytest

from conftest import ROOT

PRELUDE = """
import ctypes, sys
runtime = ctypes.CDLL(sys.argv[1], mode=ctypes.RTLD_GLOBAL)
runtime.host_runtime_launched.restype = ctypes.c_char_p
import numpy as np
from piquassoboost_amd import _capi as C
C._share_torch_hip_runtime = lambda: None  # torch would resolve to the stand-in too

def fail(name, call=1):
    runtime.host_runtime_fail(name.encode(), call)

def launched():
    return runtime.host_runtime_launched().decode().split()

def failed(call):
    try:
        call()
    except C.EngineError as e:
        return str(e)
    return None

def matrix(n, seed=1, cols=None):
    rng = np.random.default_rng(seed)
    return rng.standard_normal((n, cols or n)) + 1j * rng.standard_normal((n, cols or n))
"""


@pytest.fixture(scope="module")
def runtime(tmp_path_factory):
    cxx, include = shutil.which("g++") or shutil.which("c++"), Path("/opt/rocm/include")
    if not cxx or not include.is_dir():
        pytest.skip("no host C++ compiler or no HIP headers")
    so = tmp_path_factory.mktemp("host_runtime") / "libhost_runtime.so"
    subprocess.run([cxx, "-std=c++17", "-O1", "-shared", "-fPIC", "-D__HIP_PLATFORM_AMD__", f"-I{include}",
                    str(ROOT / "tests" / "host_runtime.cpp"), "-o", str(so)], check=True)
    return so


def run(runtime, body):
    r = subprocess.run([sys.executable, "-c", PRELUDE + body, str(runtime)], cwd=ROOT, capture_output=True, text=True,
                       timeout=100)
    assert r.returncode == 0, r.stdout + r.stderr


# calls by the route they take: one block, direct launches, the captured graph
BATCHES = """
ones = np.ones(14, np.int64)
def tiny(seed): return C.permanent_repeated(matrix(8, seed), [1] * 8, [1] * 8)
def small(count): return C.permanent_batch([(matrix(14, k), ones, ones) for k in range(count)])
def graph(): return small(65)
"""


@pytest.mark.parametrize("first", ["tiny(1)", "small(3)", "graph()"])
@pytest.mark.parametrize("then,at", [("tiny(2)", "hipLaunchKernel"), ("small(1)", "hipLaunchKernel"),
                                     ("small(5)", "hipMemcpyAsync"), ("small(5)", "hipLaunchKernel"),
                                     ("small(5)", "hipStreamSynchronize"), ("graph()", "hipLaunchKernel"),
                                     ("graph()", "hipGraphLaunch")])
def test_a_failed_batch_leaves_none_to_replay(runtime, first, then, at):
    """From its upload on a batch is written over the last one: where it fails, a replay of
    the last one would run on a mixture of both."""
    run(runtime, BATCHES + f"""
{first}
assert C.batch_replay_ms(2) > 0.0
launched()
fail({at!r})
assert failed(lambda: {then}) is not None
fail("")
launched()
assert failed(lambda: C.batch_replay_ms(2)) == "no batch has been run yet"
assert launched() == []
{first}
assert C.batch_replay_ms(2) > 0.0
""")


DOUBLE_DOUBLE = """
def wide(n, seed):
    A = matrix(n, seed)
    A[1, 2] = 1e-17  # a rounding residue
    return A
def sweeps(calls):
    return [k[k.index("rep_dd_kernel"):].split("EEEv")[0] for k in calls if "rep_dd_kernel" in k]
SPLIT, WHOLE = "rep_dd_kernelILi2ELi12ELb1", "rep_dd_kernelILi4ELi8ELb0"  # up to 24 slots
"""


def test_split_and_whole_rows_of_a_list_are_swept_apart(runtime):
    """In the double-double sweeps a matrix whose entries are too far apart to be split does
    not take many others of its list or batch along; a few small ones stay with it."""
    run(runtime, DOUBLE_DOUBLE + """
near, far, small = [matrix(22, k) for k in range(2)], [wide(22, k) for k in range(2)], [matrix(20, k) for k in range(6)]
C.permanent(near[0], precision=C.PREC_INF), C.permanent(far[0], precision=C.PREC_INF)
assert sweeps(launched()) == [SPLIT, WHOLE]
for mats, want in ((near, [SPLIT]), (far, [WHOLE]), ([near[0], far[0], near[1], far[1]], [SPLIT, WHOLE]),
                   (small, [SPLIT]), (small + far, [WHOLE])):
    C.permanent_list(mats, precision=C.PREC_INF)
    assert sweeps(launched()) == want
    ones = np.ones(22, np.int64)
    C.permanent_batch([(A, ones[:len(A)], ones[:len(A)]) for A in mats], precision=C.PREC_INF)
    assert sweeps(launched()) == want
""")


def test_repeated_tasks_of_more_than_32_slots_are_swept_apart(runtime):
    run(runtime, """
def task(m): return (matrix(6, m), [m] * 6, [m] * 6)
C.permanent_batch([task(3), task(6), task(4)])
calls = [k[k.index("rep_batch_kernel"):].split("EEEv")[0] for k in launched() if "rep_batch_kernel" in k]
assert calls == ["rep_batch_kernelILi1ELi26", "rep_batch_kernelILi33ELi40"]
""")


def test_limits_of_the_one_block_kernel(runtime):
    run(runtime, """
def kernels():
    return [next(k for k in ("tiny_kernel", "tiny_mixed", "plain_sweep", "plain_prep", "plain_mixed") if k in name)
            for name in launched()]
for rows, cols, want in ((11, 11, ["tiny_kernel"]), (11, 24, ["tiny_kernel"]), (11, 25, ["plain_sweep"]),
                         (12, 11, ["plain_sweep"]), (12, 12, ["plain_sweep"])):
    C.permanent(matrix(rows, 1, cols), precision=C.PREC_FP64)
    assert kernels() == want, (rows, cols)
for count, want in ((256, ["tiny_kernel"]), (257, ["plain_prep", "plain_sweep"])):
    buffers = [np.zeros(n) for n in (2 * 25 * count, 6 * count, C.batch_device_workspace_bytes(count, 5, 5) // 8 + 1)]
    A, out, work = (b.ctypes.data for b in buffers)
    C.permanent_batch_device(A, count, 5, 5, out, work, buffers[2].nbytes, 0)
    assert kernels() == want, count
""")
