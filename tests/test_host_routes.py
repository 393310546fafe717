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
