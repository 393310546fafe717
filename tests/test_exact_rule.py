"""The rule that admits integer matrices to the exact sweep on the FP64 pipe
(csrc/pqb_exact_rule.h), compiled for the host and compared with the same condition in
128-bit integers: c^ceil(C / 3) <= 2^46, and 2^(140 - 3 e) steps a flush, at most 256, for
products of at most 2^e."""

import shutil
import subprocess

import pytest

from conftest import ROOT

PROGRAM = r"""
#include <cstdio>
#include "pqb_exact_rule.h"

static int want(long long c, int C) {
    unsigned __int128 q = 1;
    for (int k = 0; k < (C + 2) / 3; ++k) {
        q *= (unsigned __int128)(c < 1 ? 1 : c);
        if (q >> 46 && q != (unsigned __int128)1 << 46) return 0;
    }
    int e = 0;
    while ((unsigned __int128)1 << e < q) ++e;
    const int f = 140 - 3 * e;
    return 1 << (f < 8 ? f : 8);
}

static long long wrong = 0;
static void check(long long c) {
    for (int C = 1; C <= 40; ++C)
        if (pqb::exact_fp64_flush(c, C) != want(c, C) && wrong++ < 10)
            std::printf("C = %d, column sum %lld: %d, not %d\n", C, c, pqb::exact_fp64_flush(c, C), want(c, C));
}

int main() {
    for (long long c = 0; c <= 1 << 18; ++c) check(c);
    for (long long c = 1 << 18; c <= 1 << 30; c += 997) check(c);
    for (int b = 18; b <= 30; ++b)
        for (long long c = (1ll << b) - 64; c <= (1ll << b) + 64 && c <= 1 << 30; ++c) check(c);
    // sums whose third or fourth power is a small number modulo 2^64
    for (long long c : {2642246ll, 2642247ll, 2642248ll, 2642249ll, 3329022ll, 4194304ll, 4194305ll, 5284492ll, 8388608ll})
        check(c);
    std::printf("%lld wrong\n", wrong);
    return wrong != 0;
}
"""


def test_every_product_fits(tmp_path):
    cxx = shutil.which("g++") or shutil.which("c++")
    if not cxx:
        pytest.skip("no host C++ compiler")
    (tmp_path / "rule.cpp").write_text(PROGRAM)
    # signed overflow wraps in a defined way here, as it does in most builds: the rule must not rely on it
    subprocess.run([cxx, "-O1", "-fwrapv", "-std=c++17", f"-I{ROOT / 'piquassoboost_amd' / 'csrc'}",
                    str(tmp_path / "rule.cpp"), "-o", str(tmp_path / "rule")], check=True)
    run = subprocess.run([str(tmp_path / "rule")], capture_output=True, text=True, timeout=100)
    assert run.returncode == 0, run.stdout
