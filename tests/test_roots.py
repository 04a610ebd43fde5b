"""Roots of unity of the plans' tables (csrc/roots.hpp), built with g++ beside a
driver (tests/host/roots_driver.cpp): the reflected roots against the direct
evaluation, and how many evaluations a table costs."""
import os
import shutil
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, "..", "vkfft-rs_amd", "csrc")

pytestmark = pytest.mark.skipif(shutil.which("g++") is None, reason="needs g++")


def _run(tmp_path, source, name):
    exe = str(tmp_path / name)
    subprocess.run(["g++", "-std=c++17", "-O1", "-I", CSRC, source, "-o", exe], check=True, capture_output=True, text=True)
    r = subprocess.run([exe], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stdout[-2000:]
    return r.stdout


def test_roots(tmp_path):
    assert _run(tmp_path, os.path.join(HERE, "host", "roots_driver.cpp"), "roots").startswith("ok ")


def test_evaluations(tmp_path):
    """Two for a block of the first eighth, quarter or half: 2 sqrt of its length."""
    src = tmp_path / "count.cpp"
    src.write_text("""#include <cmath>
#include <cstdio>
static long double counted(long double a);
#define cosl counted
#include "roots.hpp"
#undef cosl
static int calls = 0;
static long double counted(long double a) { ++calls; return cosl(a); }
int main() {
    for (size_t n : {1, 2, 1080, 1024, 1010, 1001}) {
        std::vector<long double> re, im;
        calls = 0;
        vkfx::roots(n, re, im);
        std::printf("%zu %d\\n", n, calls);
    }
}
""")
    got = dict(tuple(map(int, line.split())) for line in _run(tmp_path, str(src), "count").splitlines())
    assert got == {1: 1, 2: 1, 1080: 24, 1024: 24, 1010: 31, 1001: 47}
