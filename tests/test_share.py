"""The shares that a leaf's targets are dealt out in (csrc/share.hpp), on the
CPU over all 32-bit sizes: in order, without gaps, none longer than asked for."""
import ctypes
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

PROGRAM = r"""
#include "share.hpp"
// 0, or the 1-based share that is wrong
extern "C" long check_passes(int n, int per) {
  const int k = pam::share_count(n, per);
  if (static_cast<long>(k) * per < n || static_cast<long>(k - 1) * per >= n) return -1;
  int end = 0;
  for (int i = 0; i < k; i++) {
    const int b = pam::share_begin(n, i, k), e = pam::share_begin(n, i + 1, k);
    if (b != end || e < b || e > n || e - b > per) return i + 1;
    end = e;
  }
  return end == n ? 0 : -2;
}
extern "C" int begin(int n, int i, int k) { return pam::share_begin(n, i, k); }
"""


@pytest.fixture(scope="module")
def lib(tmp_path_factory):
    d = tmp_path_factory.mktemp("share")
    (d / "share_check.cpp").write_text(PROGRAM)
    out = str(d / "share_check.so")
    subprocess.run(["g++", "-O2", "-std=c++20", "-shared", "-fPIC", "-I", os.path.join(ROOT, "polatory_amd", "csrc"),
                    str(d / "share_check.cpp"), "-o", out], check=True)
    so = ctypes.CDLL(out)
    so.check_passes.restype = ctypes.c_long
    return so


# 128 and 80 targets a pass (vector units), 20 tiles a pass (matrix unit).
@pytest.mark.parametrize("per", [20, 80, 128])
@pytest.mark.parametrize("n", [1, 19, 20, 21, 80, 127, 128, 129, 207_361, 414_482, 524_288, 524_289, 600_000, 3_400_000,
                               5_000_000, 2 ** 31 - 1])
def test_passes_cover_the_targets_in_order(lib, n, per):
    assert lib.check_passes(n, per) == 0


@pytest.mark.parametrize("n", [1, 7, 8, 9, 600_000, 2 ** 31 - 1])
def test_parts_are_near_equal(lib, n):
    for k in range(1, 9):
        b = [lib.begin(n, i, k) for i in range(k + 1)]
        assert b[0] == 0 and b[-1] == n
        sizes = {y - x for x, y in zip(b, b[1:])}
        assert max(sizes) - min(sizes) <= 1
