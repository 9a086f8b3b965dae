"""The forcing phases of the library's host code against cosl/sinl rounded
once, bit for bit, over runs of the LCG from several seeds (CPU)."""
import ctypes as C
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "gturbo_amd", "csrc")

SHIM = r"""
#include <cmath>
#include <cstring>
#include <vector>
#include "gturbo_phases.hpp"
extern "C" long phases_differ(int nf, int32_t seed, int calls) {
  std::vector<double> o(2 * nf);
  long bad = 0;
  for (int c = 0; c < calls; ++c) {
    uint32_t s = (uint32_t)seed;
    gtr::forcing_phases(nf, &seed, o.data());
    for (int k = 0; k < nf; ++k) {
      s = (69069u * s + 1u) & 0x7FFFFFFFu;
      const float r = (float)((double)s / (double)0x7FFFFFFF);
      const double te = 2.0 * 3.14159265358979 * (double)r;
      const double x[2] = {(double)cosl((long double)te), (double)sinl((long double)te)};
      bad += std::memcmp(x, &o[2 * k], sizeof x) != 0;
    }
    bad += (int32_t)s != seed;
  }
  return bad;
}
"""


@pytest.fixture(scope="module")
def lib(tmp_path_factory):
    d = tmp_path_factory.mktemp("phases")
    src = d / "shim.cpp"
    src.write_text(SHIM)
    out = str(d / "phases.so")
    subprocess.run(["g++", "-O2", "-ffp-contract=off", "-shared", "-fPIC", f"-I{CSRC}", str(src),
                    os.path.join(CSRC, "gturbo_phases.cpp"), "-o", out], check=True)
    return C.CDLL(out)


# 400000 draws from each seed (the largest seed and a negative one among them)
@pytest.mark.parametrize("seed", [481929, 1, 0x7FFFFFFF, -5, 90071])
def test_phases_equal_rounded_extended_values(lib, seed):
    lib.phases_differ.restype = C.c_long
    assert lib.phases_differ(400, C.c_int32(seed), 1000) == 0
