"""Twiddle rounding of the in-place lines on the CPU: fft_core.hpp compiled for
the host, the factors that its passes apply against extended precision.

A twiddle's error is the same in every transform and so adds up over a run.
To first order a transform's relative error from it is the root of the sum over
the passes of the mean square error of the factors.  The bar: an in-place line
has no more of it than the Stockham line of its size."""
import ctypes as C
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "gturbo_amd", "csrc")

HIP = r"""
#pragma once
#include <cmath>
#define __device__
#define __host__
#define __forceinline__ inline
#define __builtin_amdgcn_fence(a, b)
#define __builtin_amdgcn_wave_barrier()
struct double2 { double x, y; };
inline double2 make_double2(double x, double y) { return {x, y}; }
inline void __syncthreads() {}
using std::fma;
"""

SRC = r"""
#include <hip/hip_runtime.h>
#include <vector>
#include "fft_core.hpp"
using namespace gt;
static double err2(double2 w, long m, long n) {  // |w - exp(-2 pi i m / n)|^2
  const long double a = 6.283185307179586476925286766559005768L * (m % n) / n;
  const long double x = w.x - cosl(a), y = w.y + sinl(a);
  return (double)(x * x + y * y);
}
static std::vector<double2> table(int n) {
  std::vector<double2> t(n);
  for (int m = 0; m < n; ++m) {
    const long double a = 6.283185307179586476925286766559005768L * m / n;
    t[m] = {(double)cosl(a), -(double)sinl(a)};
  }
  return t;
}
static const double2 one = {1.0, 0.0};
// Mean square errors of the passes of a Stockham line, added up.
template <int R>
static double stockham(int n, int ns, const double2* tw) {
  double s = 0;
  for (int k = 0; k < ns; ++k) {
    double2 t[8] = {one, one, one, one, one, one, one, one};
    apply_tw<R, -1>(t, tw[k * (n / (ns * R))]);
    for (int r = 0; r < R; ++r) s += err2(t[r], (long)k * r, (long)ns * R);
  }
  return s / (ns * R);
}
template <int L>
static double stockham_line() {
  constexpr int N = 1 << L, RL = Line<L>::RLAST;
  const auto tw = table(N);
  double s = 0;
  int ns = 8;
  for (int i = 1; i < Line<L>::NPASS8; ++i, ns *= 8) s += stockham<8>(N, ns, tw.data());
  if constexpr (RL > 1) s += stockham<RL>(N, ns, tw.data());
  return sqrt(s);
}
template <int L>
static double in_place_line() {
  constexpr int N = 1 << L, T = N / 8;
  const auto tab = table(N);
  double s = 0;
  for (int j = 0; j < T; ++j) {
    const TwFromTable<L, 1> tw{tab.data(), j};
    double2 t[3][8];
    for (auto& p : t)
      for (auto& x : p) x = one;
    apply_tw8<-1>(t[0], tw.template at<1>());
    apply_tw8<-1>(t[1], tw.template at<2>());
    apply_tw8<-1>(t[2], ip_third<L>(tw.template at<3>(), j));
    const int k[3] = {j, 8 * (j & (T / 8 - 1)), 64 * (j & (T / 64 - 1))};
    for (int p = 0; p < 3; ++p)
      for (int r = 0; r < 8; ++r) s += err2(t[p][r], (long)k[p] * r, N);
  }
  return sqrt(s / N);
}
extern "C" double line_error(int logn, int in_place) {
  switch (logn) {
    case 10: return in_place ? in_place_line<10>() : stockham_line<10>();
    case 11: return in_place ? in_place_line<11>() : stockham_line<11>();
    default: return in_place ? in_place_line<12>() : stockham_line<12>();
  }
}
"""


@pytest.fixture(scope="module")
def line_error(tmp_path_factory):
    d = tmp_path_factory.mktemp("twiddles")
    (d / "hip").mkdir()
    (d / "hip" / "hip_runtime.h").write_text(HIP)
    (d / "tw.cpp").write_text(SRC)
    out = str(d / "tw.so")
    subprocess.run(["g++", "-std=c++17", "-O1", "-ffp-contract=off", "-shared", "-fPIC", "-w",
                    f"-I{d}", f"-I{CSRC}", str(d / "tw.cpp"), "-o", out], check=True)
    f = C.CDLL(out).line_error
    f.restype = C.c_double
    return f


@pytest.mark.parametrize("logn", [10, 11, 12])
def test_in_place_line_has_no_more_twiddle_error(line_error, logn):
    """1e-17 a line is one rounding of a factor in a hundred."""
    assert 0 < line_error(logn, 1) <= line_error(logn, 0) + 1e-17
