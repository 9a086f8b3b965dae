// gturbo_phases.cpp -- forcing phases (src/forcing.f90:16-24,40-51) on the
// host; plain C++, no HIP.
#include "gturbo_phases.hpp"

#include <cmath>

namespace gtr {

namespace {

// cos and sin at the nodes i/128 of [0, 2 pi], each as a double and its
// remainder from the extended-precision value (error below 2^-64).
struct Node {
  double ch, cl, sh, sl;
};
constexpr int kNodes = 6 * 128 + 64;  // beyond 2 pi * 128 = 804.2

struct Nodes {  // static storage: the C entries that draw must not throw
  Node v[kNodes];
  Nodes() noexcept {
    for (int i = 0; i < kNodes; ++i) {
      const long double a = (long double)i / 128.0L, c = cosl(a), s = sinl(a);
      v[i].ch = (double)c;
      v[i].cl = (double)(c - (long double)v[i].ch);
      v[i].sh = (double)s;
      v[i].sl = (double)(s - (long double)v[i].sh);
    }
  }
};
const Node* nodes() {
  static const Nodes t;
  return t.v;
}

void sincos_ext(double te, double* c, double* s) {
  *c = (double)cosl((long double)te);
  *s = (double)sinl((long double)te);
}

// h + lo, |lo| small, rounded to double; false when a neighbour of the sum
// within 2^-61 rounds to another double.
inline bool round_safe(double h, double lo, double* r) {
  constexpr double kEps = 0x1p-61;
  *r = h + lo;
  return h + (lo + kEps) == *r && h + (lo - kEps) == *r;
}

// (double)cosl(te), (double)sinl(te) for 0 <= te <= 6.3.  With te = A + d,
// A the nearest node (d exact, |d| <= 2^-8),
//   cos te = cos A - sin A d + [ -cos A (1 - cos d) + sin A (d - sin d) ]
// and sin te alike: the term in d as an exact product, the bracket (below
// 2^-16) in double, together within 2^-63.  Both values round the way the
// extended-precision ones do unless they lie within 2^-61 of a rounding
// boundary; those few (about 2% of the draws) take the extended functions.
__attribute__((target("fma"))) void sincos_fma(const Node* t, double te, double* c, double* s) {
  const int i = (int)(te * 128.0 + 0.5);
  const Node n = t[i];
  const double d = te - (double)i * 0.0078125;
  const double d2 = d * d;
  // 1 - cos d and d - sin d (Taylor, |d| <= 2^-8: next terms below 2^-80)
  const double vc = d2 * (0.5 - d2 * (1.0 / 24.0 - d2 * (1.0 / 720.0 - d2 / 40320.0)));
  const double vs = d * d2 * (1.0 / 6.0 - d2 * (1.0 / 120.0 - d2 * (1.0 / 5040.0)));
  bool ok;
  {
    const double p = n.sh * d, e = __builtin_fma(n.sh, d, -p);  // sin A d, exact p + e
    const double h = n.ch - p, b = n.ch - h;
    const double l = (n.ch - (h + b)) + (b - p);  // ch - p = h + l exactly
    ok = round_safe(h, l + (((n.cl - e) - n.sl * d) - n.ch * vc + n.sh * vs), c);
  }
  {
    const double p = n.ch * d, e = __builtin_fma(n.ch, d, -p);
    const double h = n.sh + p, b = h - n.sh;
    const double l = (n.sh - (h - b)) + (p - b);
    ok = round_safe(h, l + (((n.sl + e) + n.cl * d) - n.sh * vc - n.ch * vs), s) && ok;
  }
  if (!ok) sincos_ext(te, c, s);
}

}  // namespace

void forcing_phases(int nf, int32_t* seed, double* out) {
  static const bool fast = __builtin_cpu_supports("fma");
  const double pi2 = 2.0 * 3.14159265358979;
  const Node* t = nodes();
  uint32_t s = (uint32_t)*seed;
  for (int k = 0; k < nf; ++k) {
    s = (69069u * s + 1u) & 0x7FFFFFFFu;
    const float r = (float)((double)s / (double)0x7FFFFFFF);
    const double te = pi2 * (double)r;
    if (fast) sincos_fma(t, te, out + 2 * k, out + 2 * k + 1);
    else sincos_ext(te, out + 2 * k, out + 2 * k + 1);
  }
  *seed = (int32_t)s;
}

}  // namespace gtr
