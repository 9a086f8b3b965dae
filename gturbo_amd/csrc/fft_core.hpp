// fft_core.hpp -- FP64 complex FFT building blocks for gfx950.
//
// A line of N = 2^LOGN complex doubles is spread over TPL = N/8 threads:
// thread j holds a[r] = x[j + TPL*r], r = 0..7, in registers, before and
// after the transform.  The transform is a Stockham sequence of radix-8
// passes (plus one radix-2 or radix-4 pass when log2 N is not a multiple of
// 3).  Every pass reads exactly that per-thread set; the last pass
// (Ns*R = N) writes it back in natural order, so only the transposes between
// passes go through LDS (one padded line per transform: element e sits at
// e + e/16, which spreads the strided writes over the banks).
//
// Eight elements per thread keep a transform at 32 VGPRs of data per lane,
// which lets the passes that carry a second field run at 4 waves per SIMD.
//
// Twiddles come from a table W[m] = exp(-2 pi i m / N), m < N, built on the
// host in extended precision and rounded once.  A butterfly loads only W^k
// and forms W^2k ... W^7k by complex products (at most four extra
// roundings): on gfx950 these passes are bound by memory-instruction
// latency, not by FP64 arithmetic, and one load per butterfly measured
// faster than three (and three faster than seven).
#pragma once
#include <type_traits>
#include <hip/hip_runtime.h>

namespace gt {

constexpr int kE = 8;  // complex elements per thread and line

__device__ __forceinline__ double2 cadd(double2 a, double2 b) {
  return make_double2(a.x + b.x, a.y + b.y);
}
__device__ __forceinline__ double2 csub(double2 a, double2 b) {
  return make_double2(a.x - b.x, a.y - b.y);
}
// Products with explicit fused multiply-adds.  The kernels are compiled
// without automatic contraction (-ffp-contract=off), so each product rounds
// the same way in every kernel it is inlined into: a member of a batched
// run and the same run alone give bit-identical fields.
__device__ __forceinline__ double2 cmul(double2 a, double2 b) {
  return make_double2(fma(a.x, b.x, -a.y * b.y), fma(a.x, b.y, a.y * b.x));
}
// a * conj(b)
__device__ __forceinline__ double2 cmulc(double2 a, double2 b) {
  return make_double2(fma(a.x, b.x, a.y * b.y), fma(a.y, b.x, -a.x * b.y));
}
// a * (i*S), S = +-1
template <int S>
__device__ __forceinline__ double2 mul_is(double2 a) {
  return S > 0 ? make_double2(-a.y, a.x) : make_double2(a.y, -a.x);
}

constexpr double kR2 = 0.70710678118654752440;  // cos(pi/4)

// a * exp(S*2*pi*i*M/8)
template <int S, int M>
__device__ __forceinline__ double2 w8(double2 a) {
  constexpr int m = M & 7;
  if constexpr (m == 0) return a;
  else if constexpr (m == 2) return mul_is<S>(a);
  else if constexpr (m == 4) return make_double2(-a.x, -a.y);
  else if constexpr (m == 6) return mul_is<-S>(a);
  else {
    constexpr double c = (m == 1 || m == 7) ? kR2 : -kR2;
    constexpr double s0 = (m == 1 || m == 3) ? kR2 : -kR2;
    constexpr double s = S > 0 ? s0 : -s0;
    return make_double2(fma(a.x, c, -a.y * s), fma(a.x, s, a.y * c));
  }
}

template <int S>
__device__ __forceinline__ void dft2(double2& a0, double2& a1) {
  double2 t = csub(a0, a1);
  a0 = cadd(a0, a1);
  a1 = t;
}

template <int S>
__device__ __forceinline__ void dft4(double2& a0, double2& a1, double2& a2,
                                     double2& a3) {
  double2 b0 = cadd(a0, a2), b1 = csub(a0, a2);
  double2 b2 = cadd(a1, a3), b3 = mul_is<S>(csub(a1, a3));
  a0 = cadd(b0, b2);
  a1 = cadd(b1, b3);
  a2 = csub(b0, b2);
  a3 = csub(b1, b3);
}

// Radix-8 as 4 x 2 (n = 2 n1 + n2, k = k1 + 4 k2), natural-order output.
template <int S>
__device__ __forceinline__ void dft8(double2* a) {
  dft4<S>(a[0], a[2], a[4], a[6]);
  dft4<S>(a[1], a[3], a[5], a[7]);
  a[3] = w8<S, 1>(a[3]);
  a[5] = w8<S, 2>(a[5]);
  a[7] = w8<S, 3>(a[7]);
  double2 y[8];
#pragma unroll
  for (int k1 = 0; k1 < 4; ++k1) {
    y[k1] = cadd(a[2 * k1], a[2 * k1 + 1]);
    y[k1 + 4] = csub(a[2 * k1], a[2 * k1 + 1]);
  }
#pragma unroll
  for (int i = 0; i < 8; ++i) a[i] = y[i];
}

template <int R, int S>
__device__ __forceinline__ void dft(double2* a) {
  if constexpr (R == 2) dft2<S>(a[0], a[1]);
  else if constexpr (R == 4) dft4<S>(a[0], a[1], a[2], a[3]);
  else dft8<S>(a);
}

__device__ __forceinline__ int lpad(int e) { return e + (e >> 4); }
// lpad(e + c) - lpad(e) for a power-of-two-aligned run: valid whenever c is a
// multiple of a power of two P and e mod P + c lies in the same 16-element
// block as c (the transposes below only form such sums), so one base address
// per thread plus compile-time offsets replaces a padded index per access.
__host__ __device__ constexpr int lpad_off(int c) { return c + c / 16; }

template <int LOGN>
struct Line {
  static constexpr int N = 1 << LOGN;
  static constexpr int TPL = N / kE;          // threads per line
  static constexpr int PADDED = N + N / 16;   // double2 per line in LDS
  static constexpr int NPASS8 = LOGN / 3;     // radix-8 passes
  static constexpr int RLAST = 1 << (LOGN % 3);  // trailing radix (1 = none)
};

// Entries of the twiddle table the passes of a line read: W^(k Ns') with
// k Ns' < N/8 for the radix-8 passes and < N/R for a trailing radix-R pass.
template <int LOGN>
constexpr int tw_span() {
  return (1 << LOGN) / (Line<LOGN>::RLAST > 1 ? Line<LOGN>::RLAST : 8);
}
// Up to N = 4096 the kernels keep that part of the table in LDS (at most
// 512 entries, beside their line buffers); larger lines read it from memory.
template <int LOGN>
constexpr bool tw_in_lds() { return LOGN <= 12; }
template <int LOGN>
constexpr int tw_lds_size() { return tw_in_lds<LOGN>() ? tw_span<LOGN>() : 1; }

// Copies the table's first tw_span entries to LDS (every thread of the
// workgroup calls it; ends with a barrier) and returns the table the
// transforms should read.
template <int LOGN>
__device__ __forceinline__ const double2* stage_tw(double2* twl, const double2* __restrict__ tw,
                                                   int tid, int nthr) {
  if constexpr (tw_in_lds<LOGN>()) {
    for (int i = tid; i < tw_span<LOGN>(); i += nthr) twl[i] = tw[i];
    __syncthreads();
    return twl;
  } else {
    return tw;
  }
}

// Orders a wave's LDS writes before its later reads (LDS executes one wave's
// operations in order; this keeps the compiler from moving them).
__device__ __forceinline__ void wave_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// t[r] *= W^(r k) (conjugated for S > 0), r < R, from w1 = W^k.
template <int R, int S>
__device__ __forceinline__ void apply_tw(double2* t, double2 w1) {
  double2 w[R];
  w[1] = w1;
  if constexpr (R >= 4) {
    w[2] = cmul(w[1], w[1]);
    w[3] = cmul(w[1], w[2]);
  }
  if constexpr (R == 8) {
    w[4] = cmul(w[2], w[2]);
    w[5] = cmul(w[1], w[4]);
    w[6] = cmul(w[2], w[4]);
    w[7] = cmul(w[3], w[4]);
  }
#pragma unroll
  for (int r = 1; r < R; ++r) t[r] = S < 0 ? cmul(t[r], w[r]) : cmulc(t[r], w[r]);
}

// One Stockham pass: radix R, stride Ns.  Butterfly jj (< N/R) reads
// x[jj + (N/R) r'] and writes y[(jj/Ns) Ns R + jj%Ns + Ns r'].
template <int LOGN, int S, int R, int NS, bool LAST>
__device__ __forceinline__ void reg_pass(double2* a, double2* buf, int j, const double2* tw) {
  constexpr int N = 1 << LOGN;
  constexpr int TPL = N / kE;
  constexpr int NB = kE / R;  // butterflies per thread
  // Opaque copy of the thread index: the addresses below are then computed
  // inside each pass instead of being shared (and kept live) across every
  // transform of the kernel.
  asm volatile("" : "+v"(j));
#pragma unroll
  for (int b = 0; b < NB; ++b) {
    const int jj = j + TPL * b;
    const int k = jj % NS;
    double2 t[R];
#pragma unroll
    for (int r = 0; r < R; ++r) t[r] = a[b + NB * r];
    if constexpr (NS > 1) {
      constexpr int ST = N / (NS * R);
      apply_tw<R, S>(t, tw[k * ST]);
    }
    dft<R, S>(t);
    if constexpr (LAST) {
#pragma unroll
      for (int r = 0; r < R; ++r) a[b + NB * r] = t[r];
    } else {
      // idx = (jj/NS) NS R + k with k < NS: idx + r NS never crosses into
      // another 16-element block than r NS does, so lpad splits.
      double2* p = buf + lpad((jj / NS) * NS * R + k);
#pragma unroll
      for (int r = 0; r < R; ++r) p[lpad_off(r * NS)] = t[r];
    }
  }
  if constexpr (!LAST) {
    __syncthreads();
    const double2* p = buf + lpad(j);  // j < TPL, TPL a power of two
#pragma unroll
    for (int r = 0; r < kE; ++r) a[r] = p[lpad_off(TPL * r)];
    __syncthreads();
  }
}

// Transform of one line held in registers; S = -1 forward, +1 inverse
// (unnormalised).  Every thread of the workgroup must call it (the
// transposes hold barriers); j is the thread's index within its line.
// SCHED picks the radix order when log2 N is not a multiple of 3: 0 runs
// the radix-8 passes first and the radix-2/4 pass last, 1 the other way
// round (same result up to rounding; the faster one depends on N).
template <int LOGN, int S, int SCHED = 0>
__device__ __forceinline__ void fft_reg(double2* a, double2* buf, int j, const double2* tw) {
  using L = Line<LOGN>;
  constexpr int NP = L::NPASS8 + (L::RLAST > 1 ? 1 : 0);
  constexpr int P8 = L::NPASS8;
  if constexpr (SCHED == 0 || L::RLAST == 1) {
    if constexpr (P8 >= 1) reg_pass<LOGN, S, 8, 1, NP == 1>(a, buf, j, tw);
    if constexpr (P8 >= 2) reg_pass<LOGN, S, 8, 8, NP == 2>(a, buf, j, tw);
    if constexpr (P8 >= 3) reg_pass<LOGN, S, 8, 64, NP == 3>(a, buf, j, tw);
    if constexpr (P8 >= 4) reg_pass<LOGN, S, 8, 512, NP == 4>(a, buf, j, tw);
    if constexpr (L::RLAST > 1) reg_pass<LOGN, S, L::RLAST, 1 << (3 * P8), true>(a, buf, j, tw);
  } else {
    constexpr int R0 = L::RLAST;
    reg_pass<LOGN, S, R0, 1, NP == 1>(a, buf, j, tw);
    if constexpr (P8 >= 1) reg_pass<LOGN, S, 8, R0, NP == 2>(a, buf, j, tw);
    if constexpr (P8 >= 2) reg_pass<LOGN, S, 8, R0 * 8, NP == 3>(a, buf, j, tw);
    if constexpr (P8 >= 3) reg_pass<LOGN, S, 8, R0 * 64, NP == 4>(a, buf, j, tw);
    if constexpr (P8 >= 4) reg_pass<LOGN, S, 8, R0 * 512, NP == 5>(a, buf, j, tw);
  }
}

// ---------------------------------------------------------------------------
// The same Stockham transform with the thread's twiddles in registers: one
// W^k per radix-8 pass after the first and one per butterfly of a trailing
// radix-2/4 pass, the same for every transform the thread runs, so a kernel
// loads them once, beside its data, and stages no table.  Same operations
// and roundings as fft_reg with SCHED 0.  For lines inside one wave (N <=
// 512: at most 64 threads, N/8 dividing the wave): the transposes need no
// workgroup barrier, and a line's threads may call alone.
// ---------------------------------------------------------------------------
template <int LOGN>
struct HeldTw {
  using L = Line<LOGN>;
  static constexpr int NB = L::RLAST > 1 ? kE / L::RLAST : 0;  // last-pass butterflies
  static constexpr int K = L::NPASS8 - 1 + NB;
  double2 w[K > 0 ? K : 1];
};
template <int LOGN>
__device__ __forceinline__ HeldTw<LOGN> held_tw(const double2* __restrict__ tw, int j) {
  using L = Line<LOGN>;
  HeldTw<LOGN> h;
#pragma unroll
  for (int i = 1; i < L::NPASS8; ++i) {
    const int ns = 1 << (3 * i);
    h.w[i - 1] = tw[(j % ns) * (L::N / (ns * 8))];
  }
#pragma unroll
  for (int b = 0; b < HeldTw<LOGN>::NB; ++b)
    h.w[L::NPASS8 - 1 + b] = tw[(j + L::TPL * b) % (1 << (3 * L::NPASS8))];
  return h;
}
template <int LOGN>
constexpr bool line_in_wave() { return Line<LOGN>::TPL <= 64; }
template <int LOGN, int S, int R, int NS, bool LAST>
__device__ __forceinline__ void held_pass(double2* a, double2* buf, int j, const double2* w) {
  constexpr int N = 1 << LOGN;
  constexpr int TPL = N / kE;
  constexpr int NB = kE / R;
#pragma unroll
  for (int b = 0; b < NB; ++b) {
    const int jj = j + TPL * b;
    double2 t[R];
#pragma unroll
    for (int r = 0; r < R; ++r) t[r] = a[b + NB * r];
    if constexpr (NS > 1) apply_tw<R, S>(t, w[b]);
    dft<R, S>(t);
    if constexpr (LAST) {
#pragma unroll
      for (int r = 0; r < R; ++r) a[b + NB * r] = t[r];
    } else {
      double2* p = buf + lpad((jj / NS) * NS * R + jj % NS);
#pragma unroll
      for (int r = 0; r < R; ++r) p[lpad_off(r * NS)] = t[r];
    }
  }
  if constexpr (!LAST) {
    wave_sync();
    const double2* p = buf + lpad(j);
#pragma unroll
    for (int r = 0; r < kE; ++r) a[r] = p[lpad_off(TPL * r)];
    wave_sync();
  }
}
template <int LOGN, int S>
__device__ __forceinline__ void fft_held(double2* a, double2* buf, int j,
                                         const HeldTw<LOGN>& h) {
  using L = Line<LOGN>;
  static_assert(line_in_wave<LOGN>(), "a line inside a wave");
  constexpr int P8 = L::NPASS8;
  constexpr bool T = L::RLAST > 1;
  held_pass<LOGN, S, 8, 1, P8 == 1 && !T>(a, buf, j, h.w);
  if constexpr (P8 >= 2) held_pass<LOGN, S, 8, 8, P8 == 2 && !T>(a, buf, j, h.w);
  if constexpr (P8 >= 3) held_pass<LOGN, S, 8, 64, P8 == 3 && !T>(a, buf, j, h.w + 1);
  if constexpr (T)
    held_pass<LOGN, S, L::RLAST, (1 << (3 * P8)), true>(a, buf, j, h.w + P8 - 1);
}

// ---------------------------------------------------------------------------
// In-place radix-8 transforms of a 1024-, 2048- or 4096-point line over T =
// N/8 threads (whole waves, thread j = lane + 64 wave).  The first pass combines
// the elements j + T r that thread j holds; its outputs go to LDS, and each
// later pass reads, transforms and writes back one run of the line that
// belongs to a single wave (strides T/8 and T/64: runs inside the wave's 512
// elements; the last pass eight consecutive ones, as one radix-8 butterfly at
// 4096, two radix-4 ones at 2048, four radix-2 ones at 1024).  Only the first exchange crosses waves,
// so a transform needs one workgroup barrier plus one before its first write
// (when LDS may still be read by another wave), instead of two per pass.
//   fft_dif: natural order in, out of order: thread j, register r holds
//            X[ip_row(j, r)] (the digits of 8 j + r reversed; at 4096
//            D(j) + 512 r with D the octal digit reversal of j).
//   fft_dit: the transposed algorithm (same twiddles, applied before each
//            radix-8 DFT, passes in reverse): input in that order, natural
//            order out.
// LDS element e sits at e + e/8: every pass then addresses one base per
// thread plus constants, and a wave's accesses at stride 8 or 9 spread over
// the banks.
// ---------------------------------------------------------------------------
template <int LOGN>
constexpr int ip_line() { return (1 << LOGN) + (1 << LOGN) / 8; }  // double2 in LDS
constexpr int kIpLine = ip_line<12>();

__device__ __forceinline__ int ip_pad(int e) { return e + (e >> 3); }

// Output index of fft_dif in thread j, register r.
template <int LOGN>
__host__ __device__ __forceinline__ int ip_row(int j, int r) {
  static_assert(LOGN >= 10 && LOGN <= 12, "in-place lines of 1024 to 4096 points");
  if constexpr (LOGN == 12)
    return 64 * (j & 7) + 8 * ((j >> 3) & 7) + (j >> 6) + 512 * r;
  else if constexpr (LOGN == 11)
    return (j >> 5) + 8 * ((j >> 2) & 7) + 128 * (j & 3) + 64 * (r >> 2) + 512 * (r & 3);
  else
    return (j >> 4) + 8 * ((j >> 1) & 7) + 256 * (j & 1) + 64 * (r >> 1) + 512 * (r & 1);
}

// t[r] *= W^(k r) (conjugated for S > 0), from w1 = W^k; each power is
// applied as soon as it is formed (at most four live at a time).
template <int S>
__device__ __forceinline__ void apply_tw8(double2* t, double2 w1) {
  auto ap = [](double2& x, double2 w) { x = S < 0 ? cmul(x, w) : cmulc(x, w); };
  ap(t[1], w1);
  const double2 w2 = cmul(w1, w1);
  ap(t[2], w2);
  const double2 w3 = cmul(w1, w2);
  ap(t[3], w3);
  const double2 w4 = cmul(w2, w2);
  ap(t[4], w4);
  ap(t[5], cmul(w1, w4));
  ap(t[6], cmul(w2, w4));
  ap(t[7], cmul(w3, w4));
}

// The same from W^k and W^4k, both of the table.  A twiddle's error is the
// same in every transform, so it adds up over a run where roundings of data
// do not: 1024 points, whose three passes form seven powers each where the
// Stockham passes formed them in two, take W^4k from the table too (1024^2
// SQG, 100 steps: difference to the oracle 1.1e-15; from W^k alone 1.6e-15,
// Stockham 2.4e-15; exact twiddles 0.8e-15), for 3 us of a 1024^2 RK4 step:
// 130 -> 133, Stockham 139.
struct W14 {
  double2 w1, w4;
};
template <int S>
__device__ __forceinline__ void apply_tw8(double2* t, const W14& w) {
  auto ap = [](double2& x, double2 v) { x = S < 0 ? cmul(x, v) : cmulc(x, v); };
  ap(t[1], w.w1);
  ap(t[4], w.w4);
  ap(t[5], cmul(w.w1, w.w4));
  const double2 w2 = cmul(w.w1, w.w1);
  ap(t[2], w2);
  ap(t[6], cmul(w2, w.w4));
  const double2 w3 = cmul(w.w1, w2);
  ap(t[3], w3);
  ap(t[7], cmul(w3, w.w4));
}
template <int LOGN>
using ip_w = std::conditional_t<LOGN == 10, W14, double2>;

// The twiddle of pass 3 as it is applied.  2048 points: W^k with W^4k =
// exp(-2 pi i (j % 4) / 8) from constants, so that no register is held for it
// and the table in LDS stays at its 512 entries.  Three passes of seven powers
// from W^k alone have more twiddle error than the Stockham line's two and a
// radix-4 one (3.02e-16 a line against 2.67e-16); with this third pass 2.57e-16
// (4096: 3.15e-16 both).  2048^2, 400 steps, distance to 64-bit transforms:
// alpha 1 5.96e-15 -> 5.87e-15, Stockham 6.43e-15; y stages 43.9, 42.9, 43.5 us
// (alpha 1/2) and the x pass 32.8 as before, step boundary 46.4 -> 47.7.
template <int LOGN>
__device__ __forceinline__ auto ip_third(const ip_w<LOGN>& w, int j) {
  if constexpr (LOGN == 11) {
    const int k = j & 3;
    const double c = k & 1 ? kR2 : 0.0;
    return W14{w, make_double2(k == 0 ? 1.0 : k == 3 ? -c : c, k == 2 ? -1.0 : -c)};
  } else {
    return w;
  }
}

// Twiddles of the three twiddled passes of an in-place transform in thread
// j: W^j (stride T), W^(8 (j % (T/8))), W^(64 (j % (T/64))), from the table
// read at stride TS.  The same for every transform a thread runs, so a kernel
// running several may load them once.
template <int LOGN>
struct IpTw {
  ip_w<LOGN> w1, w2, w3;
};
// Twiddle sources for fft_dif / fft_dit: at<P>() gives the twiddle of pass P
// (1-3), called where the transform first needs it in flight.
template <int LOGN, int TS>
struct TwFromTable {
  static constexpr int T = (1 << LOGN) / 8;
  const double2* __restrict__ tw;
  int j;
  template <int P>
  __device__ __forceinline__ ip_w<LOGN> at() const {
    const int k = P == 1 ? j : P == 2 ? 8 * (j & (T / 8 - 1)) : 64 * (j & (T / 64 - 1));
    if constexpr (LOGN == 10) return {tw[TS * k], tw[TS * 4 * k]};
    else return tw[TS * k];
  }
};
template <int LOGN, int TS = 1>
__device__ __forceinline__ IpTw<LOGN> ip_tw(const double2* __restrict__ tw, int j) {
  const TwFromTable<LOGN, TS> t{tw, j};
  return {t.template at<1>(), t.template at<2>(), t.template at<3>()};
}
template <int LOGN>
struct TwHeld {
  const IpTw<LOGN>& w;
  template <int P>
  __device__ __forceinline__ ip_w<LOGN> at() const {
    return P == 1 ? w.w1 : P == 2 ? w.w2 : w.w3;
  }
};

// Runs of passes 2 and 3 in LDS: thread j's first element and the padded
// distance of its r-th one.
template <int LOGN>
struct IpRun {
  static constexpr int T = (1 << LOGN) / 8, S2 = T / 8, S3 = T / 64;
  static __device__ __forceinline__ int base2(int j) {
    return ip_pad((j / S2) * T + (j & (S2 - 1)));
  }
  static __device__ __forceinline__ int base3(int j) {
    return ip_pad((j / S3) * S2 + (j & (S3 - 1)));
  }
  static constexpr int off1(int r) { return T * r + T * r / 8; }
  static constexpr int off2(int r) { return S2 * r + S2 * r / 8; }
  static constexpr int off3(int r) { return S3 * r + S3 * r / 8; }
};
// Last (stride 1) pass on the thread's eight consecutive elements.
template <int LOGN, int S>
__device__ __forceinline__ void ip_last(double2* a) {
  if constexpr (LOGN == 12) {
    dft<8, S>(a);
  } else if constexpr (LOGN == 11) {
    dft<4, S>(a);
    dft<4, S>(a + 4);
  } else {
#pragma unroll
    for (int r = 0; r < 8; r += 2) dft<2, S>(a + r);
  }
}

// bar: barrier before the first LDS write (another wave may still read
// LDS); a uniform run-time flag, so that a loop holds one copy of the code.
// act = false (uniform in a wave): the wave only meets the barriers.
template <int LOGN, int S, class TW>
__device__ __forceinline__ void fft_dif_t(double2* a, double2* buf, int j, const TW& T,
                                          bool bar, bool act = true) {
  using R = IpRun<LOGN>;
  ip_w<LOGN> wn;
  if (act) {
    wn = T.template at<1>();  // pass 1: W^(j r)
    dft<8, S>(a);
    apply_tw8<S>(a, wn);
    wn = T.template at<2>();  // pass 2, in flight across the barrier
  }
  if (bar) __syncthreads();
  if (act) {
    double2* p = buf + ip_pad(j);
#pragma unroll
    for (int r = 0; r < 8; ++r) p[R::off1(r)] = a[r];
  }
  __syncthreads();
  if (!act) return;
  {  // pass 2
    double2* p = buf + R::base2(j);
#pragma unroll
    for (int r = 0; r < 8; ++r) a[r] = p[R::off2(r)];
    dft<8, S>(a);
    apply_tw8<S>(a, wn);
    wn = T.template at<3>();
#pragma unroll
    for (int r = 0; r < 8; ++r) p[R::off2(r)] = a[r];
  }
  wave_sync();
  {  // pass 3
    double2* p = buf + R::base3(j);
#pragma unroll
    for (int r = 0; r < 8; ++r) a[r] = p[R::off3(r)];
    dft<8, S>(a);
    apply_tw8<S>(a, ip_third<LOGN>(wn, j));
#pragma unroll
    for (int r = 0; r < 8; ++r) p[R::off3(r)] = a[r];
  }
  wave_sync();
  {  // pass 4, stride 1
    const double2* p = buf + 9 * j;  // ip_pad(8 j)
#pragma unroll
    for (int r = 0; r < 8; ++r) a[r] = p[r];
    ip_last<LOGN, S>(a);
  }
}
template <int S, int TS = 1, int LOGN = 12>
__device__ __forceinline__ void fft_dif(double2* a, double2* buf, int j,
                                        const double2* __restrict__ tw, bool bar) {
  asm volatile("" : "+v"(j));
  fft_dif_t<LOGN, S>(a, buf, j, TwFromTable<LOGN, TS>{tw, j}, bar);
}
// Held twiddles enter each transform opaque, so that the compiler keeps
// forming the powers inside it rather than holding them across transforms.
__device__ __forceinline__ void hide(double2& w) { asm volatile("" : "+v"(w.x), "+v"(w.y)); }
__device__ __forceinline__ void hide(W14& w) {
  hide(w.w1);
  hide(w.w4);
}
template <int LOGN>
__device__ __forceinline__ IpTw<LOGN> opaque(IpTw<LOGN> w) {
  hide(w.w1);
  hide(w.w2);
  hide(w.w3);
  return w;
}
template <int LOGN, int S>
__device__ __forceinline__ void fft_dif_held(double2* a, double2* buf, int j,
                                             const IpTw<LOGN>& w,
                                             bool bar, bool act = true) {
  asm volatile("" : "+v"(j));
  const IpTw<LOGN> lw = opaque(w);
  fft_dif_t<LOGN, S>(a, buf, j, TwHeld<LOGN>{lw}, bar, act);
}

// Input as fft_dif leaves it; the thread's own LDS run is free to write
// (its last reader was this wave).  Ends after reads of every wave's
// elements: a barrier must precede the next LDS write.
// BAR: start with a workgroup barrier (another wave may still read this
// wave's run of LDS, e.g. after a preceding fft_dit).
template <int LOGN, int S, bool BAR, class TW>
__device__ __forceinline__ void fft_dit_t(double2* a, double2* buf, int j, const TW& T,
                                          bool act = true) {
  using R = IpRun<LOGN>;
  ip_w<LOGN> wn;
  if (act) {
    wn = T.template at<3>();
    ip_last<LOGN, S>(a);  // pass 4, stride 1
  }
  if constexpr (BAR) __syncthreads();
  if (act) {
    {
      double2* p = buf + 9 * j;
#pragma unroll
      for (int r = 0; r < 8; ++r) p[r] = a[r];
    }
    wave_sync();
    {  // pass 3
      double2* p = buf + R::base3(j);
#pragma unroll
      for (int r = 0; r < 8; ++r) a[r] = p[R::off3(r)];
      apply_tw8<S>(a, ip_third<LOGN>(wn, j));
      wn = T.template at<2>();
      dft<8, S>(a);
#pragma unroll
      for (int r = 0; r < 8; ++r) p[R::off3(r)] = a[r];
    }
    wave_sync();
    {  // pass 2
      double2* p = buf + R::base2(j);
#pragma unroll
      for (int r = 0; r < 8; ++r) a[r] = p[R::off2(r)];
      apply_tw8<S>(a, wn);
      wn = T.template at<1>();
      dft<8, S>(a);
#pragma unroll
      for (int r = 0; r < 8; ++r) p[R::off2(r)] = a[r];
    }
  }
  __syncthreads();
  if (act) {  // pass 1: natural order out
    const double2* p = buf + ip_pad(j);
#pragma unroll
    for (int r = 0; r < 8; ++r) a[r] = p[R::off1(r)];
    apply_tw8<S>(a, wn);
    dft<8, S>(a);
  }
}
template <int S, bool BAR = false, int TS = 1, int LOGN = 12>
__device__ __forceinline__ void fft_dit(double2* a, double2* buf, int j,
                                        const double2* __restrict__ tw) {
  asm volatile("" : "+v"(j));
  fft_dit_t<LOGN, S, BAR>(a, buf, j, TwFromTable<LOGN, TS>{tw, j});
}
template <int LOGN, int S, bool BAR = false>
__device__ __forceinline__ void fft_dit_held(double2* a, double2* buf, int j,
                                             const IpTw<LOGN>& w,
                                             bool act = true) {
  asm volatile("" : "+v"(j));
  const IpTw<LOGN> lw = opaque(w);
  fft_dit_t<LOGN, S, BAR>(a, buf, j, TwHeld<LOGN>{lw}, act);
}

// 8192-point lines over 1024 threads (thread t holds x[t + 1024 r]): a
// radix-2 pass (stride 4096) on the thread's own elements splits the line
// into two 4096-point problems, one exchange hands problem h to threads
// 512h..512h+511 in natural order, and each half runs the in-place
// transform above with the 8192-point table read at stride 2.  fft_dif2
// leaves thread (h, j), register r with X[2 (D(j) + 512 r) + h]; fft_dit2
// takes that order and returns natural order.  buf: two kIpLine regions.
template <int S>
__device__ __forceinline__ void fft_dif2(double2* a, double2* buf, int t,
                                         const double2* __restrict__ tw, bool bar) {
  asm volatile("" : "+v"(t));
#pragma unroll
  for (int r = 0; r < 4; ++r) {  // Y0[n] = x[n] + x[n+4096], Y1[n] = (x[n] - x[n+4096]) W^n
    const double2 d = csub(a[r], a[r + 4]);
    a[r] = cadd(a[r], a[r + 4]);
    const double2 w = tw[t + 1024 * r];
    a[r + 4] = S < 0 ? cmul(d, w) : cmulc(d, w);
  }
  if (bar) __syncthreads();
#pragma unroll
  for (int r = 0; r < 8; ++r)  // Y_(r/4)[t + 1024 (r%4)] into region r/4
    buf[(r >> 2) * kIpLine + ip_pad(t + 1024 * (r & 3))] = a[r];
  __syncthreads();
  const int j = t & 511;
  double2* hb = buf + (t >> 9) * kIpLine;
  {
    const double2* p = hb + ip_pad(j);
#pragma unroll
    for (int r = 0; r < 8; ++r) a[r] = p[576 * r];  // ip_pad(j + 512 r)
  }
  // the first pass of fft_dif writes back exactly the positions just read
  fft_dif<S, 2>(a, hb, j, tw, false);
}

// Ends after reads of every wave's elements: a barrier must precede the
// next LDS write.  BAR: start with a barrier (another wave may still read
// this wave's run, e.g. after a preceding fft_dit2).
template <int S, bool BAR = false>
__device__ __forceinline__ void fft_dit2(double2* a, double2* buf, int t,
                                         const double2* __restrict__ tw) {
  asm volatile("" : "+v"(t));
  const int j = t & 511;
  double2* hb = buf + (t >> 9) * kIpLine;
  fft_dit<S, BAR, 2>(a, hb, j, tw);  // natural order within the half
  {
    double2* p = hb + ip_pad(j);  // the positions fft_dit's last pass read
#pragma unroll
    for (int r = 0; r < 8; ++r) p[576 * r] = a[r];
  }
  __syncthreads();
#pragma unroll
  for (int r = 0; r < 4; ++r) {  // x[n] = Y0[n] + W^n Y1[n], x[n+4096] = Y0[n] - W^n Y1[n]
    const int e = ip_pad(t + 1024 * r);
    const double2 y0 = buf[e];
    const double2 w = tw[t + 1024 * r];
    const double2 y1 = S < 0 ? cmul(buf[kIpLine + e], w) : cmulc(buf[kIpLine + e], w);
    a[r] = cadd(y0, y1);
    a[r + 4] = csub(y0, y1);
  }
}

// ---------------------------------------------------------------------------
// 4096-point lines over 256 threads, sixteen elements each (thread j holds
// x[j + 256 r]): three radix-16 passes (strides 256, 16, 1) and so two
// exchanges through LDS instead of three, the second inside a wave; in place
// as fft_dif and fft_dit, element e at lpad(e).
//   dif16: natural order in; thread j, register r holds
//          X[(j >> 4) + 16 (j & 15) + 256 r].
//   dit16: that order in, natural order out.
// Twiddles: W^k and W^4k of the two twiddled passes, held (products of at
// most three factors).
// ---------------------------------------------------------------------------
constexpr int kLine16 = 4096 + 4096 / 16;  // double2 in LDS
// a * exp(S*2*pi*i*M/16)
template <int S, int M>
__device__ __forceinline__ double2 w16(double2 a) {
  constexpr int m = M & 15;
  if constexpr (m % 2 == 0) return w8<S, m / 2>(a);
  else {
    constexpr double C = 0.92387953251128675613, D = 0.38268343236508977173;
    constexpr double c = (m == 1 || m == 15)   ? C
                         : (m == 7 || m == 9)  ? -C
                         : (m == 3 || m == 13) ? D
                                               : -D;
    constexpr double s0 = (m == 1 || m == 7)    ? D
                          : (m == 9 || m == 15) ? -D
                          : (m == 3 || m == 5)  ? C
                                                : -C;
    constexpr double s = S > 0 ? s0 : -s0;
    return make_double2(fma(a.x, c, -a.y * s), fma(a.x, s, a.y * c));
  }
}
// Radix-16 as 4 x 4 (n = 4 n1 + n2, k = k1 + 4 k2), natural-order output.
template <int S>
__device__ __forceinline__ void dft16(double2* a) {
#pragma unroll
  for (int n = 0; n < 4; ++n) dft4<S>(a[n], a[n + 4], a[n + 8], a[n + 12]);
  // a[n2 + 4 k1]
  a[5] = w16<S, 1>(a[5]);
  a[9] = w16<S, 2>(a[9]);
  a[13] = w16<S, 3>(a[13]);
  a[6] = w16<S, 2>(a[6]);
  a[10] = w16<S, 4>(a[10]);
  a[14] = w16<S, 6>(a[14]);
  a[7] = w16<S, 3>(a[7]);
  a[11] = w16<S, 6>(a[11]);
  a[15] = w16<S, 9>(a[15]);
#pragma unroll
  for (int k = 0; k < 4; ++k) dft4<S>(a[4 * k], a[4 * k + 1], a[4 * k + 2], a[4 * k + 3]);
  // a[4 k1 + k2] holds X[k1 + 4 k2]: transpose
  double2 y[16];
#pragma unroll
  for (int i = 0; i < 16; ++i) y[(i >> 2) + 4 * (i & 3)] = a[i];
#pragma unroll
  for (int i = 0; i < 16; ++i) a[i] = y[i];
}
// t[r] *= W^(k r) (conjugated for S > 0) from W^k and W^4k.
template <int S>
__device__ __forceinline__ void apply_tw16(double2* t, double2 w1, double2 w4) {
  auto ap = [](double2& x, double2 w) { x = S < 0 ? cmul(x, w) : cmulc(x, w); };
  ap(t[1], w1);
  ap(t[4], w4);
  ap(t[5], cmul(w1, w4));
  const double2 w2 = cmul(w1, w1);
  ap(t[2], w2);
  ap(t[6], cmul(w2, w4));
  const double2 w3 = cmul(w1, w2);
  ap(t[3], w3);
  ap(t[7], cmul(w3, w4));
  const double2 w8v = cmul(w4, w4);
  ap(t[8], w8v);
  ap(t[9], cmul(w1, w8v));
  ap(t[10], cmul(w2, w8v));
  ap(t[11], cmul(w3, w8v));
  const double2 w12 = cmul(w4, w8v);
  ap(t[12], w12);
  ap(t[13], cmul(w1, w12));
  ap(t[14], cmul(w2, w12));
  ap(t[15], cmul(w3, w12));
}
struct Tw16 {
  double2 a1, a4, b1, b4;
};
__device__ __forceinline__ Tw16 tw16(const double2* __restrict__ tw, int j) {
  return {tw[j], tw[4 * j], tw[16 * (j & 15)], tw[64 * (j & 15)]};
}
__device__ __forceinline__ Tw16 opaque16(Tw16 w) {
  asm volatile("" : "+v"(w.a1.x), "+v"(w.a1.y), "+v"(w.a4.x), "+v"(w.a4.y), "+v"(w.b1.x),
               "+v"(w.b1.y), "+v"(w.b4.x), "+v"(w.b4.y));
  return w;
}
// bar: as fft_dif_t
template <int S>
__device__ __forceinline__ void dif16(double2* a, double2* buf, int j, const Tw16& wh, bool bar) {
  asm volatile("" : "+v"(j));
  const Tw16 w = opaque16(wh);
  dft16<S>(a);
  apply_tw16<S>(a, w.a1, w.a4);
  if (bar) __syncthreads();
  {
    double2* p = buf + lpad(j);
#pragma unroll
    for (int r = 0; r < 16; ++r) p[272 * r] = a[r];
  }
  __syncthreads();
  {
    double2* p = buf + (j >> 4) * 272 + (j & 15);
#pragma unroll
    for (int r = 0; r < 16; ++r) a[r] = p[17 * r];
    dft16<S>(a);
    apply_tw16<S>(a, w.b1, w.b4);
#pragma unroll
    for (int r = 0; r < 16; ++r) p[17 * r] = a[r];
  }
  wave_sync();
  {
    const double2* p = buf + 17 * j;
#pragma unroll
    for (int r = 0; r < 16; ++r) a[r] = p[r];
    dft16<S>(a);
  }
}
template <int S>
__device__ __forceinline__ void dit16(double2* a, double2* buf, int j, const Tw16& wh) {
  asm volatile("" : "+v"(j));
  const Tw16 w = opaque16(wh);
  dft16<S>(a);
  {
    double2* p = buf + 17 * j;
#pragma unroll
    for (int r = 0; r < 16; ++r) p[r] = a[r];
  }
  wave_sync();
  {
    double2* p = buf + (j >> 4) * 272 + (j & 15);
#pragma unroll
    for (int r = 0; r < 16; ++r) a[r] = p[17 * r];
    apply_tw16<S>(a, w.b1, w.b4);
    dft16<S>(a);
#pragma unroll
    for (int r = 0; r < 16; ++r) p[17 * r] = a[r];
  }
  __syncthreads();
  {
    const double2* p = buf + lpad(j);
#pragma unroll
    for (int r = 0; r < 16; ++r) a[r] = p[272 * r];
    apply_tw16<S>(a, w.a1, w.a4);
    dft16<S>(a);
  }
}

}  // namespace gt
