// gturbo_kernels.hip -- gfx950 kernels of the pseudospectral step.
//
// Nonlinear term N(q) = -ik.(q u)^ (src/nlt.f90) on the compact layout, as two
// kinds of pass per evaluation:
//
//  * y pass (c_pass): one workgroup per tile of BT kx-columns.  Forward part:
//    forward y transform of the two product fields, -ik. combine, 2/3
//    truncation and the RK stage update (src/rkstep.f90 stage AXPYs).  Inverse
//    part: from the next stage input, the spectral operator |k|^-alpha
//    (src/nlt.f90:22-36) for q, u, v and their inverse y transforms.
//  * x pass (r_pass_*): complex-to-real x transforms of q, u and v, the
//    products q u, q v (src/produ.f90), and their real-to-complex transforms,
//    two real rows per complex transform: q of rows y and y+1 and so on
//    (r_pass_pair, r_pass_pair16), at N = 8192 the even and odd samples of one
//    row (r_pass_row).
//  * N <= 1024: f_pass and fx_pass, the same passes with the fields of a column
//    or row side by side on their own threads; the batched passes (ens_*) run
//    c_body and r_body of every member's size.
//
// Between the passes the three (resp. two) fields live in HBM in blocks of
// kYR rows x BT columns, [field][y / kYR][tile][y % kYR][kx % BT]: the y
// pass writes whole blocks (a 128-byte line at N = 4096), the x pass reads a
// row's pieces of consecutive tiles from one DRAM page, and its workgroup
// order keeps neighbouring rows on one XCD so that they share L2 lines.
#include <mutex>

#include "fft_core.hpp"
#include "gt_internal.hpp"

namespace gt {

// ---------------------------------------------------------------------------
// helpers
// ---------------------------------------------------------------------------

__device__ __forceinline__ bool cut_mode(const Phys& ph, double fkxs,
                                         double fkys) {
  // src/trunc.f90:13-15
  double k1 = fkys / ph.fkysmax;
  double k2 = k1 + fkxs / ph.fkxsmax;
  return k2 > ph.rtrunc2;
}

// ka = k2**(alpv/2) (src/nlt.f90:27): k2 itself for alpv = 2, correctly
// rounded square roots for alpv = 1 and 1/2, the power otherwise.
__device__ __forceinline__ double kalpha(const Phys& ph, double k2) {
  switch (ph.akind) {
    case 1: return k2;
    case 2: return sqrt(k2);
    case 3: return sqrt(sqrt(k2));
    default: return pow(k2, ph.ahalf);
  }
}

// With the 2/3 rule the kept rectangle stays below |k| = 3N/8, so of a
// thread's positions p = j + r*N/8 the ones with r = 3, 4 are never kept:
// those inputs are zero and those outputs unused.  TR = 1 makes that a
// compile-time fact.
template <int TR>
__device__ __forceinline__ constexpr bool live_r(int r) {
  return TR == 0 || (r != 3 && r != 4);
}

// Cache use of the y passes at N = 4096 and 8192, where a pass moves more
// than the 256 MB Infinity Cache holds.  The state z, the RK4 accumulator
// znew and the integrating factor emk are read and written once per y pass
// and next used a whole x pass later, by when they have left the caches;
// the products Y2 are read once.  The y passes access them without
// allocating cache lines (non-temporal), which leaves the caches to the
// fields Y1 they write and the next x pass reads at once.  Measured against
// the same kernels with ordinary accesses, one process on one box, results
// bit-identical: at 4096^2 the state accesses alone y stages -8%, RK4 step
// -2.4%; the Y2 reads on top of that x pass -4%, step -1.3%; both together
// RK4 -3.5%, RK2 -2%.  At 8192^2 the state accesses RK4 step -1.7%, but
// the Y2 reads on top +2.8% (there a one-column y workgroup reads half of
// each Y2 line and the next column's workgroup the other half), so there
// only the state bypasses the caches.  Non-temporal loads in the x pass
// slow it by 9-22%.
typedef double nt_d2 __attribute__((ext_vector_type(2)));
template <bool NT>
__device__ __forceinline__ double2 ld_state(const double2* p) {
  if constexpr (NT) {
    const nt_d2 v = __builtin_nontemporal_load(reinterpret_cast<const nt_d2*>(p));
    return make_double2(v.x, v.y);
  } else {
    return *p;
  }
}
template <bool NT>
__device__ __forceinline__ double ld_state(const double* p) {
  if constexpr (NT) return __builtin_nontemporal_load(p);
  else return *p;
}
template <bool NT>
__device__ __forceinline__ void st_state(double2* p, double2 v) {
  if constexpr (NT) {
    nt_d2 w;
    w.x = v.x;
    w.y = v.y;
    __builtin_nontemporal_store(w, reinterpret_cast<nt_d2*>(p));
  } else {
    *p = v;
  }
}

// ka in a y pass specialised on the alpha kind, where it is used: AK = 1
// when alpv = 2 (ka = k2, nothing else in the kernel); AK = 2 (the batched
// passes, whose members differ in alpha) k2 for alpv = 2, else the member's
// table of ka in the compact layout, built with the same expressions as
// kalpha (no power or root code in those kernels); AK = 3 (alpv != 2, N >=
// 2048) square roots for alpv = 1 and 1/2, else the table.
template <int AK>
__device__ __forceinline__ double kalpha_t(const PassArgs& a, double k2, unsigned q) {
  if constexpr (AK == 1) return k2;
  else if constexpr (AK == 2) return a.ph.akind == 1 ? k2 : a.ka[q];
  else return a.ph.akind == 2 ? sqrt(k2) : a.ph.akind == 3 ? sqrt(sqrt(k2)) : a.ka[q];
}

// Workgroup -> tile remap so that consecutive tiles run on one XCD
// (workgroups are dealt round-robin over the 8 XCDs, each with its own L2):
// XCD x takes a contiguous run of tiles, the first nblk % 8 XCDs one more.
__device__ __forceinline__ int xcd_remap(int bid, int nblk) {
  const int q = nblk / 8, rem = nblk % 8, x = bid % 8, i = bid / 8;
  return (x < rem ? x * (q + 1) : rem * (q + 1) + (x - rem) * q) + i;
}

// Thread -> (line, index in line) for NL lines per workgroup.  Lines
// alternate every 16 lanes: one 16-lane LDS access group then touches a
// single line (contiguous indices: no bank conflicts between lines), while a
// wave's global access still covers all NL lines of a tile row or run.
template <int TPL, int NL>
__device__ __forceinline__ void line_map(int tid, int& line, int& j) {
  constexpr int G = TPL < 16 ? TPL : 16;
  const int c = tid / G;
  line = c % NL;
  j = (c / NL) * G + tid % G;
}

// The same for lines of whole waves (in-place transforms): line = wave mod NL.
template <int NL>
__device__ __forceinline__ void wave_line_map(int tid, int& line, int& j) {
  line = (tid >> 6) % NL;
  j = ((tid >> 6) / NL) * 64 + (tid & 63);
}

// ---------------------------------------------------------------------------
// y pass
// ---------------------------------------------------------------------------

// The forcing of column c (fused step boundary) on the thread's values
// s[r] of rows p = j + (N/8) r: the same operations as forcing_k's
// force_one on each forced element, in the order of the forced-mode table.
template <int LOGN, int TR>
__device__ __forceinline__ void force_column(const PassArgs& a, int c, bool colok, int j,
                                             double2* s) {
#pragma clang fp contract(off)
  constexpr int N = 1 << LOGN, TPL = N / kE;
  if (a.fcs == nullptr || !colok) return;
  const double2* ph = a.fph;
  double amp = a.famp;
  if (a.fens != nullptr) {  // a batched ensemble member: this step's phases
    ph = a.fens->phases + (size_t)(*a.fstep) * a.fens->nf;
    amp = a.fens->amp;
  }
  const int e1 = a.fcs[c + 1];
  for (int e = a.fcs[c]; e < e1; ++e) {
    const FEntry f = a.fce[e];
    const double2 cs = ph[f.k];
    const double a1 = amp * f.ff1 * cs.x, a2 = amp * f.ff2 * cs.y;
#pragma unroll
    for (int r = 0; r < kE; ++r) {
      if (live_r<TR>(r) && row_of(j + TPL * r, a.rc, N) == f.row) {
        s[r].x = s[r].x + a1;
        s[r].y = f.conj ? s[r].y - a2 : s[r].y + a2;
      }
    }
  }
}

// Nonlinear term of one mode from the forward transforms A = (q u)^,
// B = (q v)^ of its column: fft_dir normalisation /NY/NX (src/fft_dir.f90:19,
// exact for N = 2^k), -ik. (src/nlt.f90:57-58), 2/3 mask.
__device__ __forceinline__ double2 nl_term(const Phys& ph, double2 A, double2 B, double fkx,
                                           double fkxs, double fky) {
  const double2 Av = make_double2(A.x * ph.inv_n2, A.y * ph.inv_n2);
  const double2 Bv = make_double2(B.x * ph.inv_n2, B.y * ph.inv_n2);
  double2 k = make_double2(fkx * Av.y + fky * Bv.y, -fkx * Av.x - fky * Bv.x);
  if (ph.truncate == 1 && cut_mode(ph, fkxs, fky * fky)) k = make_double2(0.0, 0.0);
  return k;
}

// What the RK stage of a y pass reads of one mode (compact index q).
struct StageIn {
  double E;
  double2 z, zn;
};
template <int MODE, bool NT>
__device__ __forceinline__ StageIn stage_load(const PassArgs& a, unsigned q) {
  constexpr bool RK4S = MODE == C_RK4_2 || MODE == C_RK4_3;
  constexpr bool LAST4 = MODE == C_RK4_4 || MODE == C_RK4_4S;
  StageIn in{};
  if constexpr (MODE != C_NLT && MODE != C_START && !LAST4) {
    in.E = ld_state<NT>(&a.emk[q]);
    in.z = ld_state<NT>(&a.z[q]);
  }
  if constexpr (RK4S || LAST4) in.zn = ld_state<NT>(&a.znew[q]);
  return in;
}
// The RK stage of one mode with nonlinear term k: stores what the stage
// stores and returns the next stage input (for the fused step boundary the
// updated state, which is forced and stored by the caller).
template <int MODE, bool NT>
__device__ __forceinline__ double2 stage_update(const PassArgs& a, unsigned q, bool mean,
                                                double2 k, const StageIn& in) {
  const Phys& ph = a.ph;
  const double E = in.E;
  const double2 zz = in.z, zn = in.zn;
  double2 s = make_double2(0.0, 0.0);
  if constexpr (MODE == C_NLT) {
    if (mean) k = make_double2(0.0, 0.0);  // trunc.f90:24
    a.out[q] = k;
  } else if constexpr (MODE == C_RK4_1) {
    // rkstep.f90:96,101
    const double EE = E * E;
    st_state<NT>(&a.znew[q], make_double2(EE * (zz.x + ph.dt6 * k.x), EE * (zz.y + ph.dt6 * k.y)));
    s = make_double2(E * (zz.x + ph.dt2 * k.x), E * (zz.y + ph.dt2 * k.y));
  } else if constexpr (MODE == C_RK4_2) {
    // rkstep.f90:105,110
    const double d3E = ph.dt3 * E;
    st_state<NT>(&a.znew[q], make_double2(zn.x + d3E * k.x, zn.y + d3E * k.y));
    s = make_double2(E * zz.x + ph.dt2 * k.x, E * zz.y + ph.dt2 * k.y);
  } else if constexpr (MODE == C_RK4_3) {
    // rkstep.f90:114,119
    const double d3E = ph.dt3 * E;
    st_state<NT>(&a.znew[q], make_double2(zn.x + d3E * k.x, zn.y + d3E * k.y));
    s = make_double2(E * (E * zz.x + ph.dt * k.x), E * (E * zz.y + ph.dt * k.y));
  } else if constexpr (MODE == C_RK4_4 || MODE == C_RK4_4S) {
    // rkstep.f90:123,127
    s = make_double2(zn.x + ph.dt6 * k.x, zn.y + ph.dt6 * k.y);
    if (mean) s = make_double2(0.0, 0.0);
    if constexpr (MODE == C_RK4_4) st_state<NT>(&a.z[q], s);
  } else if constexpr (MODE == C_RK2_1) {
    // rkstep.f90:24/34 and :42
    s = make_double2(E * (zz.x + ph.dt2 * k.x), E * (zz.y + ph.dt2 * k.y));
    if (mean) s = make_double2(0.0, 0.0);
  } else if constexpr (MODE == C_RK2_2 || MODE == C_RK2_2S) {
    // rkstep.f90:54/64 and :72
    s = make_double2(E * (E * zz.x + ph.dt * k.x), E * (E * zz.y + ph.dt * k.y));
    if (mean) s = make_double2(0.0, 0.0);
    if constexpr (MODE == C_RK2_2) st_state<NT>(&a.z[q], s);
  }
  return s;
}
// Value of one mode in inverse transform f of a y pass: the stage input q
// (f = 0), u = i ky q/ka (f = 1), v = -i kx q/ka (f = 2); src/nlt.f90:31-34.
__device__ __forceinline__ double2 field_of(int f, double2 s, double fkx, double fky,
                                            double ka) {
  if (f == 0) return s;
  if (f == 1) {
    const double kyn = fky / ka;
    return make_double2(-kyn * s.y, kyn * s.x);
  }
  const double kxn = fkx / ka;
  return make_double2(kxn * s.y, -kxn * s.x);
}

// double2 of LDS of an in-place line (8192: two 4096-point problems).
template <int LOGN>
__host__ __device__ constexpr int ip_lds() {
  return LOGN == 13 ? 2 * kIpLine : ip_line<LOGN>();
}

// A group of BT kx-columns; lds holds BT padded lines, the y buffers tiles of
// LB columns.  SCHED is the radix
// order of the transforms (fft_reg).
// IP (N >= 1024): the y buffers hold the rows of a column in the order the
// in-place transforms use (slot j + N/8 r holds physical row ip_row(j, r));
// the forward transforms (fft_dit) take the loaded slots and return natural
// ky order, the inverse ones (fft_dif) return slot order for the stores.
// Each line is whole waves (wave_line_map).  The x pass transforms rows,
// whichever rows a slot pair holds.
template <int LOGN, int MODE, int AK, int TR, int BT, int SCHED, bool IP = false, int LB = BT>
__device__ __forceinline__ void c_body(const PassArgs& a, int tile, int tid,
                                       double2* lds, const double2* tw) {
  constexpr int N = 1 << LOGN, TPL = N / kE;
  constexpr int LINE = IP ? ip_lds<LOGN>() : Line<LOGN>::PADDED;
  static_assert(!IP || (LOGN == 13 && BT == 1) || (LOGN >= 10 && LOGN <= 12),
                "in-place y pass: lines of 1024 to 4096 points, or one of 8192");
  constexpr bool FWD = MODE != C_START;
  constexpr bool INV = MODE == C_START || MODE == C_RK4_1 || MODE == C_RK4_2 ||
                       MODE == C_RK4_3 || MODE == C_RK2_1 || MODE == C_RK4_4S ||
                       MODE == C_RK2_2S;
  constexpr bool NT = LOGN >= 12;    // state accesses that bypass the caches
  // ka formed or read once for u and v, not at each of them (below; alpha 1.5
  // at 4096 1332 -> 1290 us a step, at 8192 5928 -> 5829; the batched sizes
  // keep the rounding they share with f_pass)
  constexpr bool ONCE = LOGN >= 12;
  constexpr bool NT2 = LOGN == 12;   // Y2 reads likewise, at 4096 only
  int b, j;
  if constexpr (IP) wave_line_map<BT>(tid, b, j);
  else line_map<TPL, BT>(tid, b, j);
  const int c = tile * BT + b;
  const Rect rc = a.rc;
  const bool colok = c <= rc.kx;
  double2* buf = lds + b * LINE;
  const Phys& ph = a.ph;
  const double fkx = (double)c * ph.dkx;
  const double fkxs = fkx * fkx;
  const unsigned cbase = (unsigned)c * (unsigned)a.kyp;
  double2 s[kE];
  double2 z[kE];
  // the batched passes loop over items: another wave may still read the last
  // one's LDS
  constexpr bool LOOP = AK == 2;
  // in-place transforms up to 4096 points: their three twiddles, loaded once.
  constexpr bool HELD = IP && LOGN <= 12 && !LOOP;
  IpTw<LOGN> ytw{};
  if constexpr (HELD) ytw = ip_tw<LOGN>(tw, j);

  if constexpr (FWD) {
    double2 A[kE];
    const unsigned colo = ycol_off(c, LB);
    const double2* srcA = a.y2;
#pragma unroll
    for (int r = 0; r < kE; ++r) z[r] = ld_state<NT2>(&srcA[yrow_off(j + TPL * r, a.ntiles, LB) + colo]);
    if constexpr (HELD) fft_dit_held<LOGN, -1>(z, buf, j, ytw);
    else if constexpr (IP && LOOP) fft_dit<-1, true, 1, LOGN>(z, buf, j, tw);
    else if constexpr (IP) fft_dit2<-1, false>(z, buf, j, tw);
    else fft_reg<LOGN, -1, SCHED>(z, buf, j, tw);
#pragma unroll
    for (int r = 0; r < kE; ++r) A[r] = live_r<TR>(r) ? z[r] : make_double2(0.0, 0.0);
    const double2* srcB = a.y2 + (size_t)a.ntiles * N * LB;
#pragma unroll
    for (int r = 0; r < kE; ++r) z[r] = ld_state<NT2>(&srcB[yrow_off(j + TPL * r, a.ntiles, LB) + colo]);
    if constexpr (HELD) fft_dit_held<LOGN, -1, true>(z, buf, j, ytw);
    else if constexpr (IP && LOOP) fft_dit<-1, true, 1, LOGN>(z, buf, j, tw);
    else if constexpr (IP) fft_dit2<-1, true>(z, buf, j, tw);
    else fft_reg<LOGN, -1, SCHED>(z, buf, j, tw);
    int je = j;
    // The epilogue's indices (and so its loads) depend on the transform's
    // output: nothing of the epilogue is scheduled inside the last pass.
    asm volatile("" : "+v"(je) : "v"(z[0].x), "v"(z[kE - 1].y));
#pragma unroll
    for (int r = 0; r < kE; ++r) {
      const int p = je + TPL * r;
      const int row = row_of(p, rc, N);
      s[r] = make_double2(0.0, 0.0);
      if (live_r<TR>(r) && colok && row >= 0) {
        const double fky = (double)kyi_of(p, N) * ph.dky;
        const double2 k = nl_term(ph, A[r], z[r], fkx, fkxs, fky);
        const unsigned q = cbase + (unsigned)row;
        s[r] = stage_update<MODE, NT>(a, q, c == 0 && p == 0, k, stage_load<MODE, NT>(a, q));
      }
    }
    if constexpr (MODE == C_RK4_4S || MODE == C_RK2_2S) {
      // the step's forcing on this column (forcing.f90:16-33), then the
      // forced state stored: it is also the next step's stage input
      force_column<LOGN, TR>(a, c, colok, je, s);
#pragma unroll
      for (int r = 0; r < kE; ++r) {
        const int row = row_of(je + TPL * r, rc, N);
        if (live_r<TR>(r) && colok && row >= 0) st_state<NT>(&a.z[cbase + (unsigned)row], s[r]);
      }
    }
  } else {
#pragma unroll
    for (int r = 0; r < kE; ++r) {
      const int p = j + TPL * r;
      const int row = row_of(p, rc, N);
      s[r] = (live_r<TR>(r) && colok && row >= 0) ? ld_state<NT>(&a.z[cbase + (unsigned)row])
                                                   : make_double2(0.0, 0.0);
    }
  }

  if constexpr (INV) {
    if (a.sst != nullptr) {  // stage input kept for the adjoint's recompute
#pragma unroll
      for (int r = 0; r < kE; ++r) {
        const int row = row_of(j + TPL * r, rc, N);
        if (live_r<TR>(r) && colok && row >= 0) a.sst[cbase + (unsigned)row] = s[r];
      }
    }
#pragma unroll 1
    for (int f = 0; f < 3; ++f) {
      int jo = j;
      asm volatile("" : "+v"(jo));  // keep the per-row factors inside the loop
#pragma unroll
      for (int r = 0; r < kE; ++r) {
        const int p = jo + TPL * r;
        double2 v = make_double2(0.0, 0.0);
        if (live_r<TR>(r) && colok && row_of(p, rc, N) >= 0) {
          if (f == 0) {
            v = s[r];
          } else if (!(c == 0 && p == 0)) {  // nlt.f90:25
            const double fky = (double)kyi_of(p, N) * ph.dky;
            if constexpr (ONCE) {
              // q is not needed any more: q/ka in its place, ka formed (or
              // read) once for both velocity components
              if (f == 1) {
                const double kar = kalpha_t<AK>(a, fkxs + fky * fky,
                                                cbase + (unsigned)row_of(p, rc, N));
                s[r] = make_double2(s[r].x / kar, s[r].y / kar);
                v = make_double2(-fky * s[r].y, fky * s[r].x);
              } else {
                v = make_double2(fkx * s[r].y, -fkx * s[r].x);
              }
            } else {
              v = field_of(f, s[r], fkx, fky,
                           kalpha_t<AK>(a, fkxs + fky * fky,
                                        cbase + (unsigned)row_of(p, rc, N)));
            }
          }
        }
        z[r] = v;
      }
      if constexpr (IP) {
        // a barrier first unless nothing has used LDS since the table staging
        if constexpr (HELD) fft_dif_held<LOGN, +1>(z, buf, j, ytw, FWD || f > 0);
        else if constexpr (LOOP) fft_dif<+1, 1, LOGN>(z, buf, j, tw, true);
        else fft_dif2<+1>(z, buf, j, tw, FWD || f > 0);
      } else {
        fft_reg<LOGN, +1, SCHED>(z, buf, j, tw);
      }
      if constexpr (LOGN == 12) {  // row-pair blocks (y1_off)
        const int cols = y1_cols(rc.kc());
        double2* dst = a.y1 + (size_t)f * N * cols;
#pragma unroll
        for (int r = 0; r < kE; ++r) dst[y1_off(j + TPL * r, c, cols)] = z[r];
      } else {
        double2* dst = a.y1 + (size_t)f * a.ntiles * N * LB;
        const unsigned colo = ycol_off(c, LB);
#pragma unroll
        for (int r = 0; r < kE; ++r) dst[yrow_off(j + TPL * r, a.ntiles, LB) + colo] = z[r];
      }
    }
  }
}

// Which y passes use the in-place transforms, for any alpha: on the 2/3
// rectangle RK4 steps at 2048 304 (alpha 2), 356 (1), 382 (1.5) -> 292, 297,
// 301 us, at 4096 alpha 1 1252 -> 1143, at 8192 alpha 1 6228 -> 5545, 1.5
// 6397 -> 5829 (Stockham passes with ka in registers, which spilled).  On the
// full one only at 8192 (9784 -> 9324); at 4096 its eight live values a field
// leave no registers for the held twiddles (1887 -> 2080), at 2048 no change.
template <int LOGN, int TR>
__host__ __device__ constexpr bool c_pass_ip() { return TR == 1 || LOGN == 13; }
template <int LOGN, int MODE, int AK, int TR>
__global__ void __launch_bounds__(bt_of(LOGN) * (1 << LOGN) / kE, 4) c_pass(PassArgs a) {
  constexpr int BT = bt_of(LOGN);
  // Row slots in transform order (in-place transforms) on the 2/3 rectangle;
  // every y pass of a run has the same AK and TR, so the buffers' row order is
  // the same in all of them.
  constexpr bool IP = c_pass_ip<LOGN, TR>();
  // The in-place transforms up to 4096 points hold their three twiddles in
  // registers (read once from memory): no table in LDS.
  constexpr bool HELD = IP && LOGN <= 12;
  __shared__ double2 lds[BT * (IP ? ip_lds<LOGN>() : Line<LOGN>::PADDED)];
  __shared__ double2 twl[HELD ? 1 : tw_lds_size<LOGN>()];
  const double2* tw = HELD ? a.tw : stage_tw<LOGN>(twl, a.tw, threadIdx.x, blockDim.x);
  // 8192: a one-column workgroup shares each line of Y1 and Y2 with the next
  // column's, so neighbouring columns run on one XCD (y stages -5.6%).
  const int tile = LOGN == 13 ? xcd_remap(blockIdx.x, gridDim.x) : (int)blockIdx.x;
  c_body<LOGN, MODE, AK, TR, BT, 0, IP>(a, tile, threadIdx.x, lds, tw);
}

// ---------------------------------------------------------------------------
// Small grids: the fields of a column (y pass) or row (x pass) side by side.
// On these grids a pass has fewer workgroups than the chip has room for
// (43 column pairs at 256^2 on 256 CUs) and its time is the chain of loads,
// transforms and barriers inside one workgroup, not a rate.  Each of a
// column's fields therefore has its own N/8 threads (whole waves per field):
// the two forward transforms run together, then the three inverse ones (five
// one after the other otherwise), and every load of the pass -- products,
// state, twiddles, ka, forcing -- is issued before the first transform.
// Against the five-in-turn passes (kernel durations, RK4, same operations,
// bit-identical): y stage 64^2 11.1 -> 4.4 us, 256^2 12.0 -> 5.5, 512^2
// (alpha 1) 14.6 -> 7.2, 1024^2 (alpha 1) 24.0 -> 18.0; step boundary 256^2
// 15.4 -> 7.5, 1024^2 29.4 -> 20.7; x pass 5.0 -> 4.1, 5.8 -> 4.8, 7.8 ->
// 6.5, 16.8 -> 16.2.  Up to 512^2 the rest is a kernel's own start and end
// (about 2 us), two memory round trips and two transforms; at 1024^2 the
// 41 MB a stage moves take half of it (12.7 us with the transforms skipped),
// and in-place transforms, whose few barriers and held twiddles (100 instead
// of 160 VGPRs) replace Stockham ones there, the next part: y stage 18.3 ->
// 17.0 us, boundary 20.9 -> 18.5, untruncated 27 -> 24.4, x pass 16.2 -> 16.3
// (the same within a run's spread, with half the twiddle error).
// ---------------------------------------------------------------------------

// Columns per workgroup of the y pass: a wave per field where a line is
// shorter than a wave; 512: one (7.3 us; two 8.2); 1024: two (16.4 us; one,
// whose workgroups each touch half of every line, 19.2).
__host__ __device__ constexpr int fp_cols(int logn) { return logn < 9 ? 512 >> logn : logn == 9 ? 1 : 2; }
constexpr int kFpForce = 32;  // forced modes of a column staged in LDS

// Twiddles and LDS line of a field: Stockham inside a wave, in place beyond.
template <int LOGN>
__host__ __device__ constexpr int fp_line() {
  return line_in_wave<LOGN>() ? Line<LOGN>::PADDED : ip_lds<LOGN < 10 ? 10 : LOGN>();
}
template <int LOGN>
__device__ __forceinline__ auto fp_tw(const double2* __restrict__ tw, int j) {
  if constexpr (line_in_wave<LOGN>()) return held_tw<LOGN>(tw, j);
  else return ip_tw<LOGN>(tw, j);
}

template <int LOGN, int MODE, int AK, int TR>
__global__ void __launch_bounds__(fp_cols(LOGN) * 3 * (1 << LOGN) / kE) f_pass(PassArgs a) {
  constexpr int N = 1 << LOGN, TPL = N / kE, BT = bt_of(LOGN), CW = fp_cols(LOGN);
  // 1024: in-place transforms, the y buffers in their row order (see c_body)
  constexpr bool IP = !line_in_wave<LOGN>();
  constexpr int LINE = fp_line<LOGN>(), GT = CW * TPL;  // threads per field
  constexpr bool FWD = MODE != C_START;
  constexpr bool INV = MODE != C_NLT && MODE != C_RK4_4 && MODE != C_RK2_2;
  constexpr bool BOUND = MODE == C_RK4_4S || MODE == C_RK2_2S;
  constexpr int NOWN = TR ? 2 : 3;           // modes a thread updates
  constexpr int NLINE = FWD && INV ? 4 : 3;  // A, B, (scratch), stage input
  static_assert(GT % 64 == 0, "whole waves per field");
  __shared__ double2 lds[CW * NLINE * LINE];
  __shared__ double2 famp[BOUND ? CW * kFpForce : 1];
  __shared__ __align__(16) int frow[BOUND ? CW * kFpForce : 4];
  const int f = __builtin_amdgcn_readfirstlane(threadIdx.x / GT);
  const int t = threadIdx.x % GT, cw = t / TPL, j = t % TPL;
  // one-column workgroups: the two columns of a tile on one XCD
  const int c = CW == 1 ? xcd_remap(blockIdx.x, gridDim.x) : (int)blockIdx.x * CW + cw;
  const Rect rc = a.rc;
  const bool colok = c <= rc.kx;
  const Phys& ph = a.ph;
  const double fkx = (double)c * ph.dkx;
  const double fkxs = fkx * fkx;
  const unsigned cbase = (unsigned)c * (unsigned)a.kyp;
  const unsigned colo = ycol_off(c, BT);
  double2* col = lds + cw * NLINE * LINE;
  double2* buf = col + f * LINE;
  double2* sbuf = col + 3 * LINE;  // the column's stage input

  double2 z[kE];
  if constexpr (FWD) {
    if (f < 2) {
      const double2* src = a.y2 + (size_t)f * a.ntiles * N * BT;
#pragma unroll
      for (int r = 0; r < kE; ++r)
        z[r] = colok ? src[yrow_off(j + TPL * r, a.ntiles, BT) + colo] : make_double2(0.0, 0.0);
    }
  } else {
#pragma unroll
    for (int r = 0; r < kE; ++r) {
      const int row = row_of(j + TPL * r, rc, N);
      z[r] = (live_r<TR>(r) && colok && row >= 0) ? a.z[cbase + (unsigned)row]
                                                   : make_double2(0.0, 0.0);
    }
  }
  const auto tw = fp_tw<LOGN>(a.tw, j);
  // positions this thread updates: r = NOWN f + i of the live ones
  int pos[NOWN];
  bool own[NOWN];
  unsigned qi[NOWN];
  StageIn in[NOWN];
  if constexpr (FWD) {
#pragma unroll
    for (int i = 0; i < NOWN; ++i) {
      const int x = NOWN * f + i, r = TR && x >= 3 ? x + 2 : x;
      pos[i] = j + TPL * r;
      const int row = r < kE ? row_of(pos[i], rc, N) : -1;
      own[i] = colok && row >= 0;
      qi[i] = cbase + (unsigned)row;
      in[i] = own[i] ? stage_load<MODE, false>(a, qi[i]) : StageIn{};
    }
  }
  double ka[kE];
  auto load_ka = [&]() {
#pragma unroll
    for (int r = 0; r < kE; ++r) {
      const int row = row_of(j + TPL * r, rc, N);
      ka[r] = live_r<TR>(r) && colok && row >= 0 && f > 0 ? a.ka[cbase + (unsigned)row] : 1.0;
    }
  };
  if constexpr (INV && AK == 2) load_ka();

  if constexpr (FWD) {
    // The column's forcing entries (forcing.f90:25-31), formed by the third
    // field's waves while the others transform.
    const bool forced = BOUND && a.fcs != nullptr && colok;
    int e0 = 0, ne = 0;
    if constexpr (BOUND) {
      if (forced) {
        e0 = a.fcs[c];
        ne = a.fcs[c + 1] - e0;
      }
      if (f == 2) {
        for (int e = j; e < kFpForce; e += TPL) {
          int row = -1;
          if (e < ne) {
            const FEntry fe = a.fce[e0 + e];
            const double2 cs = a.fph[fe.k];
            const double a2 = a.famp * fe.ff2 * cs.y;
            famp[cw * kFpForce + e] = make_double2(a.famp * fe.ff1 * cs.x, fe.conj ? -a2 : a2);
            row = fe.row;
          }
          frow[cw * kFpForce + e] = row;
        }
      }
    }
    if constexpr (IP) {
      fft_dit_held<LOGN, -1>(z, buf, j, tw, f < 2);
      __syncthreads();  // every wave's reads done
    } else if (f < 2) {
      fft_held<LOGN, -1>(z, buf, j, tw);
    }
    if (f < 2) {
#pragma unroll
      for (int r = 0; r < kE; ++r)
        if (live_r<TR>(r)) (buf + lpad(j))[lpad_off(TPL * r)] = z[r];
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < NOWN; ++i) {
      double2 s = make_double2(0.0, 0.0);
      if (own[i]) {
        const int p = pos[i], e = lpad(p);
        const double fky = (double)kyi_of(p, N) * ph.dky;
        const double2 k = nl_term(ph, col[e], col[LINE + e], fkx, fkxs, fky);
        s = stage_update<MODE, false>(a, qi[i], c == 0 && p == 0, k, in[i]);
        if constexpr (BOUND) {  // in table order
          const int row = (int)(qi[i] - cbase);
          const int* fr = frow + cw * kFpForce;
          for (int n = 0; n < (ne < kFpForce ? ne : kFpForce); n += 8) {
            const int4 u = *reinterpret_cast<const int4*>(fr + n);
            const int4 w = *reinterpret_cast<const int4*>(fr + n + 4);
            if (u.x == row || u.y == row || u.z == row || u.w == row || w.x == row ||
                w.y == row || w.z == row || w.w == row) {
              for (int m = n; m < n + 8; ++m) {
                if (fr[m] == row) {
                  const double2 d = famp[cw * kFpForce + m];
                  s = make_double2(s.x + d.x, s.y + d.y);
                }
              }
            }
          }
          for (int n = kFpForce; n < ne; ++n) {
            const FEntry fe = a.fce[e0 + n];
            if (fe.row == row) {
              const double2 cs = a.fph[fe.k];
              const double a2 = a.famp * fe.ff2 * cs.y;
              s = make_double2(s.x + a.famp * fe.ff1 * cs.x, fe.conj ? s.y - a2 : s.y + a2);
            }
          }
          a.z[qi[i]] = s;
        }
        if constexpr (INV) {
          if (a.sst != nullptr) a.sst[qi[i]] = s;  // kept for the adjoint's recompute
        }
      }
      if constexpr (INV) {
        if (TR || NOWN * f + i < kE) sbuf[lpad(pos[i])] = s;
      }
    }
    if constexpr (INV) {
      __syncthreads();
#pragma unroll
      for (int r = 0; r < kE; ++r)
        z[r] = live_r<TR>(r) ? (sbuf + lpad(j))[lpad_off(TPL * r)] : make_double2(0.0, 0.0);
    }
  } else if (a.sst != nullptr && f == 0) {
#pragma unroll
    for (int r = 0; r < kE; ++r) {
      const int row = row_of(j + TPL * r, rc, N);
      if (live_r<TR>(r) && colok && row >= 0) a.sst[cbase + (unsigned)row] = z[r];
    }
  }

  if constexpr (INV) {
#pragma unroll
    for (int r = 0; r < kE; ++r) {
      if (!live_r<TR>(r)) continue;
      const int p = j + TPL * r;
      const double fky = (double)kyi_of(p, N) * ph.dky;
      if (c == 0 && p == 0) {  // nlt.f90:25
        if (f > 0) z[r] = make_double2(0.0, 0.0);
      } else {
        z[r] = field_of(f, z[r], fkx, fky, AK == 1 ? fkxs + fky * fky : ka[r]);
      }
    }
    if constexpr (IP) fft_dif_held<LOGN, +1>(z, buf, j, tw, false);
    else fft_held<LOGN, +1>(z, buf, j, tw);
    if (colok) {
      double2* dst = a.y1 + (size_t)f * a.ntiles * N * BT;
#pragma unroll
      for (int r = 0; r < kE; ++r) dst[yrow_off(j + TPL * r, a.ntiles, BT) + colo] = z[r];
    }
  }
}

// ---------------------------------------------------------------------------
// x pass
// ---------------------------------------------------------------------------

// Offset of column k of a y-row in the blocked layout.
template <int LOGN, int BT>
__device__ __forceinline__ unsigned koff(int k) {
  return ycol_off(k, BT);
}

// Z = F + i G over the full x-spectrum at the thread's positions
// p = j + TPL*r, from the half-spectra F, G of two real sequences (kx <=
// kx_max; the imaginary parts at kx = 0 and N/2 are not used, as in a C2R
// transform).  The inverse transform of Z is f + i g.  Built in two
// halves: the loads (zeros outside the kept half-spectrum), all issued
// before any is used so that they are in flight together, and the packing.
// Y1: the input is in row-pair blocks (y1_off) rather than tiles.
template <int LOGN, int TR, int BT, bool Y1 = false>
__device__ __forceinline__ void load_two(double2* x0, double2* x1, int j,
                                         const double2* __restrict__ y,
                                         unsigned off_f, unsigned off_g, int kxm) {
  constexpr int N = 1 << LOGN, TPL = N / kE;
#pragma unroll
  for (int r = 0; r < kE; ++r) {
    const int p = j + TPL * r;
    const int k = p <= N / 2 ? p : N - p;
    const unsigned ko = Y1 ? y1_off(0, k, 0) : koff<LOGN, BT>(k);
    x0[r] = x1[r] = make_double2(0.0, 0.0);
    if (live_r<TR>(r) && k <= kxm) {
      x0[r] = y[off_f + ko];
      x1[r] = y[off_g + ko];
    }
  }
}
template <int LOGN>
__device__ __forceinline__ void pack_two(double2* z, int j, const double2* x0,
                                         const double2* x1) {
  constexpr int N = 1 << LOGN, TPL = N / kE;
#pragma unroll
  for (int r = 0; r < kE; ++r) {
    const int p = j + TPL * r;
    if (p == 0 || p == N / 2) z[r] = make_double2(x0[r].x, x1[r].x);
    else if (p < N / 2) z[r] = make_double2(x0[r].x - x1[r].y, x0[r].y + x1[r].x);
    else z[r] = make_double2(x0[r].x + x1[r].y, x1[r].x - x0[r].y);
  }
}
template <int LOGN, int TR, int BT, bool Y1 = false>
__device__ __forceinline__ void build_two(double2* z, int j,
                                          const double2* __restrict__ y,
                                          unsigned off_f, unsigned off_g, int kxm) {
  double2 x0[kE], x1[kE];
  load_two<LOGN, TR, BT, Y1>(x0, x1, j, y, off_f, off_g, kxm);
  pack_two<LOGN>(z, j, x0, x1);
}
// Element (N - k) mod N, k = j + TPL r (r a constant), of a line in LDS;
// pm = buf + lpad(TPL - j).  For TPL >= 16 the index TPL (7 - r) + TPL - j
// splits into that base and a constant offset; k = 0 maps to element 0.
template <int LOGN>
__device__ __forceinline__ double2 mirror_at(const double2* buf, const double2* pm, int j,
                                             int r) {
  constexpr int N = 1 << LOGN, TPL = N / kE;
  if constexpr (TPL % 16 != 0) {
    return buf[lpad((N - j - TPL * r) & (N - 1))];
  } else {
    if (r == 0) return (j == 0 ? buf : pm + lpad_off(7 * TPL))[0];
    return pm[lpad_off(TPL * (7 - r))];
  }
}

// Split W = FFT(a + i b) (held at k = j + TPL*r) into the half-spectra of
// the real sequences a and b and store kx <= kx_max.  W[N-k] comes through
// LDS.
template <int LOGN, int TR, int BT>
__device__ __forceinline__ void split_store(const double2* w, double2* buf, int j,
                                            double2* __restrict__ y,
                                            unsigned off_a, unsigned off_b, int kxm) {
  constexpr int N = 1 << LOGN, TPL = N / kE;
  double2* pj = buf + lpad(j);
#pragma unroll
  for (int r = 0; r < kE; ++r)
    if (live_r<TR>(r)) pj[lpad_off(TPL * r)] = w[r];
  __syncthreads();
  const double2* pm = buf + lpad(TPL - j);
#pragma unroll
  for (int r = 0; r <= kE / 2; ++r) {  // k <= N/2 (r = kE/2 only for k = N/2)
    const int k = j + TPL * r;
    if (live_r<TR>(r) && k <= kxm && k <= N / 2) {
      const double2 W = w[r];
      const double2 Wc = mirror_at<LOGN>(buf, pm, j, r);
      y[off_a + koff<LOGN, BT>(k)] = make_double2(0.5 * (W.x + Wc.x), 0.5 * (W.y - Wc.y));
      y[off_b + koff<LOGN, BT>(k)] = make_double2(0.5 * (W.y + Wc.y), -0.5 * (W.x - Wc.x));
    }
  }
  __syncthreads();
}

// One y row per line, NL lines per workgroup (group g holds rows g*NL ..):
// q+iv and q+iu come out of one complex transform each, so each product is
// formed the moment its factors exist and only q*v is carried (as 8
// doubles) into the R2C transform of W = q*u + i q*v.  BT is the tile width
// of the y-pass buffers.  Lines alternate every 16 lanes: with two rows over
// two-column tiles a wave's access covers whole 64-byte runs of a tile.
template <int LOGN, int TR, int BT, int NL, int SCHED>
__device__ __forceinline__ void r_body(const PassArgs& a, int g, int tid,
                                       double2* lds, const double2* tw) {
  constexpr int N = 1 << LOGN, TPL = N / kE;
  constexpr bool IP = LOGN == 10;  // in-place transforms, as f_pass and fx_pass
  constexpr int LINE = IP ? ip_line<10>() : Line<LOGN>::PADDED;
  int pl, j;
  if constexpr (IP) wave_line_map<NL>(tid, pl, j);
  else line_map<TPL, NL>(tid, pl, j);
  const int yrow = g * NL + pl;
  double2* buf = lds + pl * LINE;
  const int kxm = a.rc.kx;
  const unsigned fstride = (unsigned)a.ntiles * N * BT;  // one field
  const unsigned offQ = yrow_off(yrow, a.ntiles, BT), offU = offQ + fstride,
                 offV = offU + fstride;

  double2 z[kE];
  double qv[kE];
  auto inv = [&](bool bar) {  // bar: another wave may still read LDS
    if constexpr (IP) fft_dif<+1, 1, LOGN>(z, buf, j, tw, bar);
    else fft_reg<LOGN, +1, SCHED>(z, buf, j, tw);
  };
  build_two<LOGN, TR, BT>(z, j, a.y1, offQ, offV, kxm);
  inv(false);  // an item before ended with a barrier
#pragma unroll
  for (int r = 0; r < kE; ++r) qv[r] = z[r].x * z[r].y;  // produ.f90:16
  build_two<LOGN, TR, BT>(z, j, a.y1, offQ, offU, kxm);
  inv(true);
#pragma unroll
  for (int r = 0; r < kE; ++r) z[r] = make_double2(z[r].x * z[r].y, qv[r]);  // produ.f90:15
  if constexpr (IP) {
    fft_dit<-1, false, 1, LOGN>(z, buf, j, tw);
    __syncthreads();  // every wave's reads done
  } else {
    fft_reg<LOGN, -1, SCHED>(z, buf, j, tw);
  }
  split_store<LOGN, TR, BT>(z, buf, j, a.y2, offQ, offQ + fstride, kxm);
}

// Small grids (see f_pass): a row's two inverse transforms, of q+iv and
// q+iu, each on its own N/8 threads; the operations are r_body's.  q v
// crosses to the q u threads through LDS, these run the forward transform of
// q u + i q v, and both store their half of the split spectrum.
// Rows per workgroup: 512: two (6.4 us; one 7.2); 1024: one (two 1% slower).
__host__ __device__ constexpr int fx_rows(int logn) {
  return logn == 10 ? 1 : logn == 9 ? 2 : logn == 4 ? 16 : 512 >> logn;
}
template <int LOGN, int TR>
__global__ void __launch_bounds__(2 * fx_rows(LOGN) * (1 << LOGN) / kE) fx_pass(PassArgs a) {
  constexpr int N = 1 << LOGN, TPL = N / kE, BT = bt_of(LOGN), RW = fx_rows(LOGN);
  constexpr bool IP = !line_in_wave<LOGN>();  // 1024: in-place transforms
  constexpr int LINE = fp_line<LOGN>(), GT = RW * TPL;
  __shared__ double2 lds[2 * RW * LINE];
  int f = threadIdx.x / GT;  // 0: q+iv, 1: q+iu
  if constexpr (GT % 64 == 0) f = __builtin_amdgcn_readfirstlane(f);
  const int t = threadIdx.x % GT, rw = t / TPL, j = t % TPL;
  const int yrow = xcd_remap(blockIdx.x, gridDim.x) * RW + rw;
  double2* row = lds + 2 * rw * LINE;
  double2* buf = row + f * LINE;
  const int kxm = a.rc.kx;
  const unsigned fstride = (unsigned)a.ntiles * N * BT;
  const unsigned off = yrow_off(yrow, a.ntiles, BT);
  double2 z[kE], x0[kE], x1[kE];
  load_two<LOGN, TR, BT>(x0, x1, j, a.y1, off, off + (f ? fstride : 2 * fstride), kxm);
  const auto tw = fp_tw<LOGN>(a.tw, j);
  pack_two<LOGN>(z, j, x0, x1);
  if constexpr (IP) {
    fft_dif_held<LOGN, +1>(z, buf, j, tw, false);
    __syncthreads();  // the other wave's reads of the q+iv line
  } else {
    fft_held<LOGN, +1>(z, buf, j, tw);
  }
  double* qv = reinterpret_cast<double*>(row);  // the q+iv line, free again
  if (f == 0) {
#pragma unroll
    for (int r = 0; r < kE; ++r) qv[j + TPL * r] = z[r].x * z[r].y;  // produ.f90:16
  }
  __syncthreads();
  if (f == 1) {
#pragma unroll
    for (int r = 0; r < kE; ++r)
      z[r] = make_double2(z[r].x * z[r].y, qv[j + TPL * r]);  // produ.f90:15
  }
  if constexpr (IP) {
    fft_dit_held<LOGN, -1>(z, buf, j, tw, f == 1);
    __syncthreads();
  } else if (f == 1) {
    fft_held<LOGN, -1>(z, buf, j, tw);
  }
  double2* wl = row + LINE;
  if (f == 1) {
#pragma unroll
    for (int r = 0; r < kE; ++r)
      if (live_r<TR>(r)) (wl + lpad(j))[lpad_off(TPL * r)] = z[r];
  }
  __syncthreads();
  const double2* pm = wl + lpad(TPL - j);
  double2* out = a.y2 + off + (f ? 0u : fstride);
#pragma unroll
  for (int r = 0; r <= kE / 2; ++r) {  // k <= N/2 (r = kE/2 only for k = N/2)
    const int k = j + TPL * r;
    if (live_r<TR>(r) && k <= kxm && k <= N / 2) {
      const double2 W = (wl + lpad(j))[lpad_off(TPL * r)];
      const double2 Wc = mirror_at<LOGN>(wl, pm, j, r);
      out[koff<LOGN, BT>(k)] = f ? make_double2(0.5 * (W.x + Wc.x), 0.5 * (W.y - Wc.y))
                                 : make_double2(0.5 * (W.y + Wc.y), -0.5 * (W.x - Wc.x));
    }
  }
}

// Row-pair variant: each line of N/8 threads handles rows y0 and y0+1
// (group g holds pairs g*NL ..).  The complex transform of Q0 + iQ1 gives q
// of both rows; V0 + iV1 and U0 + iU1 likewise, and the products of the two
// rows are again packed two-for-one for the forward transforms: five
// transforms per row pair, only q carried across them.
template <int LOGN, int TR, int BT, int NL, int SCHED, bool HELD = false>
__device__ __forceinline__ void pair_body(const PassArgs& a, int g, int tid,
                                          double2* lds, const double2* tw) {
  constexpr int N = 1 << LOGN, TPL = N / kE;
  // 1024- to 4096-point lines use the in-place transforms (lines of whole
  // waves): the inverse ones leave x out of order, which the pointwise
  // products do not mind, and the forward ones restore natural order for
  // split_store.
  constexpr bool IP = LOGN >= 10 && LOGN <= 12;
  constexpr int LINE = LOGN >= 10 ? ip_lds<LOGN < 10 ? 10 : LOGN>() : Line<LOGN>::PADDED;
  int pl, j;
  if constexpr (IP) wave_line_map<NL>(tid, pl, j);
  else line_map<TPL, NL>(tid, pl, j);
  double2* buf = lds + pl * LINE;
  const int y0 = 2 * (g * NL + pl);
  const int kxm = a.rc.kx;
  const unsigned fstride = (unsigned)a.ntiles * N * BT;  // one field of y2
  const unsigned r0 = yrow_off(y0, a.ntiles, BT), r1 = r0 + BT;  // rows y0, y0+1 of y2
  // y1: row-pair blocks at N = 4096 (the y pass's layout there), else tiles
  constexpr bool Y1 = LOGN == 12;
  const unsigned cols = Y1 ? (unsigned)y1_cols(a.rc.kc()) : 0u;
  const unsigned fs1 = Y1 ? N * cols : fstride;
  const unsigned i0 = Y1 ? y1_off(y0, 0, cols) : r0, i1 = Y1 ? y1_off(y0 + 1, 0, cols) : r1;
  const unsigned fq = 0, fu = fs1, fv = 2 * fs1;

  constexpr bool IP2 = LOGN == 13;  // 8192: radix 2, then two 4096s
  // HELD: the three twiddles every transform of the thread uses, loaded once
  // (from memory; a table in LDS is read where it is needed)
  IpTw<LOGN> w{};
  if constexpr (IP && HELD) w = ip_tw<LOGN>(tw, j);
  // bar: another wave may still read LDS (ignored by the Stockham transforms,
  // which synchronise on every transpose)
  auto inv = [&](double2* v, bool bar) {
    if constexpr (IP && HELD) fft_dif_held<LOGN, +1>(v, buf, j, w, bar);
    else if constexpr (IP) fft_dif<+1, 1, LOGN>(v, buf, j, tw, bar);
    else if constexpr (IP2) fft_dif2<+1>(v, buf, j, tw, bar);
    else fft_reg<LOGN, +1, SCHED>(v, buf, j, tw);
  };
  auto fwd = [&](double2* v) {
    if constexpr (IP || IP2) {
      if constexpr (IP && HELD) fft_dit_held<LOGN, -1>(v, buf, j, w);
      else if constexpr (IP) fft_dit<-1, false, 1, LOGN>(v, buf, j, tw);
      else fft_dit2<-1>(v, buf, j, tw);
      __syncthreads();  // every wave's reads done before split_store writes
    } else {
      fft_reg<LOGN, -1, SCHED>(v, buf, j, tw);
    }
  };
  double2 z[kE], qq[kE];
  build_two<LOGN, TR, BT, Y1>(z, j, a.y1, fq + i0, fq + i1, kxm);  // Q0 + i Q1
  inv(z, false);  // no LDS reader yet
#pragma unroll
  for (int r = 0; r < kE; ++r) qq[r] = z[r];                   // q0 + i q1
  build_two<LOGN, TR, BT, Y1>(z, j, a.y1, fv + i0, fv + i1, kxm);  // V0 + i V1
  inv(z, true);
#pragma unroll
  for (int r = 0; r < kE; ++r) z[r] = make_double2(qq[r].x * z[r].x, qq[r].y * z[r].y);
  fwd(z);                                                      // (q v)0 + i (q v)1
  split_store<LOGN, TR, BT>(z, buf, j, a.y2, fstride + r0, fstride + r1, kxm);
  build_two<LOGN, TR, BT, Y1>(z, j, a.y1, fu + i0, fu + i1, kxm);  // U0 + i U1
  inv(z, false);  // split_store ends with a barrier
#pragma unroll
  for (int r = 0; r < kE; ++r) z[r] = make_double2(qq[r].x * z[r].x, qq[r].y * z[r].y);
  fwd(z);                                                      // (q u)0 + i (q u)1
  split_store<LOGN, TR, BT>(z, buf, j, a.y2, r0, r1, kxm);
}

// N = 8192, one row per workgroup.  A real row x of N points is the
// M = N/2-point complex sequence z[m] = x[2m] + i x[2m+1]; with
// W = exp(-2 pi i / N) its transform is
//   Z[k] = E[k] + i O[k],  E[k] = X[k] + conj(X[M-k]),
//                          O[k] = (X[k] - conj(X[M-k])) W^-k,
// so the C2R transform of a row is one 4096-point complex transform, and
// the R2C transform of a product p the same backwards: from
// ZP = FFT(p_even + i p_odd),
//   P[k] = PE[k] + W^k PO[k],  PE[k] = (ZP[k] + conj(ZP[M-k])) / 2,
//                              PO[k] = (ZP[k] - conj(ZP[M-k])) / 2i.
// Products stay pointwise in z (even samples in .x, odd in .y), as for row
// pairs.  A row needs one 4096-point line of LDS and 512 threads: two
// workgroups share a CU, where a row pair of 8192-point lines fills one.
// The rectangle lies below 3N/8 (X[k] = 0 from k = 3M/4 on).

// W^(j + 512 r) from wj = W^j (8192-point): W^(512 r) = exp(-i pi r / 8).
template <int R>
__device__ __forceinline__ double2 w_step(double2 wj) {
  constexpr double C1 = 0.92387953251128675613, S1 = 0.38268343236508977173;
  constexpr double H = 0.70710678118654752440;
  if constexpr (R == 0) return wj;
  if constexpr (R == 4) return make_double2(wj.y, -wj.x);
  constexpr double c = R == 1 ? C1 : R == 2 ? H : R == 3 ? S1 : R == 5 ? -S1 : R == 6 ? -H : -C1;
  constexpr double s = R == 1 ? -S1 : R == 2 ? -H : R == 3 ? -C1 : R == 5 ? -C1 : R == 6 ? -H : -S1;
  return cmul(wj, make_double2(c, s));
}
// z[R..7] = E + i O from A = X[k], B = X[M-k], k = j + 512 R.
template <int R>
__device__ __forceinline__ void row_pack(double2* z, const double2* A, const double2* B,
                                         double2 wj) {
  if constexpr (R < kE) {
    const double2 a = A[R], b = B[R];
    const double2 e = make_double2(a.x + b.x, a.y - b.y);
    const double2 o = cmulc(make_double2(a.x - b.x, a.y + b.y), w_step<R>(wj));
    z[R] = make_double2(e.x - o.y, e.y + o.x);
    row_pack<R + 1>(z, A, B, wj);
  }
}
// Z of one row of a field (element k at off + kYR k: tiles of one column).
__device__ __forceinline__ void row_build(double2* z, int j, const double2* __restrict__ y,
                                          unsigned off, int kxm,
                                          const double2* __restrict__ tw) {
  constexpr int M = 4096;
  asm volatile("" : "+v"(j));  // offsets formed here, not held from another field's
  const double2 wj = tw[j];
  double2 A[kE], B[kE];
#pragma unroll
  for (int r = 0; r < kE; ++r) {  // all loads in flight together
    const int k = j + 512 * r, mk = M - k;
    A[r] = B[r] = make_double2(0.0, 0.0);
    if (r < 6 && k <= kxm) A[r] = y[off + ycol_off(k, 1)];    // k < 3M/4
    if (r >= 2 && mk <= kxm) B[r] = y[off + ycol_off(mk, 1)];  // M - k < 3M/4
  }
  if (j == 0) A[0].y = 0.0;  // Im X[0] is not used (C2R)
  row_pack<0>(z, A, B, wj);
}
// Store P[k], k <= kx_max, of the product whose ZP the thread holds in
// natural order (k = j + 512 r).  ZP[M-k] comes through LDS.
__device__ __forceinline__ void row_split_store(const double2* w, double2* buf, int j,
                                                double2* __restrict__ y, unsigned off,
                                                int kxm, const double2* __restrict__ tw) {
  constexpr int TPL = 512;
  asm volatile("" : "+v"(j));
  const double2 wj = tw[j];
  double2* pj = buf + lpad(j);
#pragma unroll
  for (int r = 0; r < kE; ++r) pj[lpad_off(TPL * r)] = w[r];
  __syncthreads();
  const double2* pm = buf + lpad(TPL - j);
  auto one = [&](auto RC) {
    constexpr int r = decltype(RC)::value;
    const int k = j + TPL * r;
    if (k <= kxm) {
      const double2 W = w[r];
      const double2 Wc = mirror_at<12>(buf, pm, j, r);
      const double2 pe = make_double2(0.5 * (W.x + Wc.x), 0.5 * (W.y - Wc.y));
      const double2 po = make_double2(0.5 * (W.y + Wc.y), -0.5 * (W.x - Wc.x));
      y[off + ycol_off(k, 1)] = cadd(pe, cmul(w_step<r>(wj), po));
    }
  };
  one(std::integral_constant<int, 0>{});
  one(std::integral_constant<int, 1>{});
  one(std::integral_constant<int, 2>{});
  one(std::integral_constant<int, 3>{});
  one(std::integral_constant<int, 4>{});
  one(std::integral_constant<int, 5>{});
  __syncthreads();
}
__device__ __forceinline__ void row_body13(const PassArgs& a, int y, int j, double2* buf,
                                           const double2* __restrict__ tw) {
  constexpr int N = 8192;
  const int kxm = a.rc.kx;
  const unsigned fstride = (unsigned)a.ntiles * N;  // one field (tiles of one column)
  const unsigned ro = yrow_off(y, a.ntiles, 1);
  double2 z[kE], qq[kE];
  row_build(z, j, a.y1, ro, kxm, tw);  // Q
  fft_dif<+1, 2>(z, buf, j, tw, false);
#pragma unroll
  for (int r = 0; r < kE; ++r) qq[r] = z[r];  // q_even + i q_odd
  row_build(z, j, a.y1, 2 * fstride + ro, kxm, tw);  // V
  fft_dif<+1, 2>(z, buf, j, tw, true);
#pragma unroll
  for (int r = 0; r < kE; ++r) z[r] = make_double2(qq[r].x * z[r].x, qq[r].y * z[r].y);
  fft_dit<-1, false, 2>(z, buf, j, tw);
  __syncthreads();  // every wave's reads done before the split's writes
  row_split_store(z, buf, j, a.y2, fstride + ro, kxm, tw);  // q v
  row_build(z, j, a.y1, fstride + ro, kxm, tw);  // U
  fft_dif<+1, 2>(z, buf, j, tw, false);  // the split ends with a barrier
#pragma unroll
  for (int r = 0; r < kE; ++r) z[r] = make_double2(qq[r].x * z[r].x, qq[r].y * z[r].y);
  fft_dit<-1, false, 2>(z, buf, j, tw);
  __syncthreads();
  row_split_store(z, buf, j, a.y2, ro, kxm, tw);  // q u
}
template <int LOGN>
__global__ void __launch_bounds__(512, 4) r_pass_row(PassArgs a) {
  static_assert(LOGN == 13, "one-row x pass: 8192-point rows only");
  __shared__ double2 lds[kIpLine];
  row_body13(a, xcd_remap(blockIdx.x, gridDim.x), threadIdx.x, lds, a.tw);
}

// One row pair per workgroup: four workgroups share a CU at N = 2048, two at
// 4096 (at 8192 one fills it: the rectangle wider than 3N/8 only).  Twiddles
// come from memory: the three of a thread loaded once and held, at 8192 each
// where a transform needs it.
template <int LOGN, int TR>
__global__ void __launch_bounds__((1 << LOGN) / kE, 4)
    r_pass_pair(PassArgs a) {
  // Twiddles from memory: these workgroups are short-lived (one row pair),
  // and staging the table in LDS measured slower here.
  __shared__ double2 lds[ip_lds<LOGN>()];
  pair_body<LOGN, TR, bt_of(LOGN), 1, 0, true>(a, xcd_remap(blockIdx.x, gridDim.x),
                                               threadIdx.x, lds, a.tw);
}

// N = 4096 on the 2/3 rectangle: the row pair with sixteen elements a thread
// (pair_body's steps).  A row pair's transforms move a third less through LDS
// and form fewer twiddles; two workgroups of four waves share a CU as two of
// eight did, each lane with twice the loads in flight.  x pass 128 -> 123.5
// us, RK4 step 1130 -> 1105, RK2 549 -> 540 (its memory side alone, without
// transforms, 96 us, the rest with cached lines 104).  On the full rectangle
// the loads of sixteen live positions spill (205 -> 221 us), and the 8192-point
// rows gain 1% (718 -> 712): both keep eight.

// Positions j + 256 r the rectangle can keep (below 3N/8): not r = 6..9.
__device__ __forceinline__ constexpr bool live16(int r) { return r < 6 || r > 9; }
// As build_two / split_store, from the row-pair blocks of y1 and to y2.
__device__ __forceinline__ void build16(double2* z, int j, const double2* __restrict__ y,
                                        unsigned off, int kxm) {
  constexpr int N = 4096;
  double2 x0[16], x1[16];
#pragma unroll
  for (int r = 0; r < 16; ++r) {
    const int p = j + 256 * r, k = r < 8 ? p : N - p;
    x0[r] = x1[r] = make_double2(0.0, 0.0);
    if (live16(r) && k <= kxm) {
      const double2* q = y + off + y1_off(0, k, 0);
      x0[r] = q[0];
      x1[r] = q[1];
    }
  }
#pragma unroll
  for (int r = 0; r < 16; ++r) {
    if ((r == 0 || r == 8) && j == 0) z[r] = make_double2(x0[r].x, x1[r].x);
    else if (r < 8) z[r] = make_double2(x0[r].x - x1[r].y, x0[r].y + x1[r].x);
    else z[r] = make_double2(x0[r].x + x1[r].y, x1[r].x - x0[r].y);
  }
}
__device__ __forceinline__ void split16(const double2* w, double2* buf, int j,
                                        double2* __restrict__ y, unsigned off_a, unsigned off_b,
                                        int kxm) {
  double2* pj = buf + lpad(j);
#pragma unroll
  for (int r = 0; r < 16; ++r)
    if (live16(r)) pj[272 * r] = w[r];
  __syncthreads();
  const double2* pm = buf + lpad(256 - j);
#pragma unroll
  for (int r = 0; r <= 8; ++r) {
    const int k = j + 256 * r;
    if (live16(r) && k <= kxm && k <= 2048) {
      const double2 W = w[r];
      const double2 Wc = r == 0 ? (j == 0 ? buf : pm + 272 * 15)[0] : pm[272 * (15 - r)];
      y[off_a + koff<12, 2>(k)] = make_double2(0.5 * (W.x + Wc.x), 0.5 * (W.y - Wc.y));
      y[off_b + koff<12, 2>(k)] = make_double2(0.5 * (W.y + Wc.y), -0.5 * (W.x - Wc.x));
    }
  }
  __syncthreads();
}
template <int LOGN>
__global__ void __launch_bounds__(256, 2) r_pass_pair16(PassArgs a) {
  static_assert(LOGN == 12, "row pairs of 4096 points");
  __shared__ double2 buf[kLine16];
  const int j = threadIdx.x;
  const int y0 = 2 * xcd_remap(blockIdx.x, gridDim.x);
  const int kxm = a.rc.kx;
  const unsigned fstride = (unsigned)a.ntiles * 4096 * 2;
  const unsigned r0 = yrow_off(y0, a.ntiles, 2), r1 = r0 + 2;
  const unsigned cols = (unsigned)y1_cols(a.rc.kc());
  const unsigned fs1 = 4096 * cols;
  const unsigned i0 = y1_off(y0, 0, cols);
  const Tw16 w = tw16(a.tw, j);
  double2 z[16], qq[16];
  build16(z, j, a.y1, i0, kxm);
  dif16<+1>(z, buf, j, w, false);
#pragma unroll
  for (int r = 0; r < 16; ++r) qq[r] = z[r];
  build16(z, j, a.y1, 2 * fs1 + i0, kxm);
  dif16<+1>(z, buf, j, w, true);
#pragma unroll
  for (int r = 0; r < 16; ++r) z[r] = make_double2(qq[r].x * z[r].x, qq[r].y * z[r].y);
  dit16<-1>(z, buf, j, w);
  __syncthreads();
  split16(z, buf, j, a.y2, fstride + r0, fstride + r1, kxm);
  build16(z, j, a.y1, fs1 + i0, kxm);
  dif16<+1>(z, buf, j, w, false);
#pragma unroll
  for (int r = 0; r < 16; ++r) z[r] = make_double2(qq[r].x * z[r].x, qq[r].y * z[r].y);
  dit16<-1>(z, buf, j, w);
  __syncthreads();
  split16(z, buf, j, a.y2, r0, r1, kxm);
}

// ---------------------------------------------------------------------------
// 2D transforms of a physical field in the reference layout (real rows of
// N+2 doubles; src/fft_dir.f90, src/fft_inv.f90) to and from a spectrum in
// the compact layout.  The x transforms (io_rows_*) and y transforms
// (io_cols_*) meet in the passes' block layout: the y part then reads and
// writes whole blocks on one side and contiguous columns on the other, and
// only the kept columns travel.  A y transform in place on the reference
// layout touches 16 or 32 bytes of each row's line.  Both directions with
// trunc between them, 4096^2: 505 us with transforms in the reference layout
// and gather/scatter, 242 us; 8192^2: 3040 and 1163 us.
// ---------------------------------------------------------------------------

// Physical row held by slot s of a column: the in-place transforms' order at
// N = 4096 and 8192 (see c_body), else s.
template <int LOGN>
__device__ __forceinline__ int slot_row(int s) {
  if constexpr (LOGN == 12) return ip_row<12>(s & 511, s >> 9);
  else if constexpr (LOGN == 13) return 2 * ip_row<12>(s & 511, s >> 10) + ((s >> 9) & 1);
  else return s;
}

// Row pairs per workgroup of the x parts: one wave's worth of short lines.
__host__ __device__ constexpr int io_pairs(int logn) {
  return logn >= 9 ? 1 : logn == 4 ? 8 : 512 >> logn;
}
template <int LOGN, int S>
__device__ __forceinline__ void io_fft(double2* w, double2* buf, int j,
                                       const double2* __restrict__ tw) {
  if constexpr (line_in_wave<LOGN>()) fft_held<LOGN, S>(w, buf, j, held_tw<LOGN>(tw, j));
  else fft_reg<LOGN, S>(w, buf, j, tw);
}

// Slots 2i, 2i+1 (two real rows per complex transform) -> block layout,
// columns kx <= kxm.
template <int LOGN>
__global__ void __launch_bounds__(io_pairs(LOGN) * (1 << LOGN) / kE)
    io_rows_fwd(const double* __restrict__ z, const double2* __restrict__ tw,
                double2* __restrict__ y, int ntiles, int kxm) {
  constexpr int N = 1 << LOGN, TPL = N / kE, RP = io_pairs(LOGN), BT = bt_of(LOGN);
  constexpr int LINE = Line<LOGN>::PADDED;
  __shared__ double2 lds[RP * LINE];
  const int pl = threadIdx.x / TPL, j = threadIdx.x % TPL;
  const int s0 = 2 * (xcd_remap(blockIdx.x, gridDim.x) * RP + pl);
  double2* buf = lds + pl * LINE;
  const size_t ld = (size_t)N + 2;
  const double* r0 = z + ld * slot_row<LOGN>(s0);
  const double* r1 = z + ld * slot_row<LOGN>(s0 + 1);
  double2 w[kE];
#pragma unroll
  for (int r = 0; r < kE; ++r) {
    const int x = j + TPL * r;
    w[r] = make_double2(r0[x], r1[x]);
  }
  io_fft<LOGN, -1>(w, buf, j, tw);
  if constexpr (line_in_wave<LOGN>()) wave_sync();
  const unsigned off = yrow_off(s0, ntiles, BT);
  split_store<LOGN, 0, BT>(w, buf, j, y, off, off + BT, kxm);
}

template <int LOGN>
__global__ void __launch_bounds__(io_pairs(LOGN) * (1 << LOGN) / kE)
    io_rows_inv(double* __restrict__ z, const double2* __restrict__ tw,
                const double2* __restrict__ y, int ntiles, int kxm) {
  constexpr int N = 1 << LOGN, TPL = N / kE, RP = io_pairs(LOGN), BT = bt_of(LOGN);
  constexpr int LINE = Line<LOGN>::PADDED;
  __shared__ double2 lds[RP * LINE];
  const int pl = threadIdx.x / TPL, j = threadIdx.x % TPL;
  const int s0 = 2 * (xcd_remap(blockIdx.x, gridDim.x) * RP + pl);
  double2* buf = lds + pl * LINE;
  const unsigned off = yrow_off(s0, ntiles, BT);
  double2 w[kE];
  build_two<LOGN, 0, BT>(w, j, y, off, off + BT, kxm);
  io_fft<LOGN, +1>(w, buf, j, tw);
  const size_t ld = (size_t)N + 2;
  double* r0 = z + ld * slot_row<LOGN>(s0);
  double* r1 = z + ld * slot_row<LOGN>(s0 + 1);
#pragma unroll
  for (int r = 0; r < kE; ++r) {
    const int x = j + TPL * r;
    r0[x] = w[r].x;
    r1[x] = w[r].y;
  }
  if (j < 2) {
    r0[N + j] = 0.0;
    r1[N + j] = 0.0;
  }
}

// Columns per workgroup of the y parts.
__host__ __device__ constexpr int io_cols(int logn) {
  return logn <= 8 ? 512 >> logn : bt_of(logn);
}
template <int LOGN>
__host__ __device__ constexpr int io_line() {
  return LOGN == 12 ? kIpLine : LOGN == 13 ? 2 * kIpLine : Line<LOGN>::PADDED;
}
// Thread -> (column in workgroup, index in line); each line whole waves (or
// a wave's share) as the in-place transforms need.
template <int LOGN>
__device__ __forceinline__ void io_map(int tid, int& b, int& j) {
  constexpr int TPL = (1 << LOGN) / kE;
  if constexpr (LOGN == 12) {
    wave_line_map<2>(tid, b, j);
  } else {
    b = tid / TPL;
    j = tid % TPL;
  }
}

// Block layout -> compact column, /NY/NX (src/fft_dir.f90:19; a power of
// two: exact), with the mask of src/trunc.f90 when apply_trunc is set.  mark
// (if set) lies in the physical field, which io_rows_fwd has read by now.
template <int LOGN>
__global__ void __launch_bounds__(io_cols(LOGN) * (1 << LOGN) / kE)
    io_cols_fwd(Phys ph, const double2* __restrict__ tw, const double2* __restrict__ y,
                int ntiles, Rect rc, int kyp, double2* __restrict__ cmp, int apply_trunc,
                unsigned long long* mark, double2* __restrict__ dual) {
  constexpr int N = 1 << LOGN, TPL = N / kE, CW = io_cols(LOGN), BT = bt_of(LOGN);
  __shared__ double2 lds[CW * io_line<LOGN>()];
  int b, j;
  io_map<LOGN>(threadIdx.x, b, j);
  const int wg = LOGN == 13 ? xcd_remap(blockIdx.x, gridDim.x) : (int)blockIdx.x;
  if (mark != nullptr && blockIdx.x == 0 && threadIdx.x == 0) *mark = kIoMark;
  const int c = wg * CW + b;
  const bool ok = c <= rc.kx;
  double2* buf = lds + b * io_line<LOGN>();
  const unsigned colo = ycol_off(c, BT);
  double2 w[kE];
#pragma unroll
  for (int r = 0; r < kE; ++r)
    w[r] = ok ? y[yrow_off(j + TPL * r, ntiles, BT) + colo] : make_double2(0.0, 0.0);
  if constexpr (LOGN == 12) fft_dit<-1>(w, buf, j, tw);
  else if constexpr (LOGN == 13) fft_dit2<-1>(w, buf, j, tw);
  else io_fft<LOGN, -1>(w, buf, j, tw);
  if (!ok) return;
  const double fkx = (double)c * ph.dkx;
#pragma unroll
  for (int r = 0; r < kE; ++r) {
    const int p = j + TPL * r, row = row_of(p, rc, N);
    if (row < 0) continue;
    double2 v = make_double2(w[r].x * ph.inv_n2, w[r].y * ph.inv_n2);
    const double fky = (double)kyi_of(p, N) * ph.dky;
    if (apply_trunc && (cut_mode(ph, fkx * fkx, fky * fky) || (c == 0 && p == 0)))
      v = make_double2(0.0, 0.0);
    cmp[(size_t)c * kyp + row] = v;
    if (LOGN <= kIoDirect && dual != nullptr) dual[(size_t)p * (N / 2 + 1) + c] = v;
  }
}

// Column of a spectrum (element (c, row) at c cs + row rs; zero outside the
// rectangle) -> block layout.
template <int LOGN>
__global__ void __launch_bounds__(io_cols(LOGN) * (1 << LOGN) / kE)
    io_cols_inv(const double2* __restrict__ tw, double2* __restrict__ y, int ntiles, Rect rc,
                int cs, int rs, const double2* __restrict__ cmp) {
  constexpr int N = 1 << LOGN, TPL = N / kE, CW = io_cols(LOGN), BT = bt_of(LOGN);
  __shared__ double2 lds[CW * io_line<LOGN>()];
  int b, j;
  io_map<LOGN>(threadIdx.x, b, j);
  const int wg = LOGN == 13 ? xcd_remap(blockIdx.x, gridDim.x) : (int)blockIdx.x;
  const int c = wg * CW + b;
  const bool ok = c <= rc.kx;
  double2* buf = lds + b * io_line<LOGN>();
  double2 w[kE];
#pragma unroll
  for (int r = 0; r < kE; ++r) {
    const int row = row_of(j + TPL * r, rc, N);
    w[r] = ok && row >= 0 ? cmp[(size_t)c * cs + (size_t)row * rs] : make_double2(0.0, 0.0);
  }
  if constexpr (LOGN == 12) fft_dif<+1>(w, buf, j, tw, false);
  else if constexpr (LOGN == 13) fft_dif2<+1>(w, buf, j, tw, false);
  else io_fft<LOGN, +1>(w, buf, j, tw);
  if (!ok) return;
  const unsigned colo = ycol_off(c, BT);
#pragma unroll
  for (int r = 0; r < kE; ++r) y[yrow_off(j + TPL * r, ntiles, BT) + colo] = w[r];
}

// ---------------------------------------------------------------------------
// Adjoint passes.  With q, u, v the physical fields of a stage state s and
// lambda_x,y = G(i k_x,y a) those of the adjoint input a (G the unscaled
// inverse transform, F = G^-1), the transpose of the linearised nonlinear
// term in the Parseval inner product is
//   J(s)^T a = P [ F(u lambda_x + v lambda_y)
//                  + (-i k_y F(q lambda_x) + i k_x F(q lambda_y)) / |k|^alpha ]
// (P the 2/3 mask, the mean mode zero).  The adjoint y pass holds the
// forward y transforms of the three products and their combination, the
// reversed RK stage (JMode) and the inverse y transforms of lambda_x,
// lambda_y, q, u, v for the next transposed term; the adjoint x pass forms
// the products.
// ---------------------------------------------------------------------------

// What the reversed stage of an adjoint y pass reads of one mode.
struct JIn {
  double E;
  double2 mu, l;
};
template <int MODE>
__device__ __forceinline__ JIn j_load(const AdjArgs& a, unsigned q, bool mean) {
  JIn in{};
  if constexpr (MODE != J_END) in.E = a.emk[q];
  if constexpr (MODE != J_START4 && MODE != J_START2) in.l = a.lacc[q];
  if constexpr (MODE != J_END && MODE != J_BOUND4 && MODE != J_BOUND2)
    in.mu = mean ? make_double2(0.0, 0.0) : a.lam[q];
  return in;
}
// The transposed term of one mode from the forward transforms C = F(q
// lambda_x), Z = F(q lambda_y) (j_oper) and D = F(u lambda_x + v lambda_y),
// with fft_dir's 1/N^2.
__device__ __forceinline__ double2 j_oper(double2 C, double2 Z, double fkx, double fky,
                                          double kar) {
  return make_double2((fky * C.y - fkx * Z.y) / kar, (fkx * Z.x - fky * C.x) / kar);
}
__device__ __forceinline__ double2 j_term(const Phys& ph, double2 D, double2 v, double fkxs,
                                          double fky, bool mean) {
  if (mean || (ph.truncate == 1 && cut_mode(ph, fkxs, fky * fky))) return make_double2(0.0, 0.0);
  return make_double2((D.x + v.x) * ph.inv_n2, (D.y + v.y) * ph.inv_n2);
}
// The reversed stage (JMode) with transposed term t: stores lam / lacc and
// returns the adjoint input of the next transposed term.
template <int MODE>
__device__ __forceinline__ double2 j_update(const AdjArgs& a, unsigned q, bool mean, double2 t,
                                            const JIn& in) {
  const Phys& ph = a.ph;
  const double E = in.E;
  const double2 mu = in.mu;
  double2 l = in.l;
  if constexpr (MODE == J_END || MODE == J_BOUND4 || MODE == J_BOUND2) {
    double2 m = make_double2(l.x + t.x, l.y + t.y);
    a.lam[q] = m;
    if constexpr (MODE == J_END) return m;
    if (mean) m = make_double2(0.0, 0.0);
    const double EE = E * E;
    a.lacc[q] = make_double2(EE * m.x, EE * m.y);
    if constexpr (MODE == J_BOUND4) return make_double2(ph.dt6 * m.x, ph.dt6 * m.y);
    else return make_double2(ph.dt * E * m.x, ph.dt * E * m.y);
  } else if constexpr (MODE == J_START4 || MODE == J_START2) {
    const double EE = E * E;
    a.lacc[q] = make_double2(EE * mu.x, EE * mu.y);
    if constexpr (MODE == J_START4) return make_double2(ph.dt6 * mu.x, ph.dt6 * mu.y);
    else return make_double2(ph.dt * E * mu.x, ph.dt * E * mu.y);
  } else {
    double2 av;
    if constexpr (MODE == J_RK4_3) {
      const double EE = E * E;
      l = make_double2(l.x + EE * t.x, l.y + EE * t.y);
      av = make_double2(ph.dt3 * E * mu.x + ph.dt * E * t.x, ph.dt3 * E * mu.y + ph.dt * E * t.y);
    } else if constexpr (MODE == J_RK4_2) {
      l = make_double2(l.x + E * t.x, l.y + E * t.y);
      av = make_double2(ph.dt3 * E * mu.x + ph.dt2 * t.x, ph.dt3 * E * mu.y + ph.dt2 * t.y);
    } else if constexpr (MODE == J_RK4_1) {
      const double EE = E * E;
      l = make_double2(l.x + E * t.x, l.y + E * t.y);
      av = make_double2(ph.dt6 * EE * mu.x + ph.dt2 * E * t.x,
                        ph.dt6 * EE * mu.y + ph.dt2 * E * t.y);
    } else {  // J_RK2_1
      l = make_double2(l.x + E * t.x, l.y + E * t.y);
      av = make_double2(ph.dt2 * E * t.x, ph.dt2 * E * t.y);
    }
    a.lacc[q] = l;
    return av;
  }
}
// Value of one mode in inverse transform f of an adjoint y pass: i kx a, i ky
// a of the adjoint input, then q, u, v of the stage state.
__device__ __forceinline__ double2 j_field(int f, double2 v, double fkx, double fky, double kar) {
  if (f == 0) return make_double2(-fkx * v.y, fkx * v.x);
  if (f == 1) return make_double2(-fky * v.y, fky * v.x);
  return field_of(f - 2, v, fkx, fky, kar);
}

template <int LOGN, int MODE, int AK, int TR>
__global__ void __launch_bounds__(bt_of(LOGN) * (1 << LOGN) / kE, AK == 1 ? 4 : 1)
    j_pass(AdjArgs a) {
  constexpr int N = 1 << LOGN, TPL = N / kE, BT = bt_of(LOGN);
  constexpr int LINE = Line<LOGN>::PADDED;
  constexpr bool FWD = MODE != J_START4 && MODE != J_START2;
  constexpr bool INV = MODE != J_END;
  __shared__ double2 lds[BT * LINE];
  __shared__ double2 twl[tw_lds_size<LOGN>()];
  const double2* tw = stage_tw<LOGN>(twl, a.tw, threadIdx.x, blockDim.x);
  int b, j;
  line_map<TPL, BT>(threadIdx.x, b, j);
  const int tile = blockIdx.x;
  const int c = tile * BT + b;
  const Rect rc = a.rc;
  const bool colok = c <= rc.kx;
  double2* buf = lds + b * LINE;
  const Phys& ph = a.ph;
  const double fkx = (double)c * ph.dkx;
  const double fkxs = fkx * fkx;
  const unsigned cbase = (unsigned)c * (unsigned)a.kyp;
  double2 z[kE];
  double2 av[kE];  // adjoint input of the next transposed term

  if constexpr (FWD) {
    double2 C[kE];
    const double2* y2 = a.y2;
    const size_t fs = (size_t)a.ntiles * N * BT;
    const unsigned colo = ycol_off(c, BT);
#pragma unroll
    for (int r = 0; r < kE; ++r) z[r] = y2[fs + yrow_off(j + TPL * r, a.ntiles, BT) + colo];
    fft_reg<LOGN, -1>(z, buf, j, tw);  // F(q lambda_x)
#pragma unroll
    for (int r = 0; r < kE; ++r) C[r] = live_r<TR>(r) ? z[r] : make_double2(0.0, 0.0);
#pragma unroll
    for (int r = 0; r < kE; ++r) z[r] = y2[2 * fs + yrow_off(j + TPL * r, a.ntiles, BT) + colo];
    fft_reg<LOGN, -1>(z, buf, j, tw);  // F(q lambda_y)
    int jc = j;
    asm volatile("" : "+v"(jc) : "v"(z[0].x), "v"(z[kE - 1].y));
#pragma unroll
    for (int r = 0; r < kE; ++r) {
      const int p = jc + TPL * r;
      double2 v = make_double2(0.0, 0.0);
      if (live_r<TR>(r) && colok && row_of(p, rc, N) >= 0 && !(c == 0 && p == 0)) {
        const double fky = (double)kyi_of(p, N) * ph.dky;
        const double k2 = fkxs + fky * fky;
        v = j_oper(C[r], z[r], fkx, fky, AK == 1 ? k2 : kalpha(ph, k2));
      }
      C[r] = v;
    }
#pragma unroll
    for (int r = 0; r < kE; ++r) z[r] = y2[yrow_off(j + TPL * r, a.ntiles, BT) + colo];
    fft_reg<LOGN, -1>(z, buf, j, tw);  // F(u lambda_x + v lambda_y)
    int je = j;
    asm volatile("" : "+v"(je) : "v"(z[0].x), "v"(z[kE - 1].y));
#pragma unroll
    for (int r = 0; r < kE; ++r) {
      const int p = je + TPL * r;
      const int row = row_of(p, rc, N);
      av[r] = make_double2(0.0, 0.0);
      if (live_r<TR>(r) && colok && row >= 0) {
        const double fky = (double)kyi_of(p, N) * ph.dky;
        const bool mean = (c == 0 && p == 0);
        const unsigned q = cbase + (unsigned)row;
        const double2 t = j_term(ph, z[r], C[r], fkxs, fky, mean);
        av[r] = j_update<MODE>(a, q, mean, t, j_load<MODE>(a, q, mean));
      }
    }
  } else {
#pragma unroll
    for (int r = 0; r < kE; ++r) {
      const int p = j + TPL * r;
      const int row = row_of(p, rc, N);
      av[r] = make_double2(0.0, 0.0);
      if (live_r<TR>(r) && colok && row >= 0) {
        const unsigned q = cbase + (unsigned)row;
        const bool mean = c == 0 && p == 0;
        av[r] = j_update<MODE>(a, q, mean, av[r], j_load<MODE>(a, q, mean));
      }
    }
  }

  if constexpr (INV) {
#pragma unroll 1
    for (int f = 0; f < 5; ++f) {
      int jo = j;
      asm volatile("" : "+v"(jo));
#pragma unroll
      for (int r = 0; r < kE; ++r) {
        const int p = jo + TPL * r;
        const int row = row_of(p, rc, N);
        double2 v = make_double2(0.0, 0.0);
        if (live_r<TR>(r) && colok && row >= 0) {
          const double fky = (double)kyi_of(p, N) * ph.dky;
          const double k2 = fkxs + fky * fky;
          if (f < 3 || !(c == 0 && p == 0))  // u, v: src/nlt.f90:25-34
            v = j_field(f, f < 2 ? av[r] : a.snext[cbase + (unsigned)row], fkx, fky,
                        AK == 1 || f < 3 ? k2 : kalpha(ph, k2));
        }
        z[r] = v;
      }
      fft_reg<LOGN, +1>(z, buf, j, tw);
      double2* dst = a.y1 + (size_t)f * a.ntiles * N * BT;
      const unsigned colo = ycol_off(c, BT);
#pragma unroll
      for (int r = 0; r < kE; ++r) dst[yrow_off(j + TPL * r, a.ntiles, BT) + colo] = z[r];
    }
  }
}

// Half-spectrum (kx <= kx_max) of one real row -> its full x-spectrum at
// the thread's positions (as build_two with g = 0).
template <int LOGN, int TR, int BT>
__device__ __forceinline__ void build_one(double2* z, int j, const double2* __restrict__ y,
                                          unsigned off, int kxm) {
  constexpr int N = 1 << LOGN, TPL = N / kE;
#pragma unroll
  for (int r = 0; r < kE; ++r) {
    const int p = j + TPL * r;
    double2 v = make_double2(0.0, 0.0);
    const int k = p <= N / 2 ? p : N - p;
    if (live_r<TR>(r) && k <= kxm) {
      const double2 x0 = y[off + koff<LOGN, BT>(k)];
      if (p == 0 || p == N / 2) v = make_double2(x0.x, 0.0);
      else if (p < N / 2) v = x0;
      else v = make_double2(x0.x, -x0.y);
    }
    z[r] = v;
  }
}

// Adjoint x pass, one row per line: C2R of lambda_x + i lambda_y, of q + i u
// and of v; R2C of q lambda_x + i q lambda_y and of u lambda_x + v lambda_y.
template <int LOGN, int TR>
__global__ void __launch_bounds__(rows_of(LOGN) * (1 << LOGN) / kE)
    jr_pass(AdjArgs a) {
  constexpr int N = 1 << LOGN, TPL = N / kE, RP = rows_of(LOGN), BT = bt_of(LOGN);
  constexpr int LINE = Line<LOGN>::PADDED;
  __shared__ double2 lds[RP * LINE];
  __shared__ double2 twl[tw_lds_size<LOGN>()];
  const double2* tw = stage_tw<LOGN>(twl, a.tw, threadIdx.x, blockDim.x);
  int pl, j;
  line_map<TPL, RP>(threadIdx.x, pl, j);
  const int yrow = xcd_remap(blockIdx.x, gridDim.x) * RP + pl;
  double2* buf = lds + pl * LINE;
  const int kxm = a.rc.kx;
  const unsigned fs = (unsigned)a.ntiles * N * BT;
  const unsigned off = yrow_off(yrow, a.ntiles, BT);

  double2 z[kE], l[kE];
  double ap[kE];
  build_two<LOGN, TR, BT>(z, j, a.y1, off, off + fs, kxm);  // LX + i LY
  fft_reg<LOGN, +1>(z, buf, j, tw);
#pragma unroll
  for (int r = 0; r < kE; ++r) l[r] = z[r];                   // lambda_x + i lambda_y
  build_two<LOGN, TR, BT>(z, j, a.y1, off + 2 * fs, off + 3 * fs, kxm);  // Q + i U
  fft_reg<LOGN, +1>(z, buf, j, tw);
#pragma unroll
  for (int r = 0; r < kE; ++r) {
    ap[r] = z[r].y * l[r].x;                                  // u lambda_x
    z[r] = make_double2(z[r].x * l[r].x, z[r].x * l[r].y);    // q lambda_x + i q lambda_y
  }
  fft_reg<LOGN, -1>(z, buf, j, tw);
  split_store<LOGN, TR, BT>(z, buf, j, a.y2, off + fs, off + 2 * fs, kxm);
  build_one<LOGN, TR, BT>(z, j, a.y1, off + 4 * fs, kxm);   // V
  fft_reg<LOGN, +1>(z, buf, j, tw);
#pragma unroll
  for (int r = 0; r < kE; ++r) z[r] = make_double2(ap[r] + z[r].x * l[r].y, 0.0);
  fft_reg<LOGN, -1>(z, buf, j, tw);                          // F(u lambda_x + v lambda_y)
#pragma unroll
  for (int r = 0; r <= kE / 2; ++r) {
    const int k = j + TPL * r;
    if (live_r<TR>(r) && k <= kxm && k <= N / 2) a.y2[off + koff<LOGN, BT>(k)] = z[r];
  }
}

// Small grids (see f_pass): the adjoint passes with a column's three forward
// and five inverse transforms, and a row's three inverse and two forward
// ones, on their own threads: two transforms deep instead of eight and five.
// 512^2, alpha 1: y stage 25.2 -> 10.0 us, x pass 12.0 -> 9.0, and a step's
// end and the next one's start (10.0 + 18.1 us) in one pass, 10.1; results
// bit-identical.  At 1024^2 a column fills 104 KB of LDS and the passes in
// turn stay ahead: a gradient step 541 us, 582 with these.
template <int LOGN, int MODE, int AK>
__global__ void __launch_bounds__(fp_cols(LOGN) * 5 * (1 << LOGN) / kE) fj_pass(AdjArgs a) {
  constexpr int N = 1 << LOGN, TPL = N / kE, BT = bt_of(LOGN), CW = fp_cols(LOGN);
  constexpr int LINE = Line<LOGN>::PADDED, GT = CW * TPL;
  constexpr bool FWD = MODE != J_START4 && MODE != J_START2;
  constexpr bool INV = MODE != J_END;
  constexpr int NLINE = INV ? 6 : 3;  // a line per field, the adjoint input
  static_assert(GT % 64 == 0 && line_in_wave<LOGN>(), "whole waves per field");
  __shared__ double2 lds[CW * NLINE * LINE];
  const int f = __builtin_amdgcn_readfirstlane(threadIdx.x / GT);
  const int t = threadIdx.x % GT, cw = t / TPL, j = t % TPL;
  const int c = CW == 1 ? xcd_remap(blockIdx.x, gridDim.x) : (int)blockIdx.x * CW + cw;
  const Rect rc = a.rc;
  const bool colok = c <= rc.kx;
  const Phys& ph = a.ph;
  const double fkx = (double)c * ph.dkx;
  const double fkxs = fkx * fkx;
  const unsigned cbase = (unsigned)c * (unsigned)a.kyp;
  const unsigned colo = ycol_off(c, BT);
  const size_t fs = (size_t)a.ntiles * N * BT;
  double2* col = lds + cw * NLINE * LINE;
  double2* buf = col + (NLINE == 6 || f < 3 ? f : 0) * LINE;
  double2* abuf = col + 5 * LINE;

  double2 z[kE], sv[kE];
  double ka[kE];
  if constexpr (FWD) {
    if (f < 3) {  // F(q lambda_x), F(q lambda_y), F(u lambda_x + v lambda_y)
      const double2* src = a.y2 + (f == 2 ? 0 : (f + 1) * fs);
#pragma unroll
      for (int r = 0; r < kE; ++r)
        z[r] = colok ? src[yrow_off(j + TPL * r, a.ntiles, BT) + colo] : make_double2(0.0, 0.0);
    }
  }
  const HeldTw<LOGN> tw = held_tw<LOGN>(a.tw, j);
  int pos[2];
  bool own[2];
  unsigned qi[2];
  JIn in[2];
  double kao[2];
#pragma unroll
  for (int i = 0; i < 2; ++i) {  // modes this thread updates (fields 0-2)
    const int x = 2 * f + i, r = x >= 3 ? x + 2 : x;
    pos[i] = j + TPL * r;
    const int row = f < 3 ? row_of(pos[i], rc, N) : -1;
    own[i] = colok && row >= 0;
    qi[i] = cbase + (unsigned)row;
    in[i] = own[i] ? j_load<MODE>(a, qi[i], c == 0 && pos[i] == 0) : JIn{};
    kao[i] = AK == 2 && FWD && own[i] ? a.ka[qi[i]] : 1.0;
  }
  if constexpr (INV) {
#pragma unroll
    for (int r = 0; r < kE; ++r) {  // the stage state of the next transposed term
      const int row = row_of(j + TPL * r, rc, N);
      const bool ok = f >= 2 && live_r<1>(r) && colok && row >= 0;
      sv[r] = ok ? a.snext[cbase + (unsigned)row] : make_double2(0.0, 0.0);
      ka[r] = AK == 2 && ok && f > 2 ? a.ka[cbase + (unsigned)row] : 1.0;
    }
  }
  if constexpr (FWD) {
    if (f < 3) {
      fft_held<LOGN, -1>(z, buf, j, tw);
#pragma unroll
      for (int r = 0; r < kE; ++r)
        if (live_r<1>(r)) (buf + lpad(j))[lpad_off(TPL * r)] = z[r];
    }
    __syncthreads();
  }
  if (f < 3) {
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      double2 v = make_double2(0.0, 0.0);
      if (own[i]) {
        const int p = pos[i], e = lpad(p);
        const bool mean = c == 0 && p == 0;
        double2 tm = v;
        if constexpr (FWD) {
          const double fky = (double)kyi_of(p, N) * ph.dky;
          if (!mean)
            tm = j_oper(col[e], col[LINE + e], fkx, fky, AK == 1 ? fkxs + fky * fky : kao[i]);
          tm = j_term(ph, col[2 * LINE + e], tm, fkxs, fky, mean);
        }
        v = j_update<MODE>(a, qi[i], mean, tm, in[i]);
      }
      if constexpr (INV) abuf[lpad(pos[i])] = v;
    }
  }
  if constexpr (INV) {
    __syncthreads();
#pragma unroll
    for (int r = 0; r < kE; ++r) {
      z[r] = make_double2(0.0, 0.0);
      if (!live_r<1>(r)) continue;
      const int p = j + TPL * r;
      const double fky = (double)kyi_of(p, N) * ph.dky;
      const double2 av = (abuf + lpad(j))[lpad_off(TPL * r)];
      const double2 v = make_double2(f < 2 ? av.x : sv[r].x, f < 2 ? av.y : sv[r].y);
      if (f < 3 || !(c == 0 && p == 0))
        z[r] = j_field(f, v, fkx, fky, AK == 1 || f < 3 ? fkxs + fky * fky : ka[r]);
    }
    fft_held<LOGN, +1>(z, buf, j, tw);
    if (colok) {
      double2* dst = a.y1 + f * fs;
#pragma unroll
      for (int r = 0; r < kE; ++r) dst[yrow_off(j + TPL * r, a.ntiles, BT) + colo] = z[r];
    }
  }
}

template <int LOGN>
__global__ void __launch_bounds__(3 * fx_rows(LOGN) * (1 << LOGN) / kE) fjr_pass(AdjArgs a) {
  constexpr int N = 1 << LOGN, TPL = N / kE, BT = bt_of(LOGN), RW = fx_rows(LOGN);
  constexpr int LINE = Line<LOGN>::PADDED, GT = RW * TPL;
  static_assert(line_in_wave<LOGN>(), "a line inside a wave");
  __shared__ double2 lds[4 * RW * LINE];
  int f = threadIdx.x / GT;  // 0: lambda_x + i lambda_y, 1: q + iu, 2: v
  if constexpr (GT % 64 == 0) f = __builtin_amdgcn_readfirstlane(f);
  const int t = threadIdx.x % GT, rw = t / TPL, j = t % TPL;
  const int yrow = xcd_remap(blockIdx.x, gridDim.x) * RW + rw;
  double2* row = lds + 4 * rw * LINE;
  double2* buf = row + f * LINE;
  double* ub = reinterpret_cast<double*>(row + 3 * LINE);
  const int kxm = a.rc.kx;
  const unsigned fs = (unsigned)a.ntiles * N * BT;
  const unsigned off = yrow_off(yrow, a.ntiles, BT);
  double2 z[kE];
  {
    double2 x0[kE], x1[kE];
    const unsigned of = off + 2 * f * fs;
    load_two<LOGN, 1, BT>(x0, x1, j, a.y1, of, f == 2 ? of : of + fs, kxm);
    if (f == 2) {
#pragma unroll
      for (int r = 0; r < kE; ++r) x1[r] = make_double2(0.0, 0.0);
    }
    pack_two<LOGN>(z, j, x0, x1);
  }
  const HeldTw<LOGN> tw = held_tw<LOGN>(a.tw, j);
  fft_held<LOGN, +1>(z, buf, j, tw);
  if (f == 0) {
#pragma unroll
    for (int r = 0; r < kE; ++r) (buf + lpad(j))[lpad_off(TPL * r)] = z[r];
  } else if (f == 1) {
#pragma unroll
    for (int r = 0; r < kE; ++r) ub[j + TPL * r] = z[r].y;
  }
  __syncthreads();
  if (f > 0) {
#pragma unroll
    for (int r = 0; r < kE; ++r) {
      const double2 l = (row + lpad(j))[lpad_off(TPL * r)];
      z[r] = f == 1 ? make_double2(z[r].x * l.x, z[r].x * l.y)  // q lambda_x + i q lambda_y
                    : make_double2(ub[j + TPL * r] * l.x + z[r].x * l.y, 0.0);
    }
    fft_held<LOGN, -1>(z, buf, j, tw);
  }
  if (f == 1) {
#pragma unroll
    for (int r = 0; r < kE; ++r)
      if (live_r<1>(r)) (buf + lpad(j))[lpad_off(TPL * r)] = z[r];
  }
  __syncthreads();
  double2* wl = row + LINE;
  const double2* pm = wl + lpad(TPL - j);
  double2* out = a.y2 + off + (f == 2 ? 0u : (f + 1) * fs);
#pragma unroll
  for (int r = 0; r <= kE / 2; ++r) {
    const int k = j + TPL * r;
    if (live_r<1>(r) && k <= kxm && k <= N / 2) {
      if (f == 2) {  // F(u lambda_x + v lambda_y)
        out[koff<LOGN, BT>(k)] = z[r];
      } else {
        const double2 W = (wl + lpad(j))[lpad_off(TPL * r)];
        const double2 Wc = mirror_at<LOGN>(wl, pm, j, r);
        out[koff<LOGN, BT>(k)] = f == 0
                                     ? make_double2(0.5 * (W.x + Wc.x), 0.5 * (W.y - Wc.y))
                                     : make_double2(0.5 * (W.y + Wc.y), -0.5 * (W.x - Wc.x));
      }
    }
  }
}

// ---------------------------------------------------------------------------
// launchers.  Each grid size is instantiated in its own translation unit
// (compiled with -DGT_INST_LOGN=L); the dispatchers and the size-independent
// kernels are in the one compiled with -DGT_INST_COMMON.
// ---------------------------------------------------------------------------

template <int L>
hipError_t c_pass_launch(int mode, const PassArgs& a, hipStream_t s);
template <int L>
hipError_t r_pass_launch(const PassArgs& a, hipStream_t s);
template <int L>
hipError_t io_launch(const IoArgs& a, hipStream_t s);
template <int L>
hipError_t j_pass_launch(int mode, const AdjArgs& a, hipStream_t s);
template <int L>
hipError_t jr_pass_launch(const AdjArgs& a, hipStream_t s);
template <int T, int SCHED>
hipError_t ens_c_launch(int mode, const PassArgs* d, const uint32_t* it, int n, int grid,
                        hipStream_t s);
template <int TX, int SCHED>
hipError_t ens_r_launch(int ty, const PassArgs* d, const uint32_t* it, int n, int grid,
                        hipStream_t s);

#if defined(GT_INST_LOGN)
template <int L, int MODE, int AK, int TR>
static void y_launch(const PassArgs& a, hipStream_t s) {
  if constexpr (L <= kFpMaxLogn) {
    constexpr int CW = fp_cols(L);
    const int g = (a.rc.kc() + CW - 1) / CW;
    f_pass<L, MODE, AK, TR><<<dim3(g), dim3(CW * 3 * (1 << L) / kE), 0, s>>>(a);
  } else {
    c_pass<L, MODE, AK, TR><<<dim3(a.ntiles), dim3(bt_of(L) * (1 << L) / kE), 0, s>>>(a);
  }
}
template <int L, int AK, int TR>
static hipError_t c_pass_launch_ak(int mode, const PassArgs& a, hipStream_t s) {
  switch (mode) {
    case C_START: y_launch<L, C_START, AK, TR>(a, s); break;
    case C_NLT: y_launch<L, C_NLT, AK, TR>(a, s); break;
    case C_RK4_1: y_launch<L, C_RK4_1, AK, TR>(a, s); break;
    case C_RK4_2: y_launch<L, C_RK4_2, AK, TR>(a, s); break;
    case C_RK4_3: y_launch<L, C_RK4_3, AK, TR>(a, s); break;
    case C_RK4_4: y_launch<L, C_RK4_4, AK, TR>(a, s); break;
    case C_RK2_1: y_launch<L, C_RK2_1, AK, TR>(a, s); break;
    case C_RK2_2: y_launch<L, C_RK2_2, AK, TR>(a, s); break;
    case C_RK4_4S: y_launch<L, C_RK4_4S, AK, TR>(a, s); break;
    case C_RK2_2S: y_launch<L, C_RK2_2S, AK, TR>(a, s); break;
    default: return hipErrorInvalidValue;
  }
  return hipGetLastError();
}

// TR = 1 when the rectangle lies below 3N/8 on both axes (always so with
// the 2/3 rule); the position set of a thread is j + r*N/8.
__host__ __device__ inline int rect_tr(const Rect& rc, int n) {
  const int lim = 3 * (n / kE);
  return (rc.kx < lim && rc.p < lim && rc.q < lim && n >= 16) ? 1 : 0;
}

template <int L>
hipError_t c_pass_launch(int mode, const PassArgs& a, hipStream_t s) {
  const int tr = rect_tr(a.rc, 1 << L);
  constexpr int AK = L <= kFpMaxLogn ? 2 : 3;
  if (a.ph.akind == 1)
    return tr ? c_pass_launch_ak<L, 1, 1>(mode, a, s) : c_pass_launch_ak<L, 1, 0>(mode, a, s);
  return tr ? c_pass_launch_ak<L, AK, 1>(mode, a, s) : c_pass_launch_ak<L, AK, 0>(mode, a, s);
}

template <int L>
hipError_t r_pass_launch(const PassArgs& a, hipStream_t s) {
  if constexpr (L > kFpMaxLogn) {  // one row pair per workgroup (8192: one row)
    constexpr int T = (1 << L) / kE;
    if (rect_tr(a.rc, 1 << L)) {
      if constexpr (L == 13)
        r_pass_row<L><<<dim3(1 << L), dim3(T / 2), 0, s>>>(a);
      else if constexpr (L == 12)
        r_pass_pair16<L><<<dim3((1 << L) / 2), dim3(T / 2), 0, s>>>(a);
      else
        r_pass_pair<L, 1><<<dim3((1 << L) / 2), dim3(T), 0, s>>>(a);
    } else {
      r_pass_pair<L, 0><<<dim3((1 << L) / 2), dim3(T), 0, s>>>(a);
    }
  } else {
    constexpr int RW = fx_rows(L), T = 2 * RW * (1 << L) / kE;
    if (rect_tr(a.rc, 1 << L))
      fx_pass<L, 1><<<dim3((1 << L) / RW), dim3(T), 0, s>>>(a);
    else
      fx_pass<L, 0><<<dim3((1 << L) / RW), dim3(T), 0, s>>>(a);
  }
  return hipGetLastError();
}

template <int L>
hipError_t io_launch(const IoArgs& a, hipStream_t s) {
  constexpr int N = 1 << L, RP = io_pairs(L), CW = io_cols(L), BT = bt_of(L);
  const dim3 gr(N / 2 / RP), br(RP * N / kE), bc(CW * N / kE);
  const dim3 gc((a.rc.kc() + CW - 1) / CW);
  const int nt = (a.rc.kc() + BT - 1) / BT;
  if (a.dir < 0) {
    io_rows_fwd<L><<<gr, br, 0, s>>>(a.ref, a.tw, a.y, nt, a.rc.kx);
    io_cols_fwd<L><<<gc, bc, 0, s>>>(a.ph, a.tw, a.y, nt, a.rc, a.kyp, a.cmp, a.apply_trunc,
                                       a.mark, a.dual);
  } else {
    io_cols_inv<L><<<gc, bc, 0, s>>>(a.tw, a.y, nt, a.rc, a.kyp, a.rs, a.cmp);
    io_rows_inv<L><<<gr, br, 0, s>>>(a.ref, a.tw, a.y, nt, a.rc.kx);
  }
  return hipGetLastError();
}

template <int L, int MODE, int AK>
static void j_launch(const AdjArgs& a, hipStream_t s) {
  if constexpr (L <= kFjMaxLogn) {
    constexpr int CW = fp_cols(L);
    const int g = (a.rc.kc() + CW - 1) / CW;
    fj_pass<L, MODE, AK><<<dim3(g), dim3(CW * 5 * (1 << L) / kE), 0, s>>>(a);
  } else {
    j_pass<L, MODE, AK, 1><<<dim3(a.ntiles), dim3(bt_of(L) * (1 << L) / kE), 0, s>>>(a);
  }
}
template <int L, int AK>
static hipError_t j_pass_launch_ak(int mode, const AdjArgs& a, hipStream_t s) {
  switch (mode) {
    case J_START4: j_launch<L, J_START4, AK>(a, s); break;
    case J_RK4_3: j_launch<L, J_RK4_3, AK>(a, s); break;
    case J_RK4_2: j_launch<L, J_RK4_2, AK>(a, s); break;
    case J_RK4_1: j_launch<L, J_RK4_1, AK>(a, s); break;
    case J_END: j_launch<L, J_END, AK>(a, s); break;
    case J_START2: j_launch<L, J_START2, AK>(a, s); break;
    case J_RK2_1: j_launch<L, J_RK2_1, AK>(a, s); break;
    case J_BOUND4: j_launch<L, J_BOUND4, AK>(a, s); break;
    case J_BOUND2: j_launch<L, J_BOUND2, AK>(a, s); break;
    default: return hipErrorInvalidValue;
  }
  return hipGetLastError();
}

// The adjoint needs the 2/3 rectangle (TR = 1).
template <int L>
hipError_t j_pass_launch(int mode, const AdjArgs& a, hipStream_t s) {
  constexpr int AK = L <= kFjMaxLogn ? 2 : 0;
  if (!rect_tr(a.rc, 1 << L)) return hipErrorInvalidValue;
  return a.ph.akind == 1 ? j_pass_launch_ak<L, 1>(mode, a, s)
                         : j_pass_launch_ak<L, AK>(mode, a, s);
}

template <int L>
hipError_t jr_pass_launch(const AdjArgs& a, hipStream_t s) {
  if (!rect_tr(a.rc, 1 << L)) return hipErrorInvalidValue;
  if constexpr (L <= kFjMaxLogn) {
    constexpr int RW = fx_rows(L);
    fjr_pass<L><<<dim3((1 << L) / RW), dim3(3 * RW * (1 << L) / kE), 0, s>>>(a);
  } else {
    constexpr int RP = rows_of(L), T = RP * (1 << L) / kE;
    jr_pass<L, 1><<<dim3((1 << L) / RP), dim3(T), 0, s>>>(a);
  }
  return hipGetLastError();
}

template hipError_t j_pass_launch<GT_INST_LOGN>(int, const AdjArgs&, hipStream_t);
template hipError_t jr_pass_launch<GT_INST_LOGN>(const AdjArgs&, hipStream_t);
template hipError_t c_pass_launch<GT_INST_LOGN>(int, const PassArgs&, hipStream_t);
template hipError_t r_pass_launch<GT_INST_LOGN>(const PassArgs&, hipStream_t);
template hipError_t io_launch<GT_INST_LOGN>(const IoArgs&, hipStream_t);
#endif  // GT_INST_LOGN

#if defined(GT_INST_ENS)
// ---------------------------------------------------------------------------
// Batched ensemble passes.  One launch covers the pass of every member,
// whatever its N and alpha: the workgroups loop over a list of work items
// (member, tile) and run the pass body of the member's size.  For T threads
// a workgroup holds T*8/N lines of N points, T*8 elements of any N; padded they
// take T*17/2 double2 of LDS (Stockham lines, N + N/16) or T*9 (in-place lines,
// N + N/8, from 1024 on), so the sizes share one allocation of T*9.  Alpha enters through
// kalpha_t<2>, the x-pass packing per member through PassArgs::xvar, the
// radix order (SCHED) per launch.  Every member has the 2/3 rectangle
// (TR = 1).  Compiled once per (T, SCHED): -DGT_INST_ENS=T
// -DGT_ENS_SCHED=SCHED.
// ---------------------------------------------------------------------------

// Twiddles of the item's size in LDS: staged again only when the member's
// table changes (barriers on both sides: the previous item's last pass may
// still read the old table).
__device__ __forceinline__ const double2* ens_stage_tw(double2* twl, const PassArgs& a,
                                                       const double2*& cur) {
  if (a.tw != cur) {
    __syncthreads();
    const int n = a.ph.n;
    const int span = n == 128 ? tw_span<7>() : n == 256 ? tw_span<8>()
                   : n == 512 ? tw_span<9>() : n == 1024 ? tw_span<10>() : tw_span<11>();
    for (int i = threadIdx.x; i < span; i += blockDim.x) twl[i] = a.tw[i];
    __syncthreads();
    cur = a.tw;
  }
  return twl;
}

template <int T, int MODE, int SCHED, int L>
__device__ __forceinline__ void ens_c_one(const PassArgs& a, int tile, int tid,
                                          double2* lds, const double2* tw) {
  c_body<L, MODE, 2, 1, ens_lines(T, L), SCHED, L >= 10, ens_tile(T, L)>(a, tile, tid,
                                                                               lds, tw);
}

template <int T, int MODE, int SCHED>
__global__ void __launch_bounds__(T, 4)
    ens_c_pass(const PassArgs* __restrict__ descs, const uint32_t* __restrict__ items,
               int nitems) {
  __shared__ double2 lds[T * 9];
  __shared__ double2 twl[tw_span<kEnsMaxLogn>()];
  const double2* cur = nullptr;
  for (int w = blockIdx.x; w < nitems; w += gridDim.x) {
    const uint32_t it = items[w];
    const PassArgs& a = descs[it >> 16];
    const int tile = (int)(it & 0xFFFFu);
    const double2* tw = ens_stage_tw(twl, a, cur);
    // Opaque per item: nothing derived from the thread index is hoisted out
    // of the loop (and kept live over every size's code).
    int tid = threadIdx.x;
    asm volatile("" : "+v"(tid));
    switch (a.ph.n) {
      case 128: ens_c_one<T, MODE, SCHED, 7>(a, tile, tid, lds, tw); break;
      case 256: ens_c_one<T, MODE, SCHED, 8>(a, tile, tid, lds, tw); break;
      case 512: ens_c_one<T, MODE, SCHED, 9>(a, tile, tid, lds, tw); break;
      case 1024: ens_c_one<T, MODE, SCHED, 10>(a, tile, tid, lds, tw); break;
      case 2048: ens_c_one<T, MODE, SCHED, 11>(a, tile, tid, lds, tw); break;
      default: break;
    }
  }
}

template <int TX, int TY, int SCHED, int L>
__device__ __forceinline__ void ens_r_one(const PassArgs& a, int g, int tid, double2* lds,
                                          const double2* tw) {
  constexpr int NL = ens_lines(TX, L), BT = ens_tile(TY, L);
  if (a.xvar) pair_body<L, 1, BT, NL, SCHED>(a, g, tid, lds, tw);
  else r_body<L, 1, BT, NL, SCHED>(a, g, tid, lds, tw);
}

template <int TX, int TY, int SCHED>
__global__ void __launch_bounds__(TX, 4)
    ens_r_pass(const PassArgs* __restrict__ descs, const uint32_t* __restrict__ items,
               int nitems) {
  __shared__ double2 lds[TX * 9];
  __shared__ double2 twl[tw_span<kEnsMaxLogn>()];
  const double2* cur = nullptr;
  for (int w = blockIdx.x; w < nitems; w += gridDim.x) {
    const uint32_t it = items[w];
    const PassArgs& a = descs[it >> 16];
    const int g = (int)(it & 0xFFFFu);
    const double2* tw = ens_stage_tw(twl, a, cur);
    int tid = threadIdx.x;
    asm volatile("" : "+v"(tid));
    switch (a.ph.n) {
      case 128: ens_r_one<TX, TY, SCHED, 7>(a, g, tid, lds, tw); break;
      case 256: ens_r_one<TX, TY, SCHED, 8>(a, g, tid, lds, tw); break;
      case 512: ens_r_one<TX, TY, SCHED, 9>(a, g, tid, lds, tw); break;
      case 1024: ens_r_one<TX, TY, SCHED, 10>(a, g, tid, lds, tw); break;
      case 2048: ens_r_one<TX, TY, SCHED, 11>(a, g, tid, lds, tw); break;
      default: break;
    }
  }
}

template <int T, int SCHED>
hipError_t ens_c_launch(int mode, const PassArgs* d, const uint32_t* it, int n, int grid,
                        hipStream_t s) {
  const dim3 g(grid), b(T);
  switch (mode) {
    case C_START: ens_c_pass<T, C_START, SCHED><<<g, b, 0, s>>>(d, it, n); break;
    case C_RK4_1: ens_c_pass<T, C_RK4_1, SCHED><<<g, b, 0, s>>>(d, it, n); break;
    case C_RK4_2: ens_c_pass<T, C_RK4_2, SCHED><<<g, b, 0, s>>>(d, it, n); break;
    case C_RK4_3: ens_c_pass<T, C_RK4_3, SCHED><<<g, b, 0, s>>>(d, it, n); break;
    case C_RK4_4: ens_c_pass<T, C_RK4_4, SCHED><<<g, b, 0, s>>>(d, it, n); break;
    case C_RK2_1: ens_c_pass<T, C_RK2_1, SCHED><<<g, b, 0, s>>>(d, it, n); break;
    case C_RK2_2: ens_c_pass<T, C_RK2_2, SCHED><<<g, b, 0, s>>>(d, it, n); break;
    case C_RK4_4S: ens_c_pass<T, C_RK4_4S, SCHED><<<g, b, 0, s>>>(d, it, n); break;
    case C_RK2_2S: ens_c_pass<T, C_RK2_2S, SCHED><<<g, b, 0, s>>>(d, it, n); break;
    default: return hipErrorInvalidValue;
  }
  return hipGetLastError();
}

template <int TX, int SCHED>
hipError_t ens_r_launch(int ty, const PassArgs* d, const uint32_t* it, int n, int grid,
                        hipStream_t s) {
  const dim3 g(grid), b(TX);
  if (ty == 256) ens_r_pass<TX, 256, SCHED><<<g, b, 0, s>>>(d, it, n);
  else if (ty == 512) ens_r_pass<TX, 512, SCHED><<<g, b, 0, s>>>(d, it, n);
  else return hipErrorInvalidValue;
  return hipGetLastError();
}

template hipError_t ens_c_launch<GT_INST_ENS, GT_ENS_SCHED>(int, const PassArgs*,
                                                            const uint32_t*, int, int,
                                                            hipStream_t);
template hipError_t ens_r_launch<GT_INST_ENS, GT_ENS_SCHED>(int, const PassArgs*,
                                                            const uint32_t*, int, int,
                                                            hipStream_t);
#endif  // GT_INST_ENS

#if defined(GT_INST_COMMON)
// ---------------------------------------------------------------------------
// Elementwise operators
// ---------------------------------------------------------------------------

// src/produ.f90:11-23
__global__ void produ_k(int n, const double* __restrict__ z, double* u,
                        double* v) {
  const size_t ld = (size_t)n + 2, tot = ld * n;
  for (size_t e = blockIdx.x * (size_t)blockDim.x + threadIdx.x; e < tot;
       e += (size_t)gridDim.x * blockDim.x) {
    const size_t i = e % ld;
    if (i < (size_t)n) {
      u[e] = z[e] * u[e];
      v[e] = z[e] * v[e];
    } else {
      u[e] = 0.0;
      v[e] = 0.0;
    }
  }
}

// src/trunc.f90:10-25 on a compact rectangle.
__global__ void trunc_cmp_k(Phys ph, Rect rc, int kyp, double2* z) {
  const int n = ph.n, ky = rc.ky();
  const size_t tot = (size_t)rc.kc() * ky;
  for (size_t e = blockIdx.x * (size_t)blockDim.x + threadIdx.x; e < tot;
       e += (size_t)gridDim.x * blockDim.x) {
    const int c = (int)(e / ky), r = (int)(e % ky);
    const int p = fft_of(r, rc, n);
    const double fkx = (double)c * ph.dkx, fky = (double)kyi_of(p, n) * ph.dky;
    if (cut_mode(ph, fkx * fkx, fky * fky) || (c == 0 && r == 0))
      z[(size_t)c * kyp + r] = make_double2(0.0, 0.0);
  }
}

// Reference half-spectrum -> compact rectangle (optionally truncated).
__global__ void gather_k(Phys ph, Rect rc, int kyp, const double2* __restrict__ ref,
                         double2* cmp, int apply_trunc) {
  const int n = ph.n, nh = n / 2 + 1, ky = rc.ky(), kc = rc.kc();
  const size_t tot = (size_t)kc * ky;
  for (size_t e = blockIdx.x * (size_t)blockDim.x + threadIdx.x; e < tot;
       e += (size_t)gridDim.x * blockDim.x) {
    const int c = (int)(e % kc), r = (int)(e / kc);
    const int p = fft_of(r, rc, n);
    double2 v = ref[c + (size_t)nh * p];
    if (apply_trunc) {
      const double fkx = (double)c * ph.dkx, fky = (double)kyi_of(p, n) * ph.dky;
      if (cut_mode(ph, fkx * fkx, fky * fky) || (c == 0 && p == 0))
        v = make_double2(0.0, 0.0);
    }
    cmp[(size_t)c * kyp + r] = v;
  }
}

// Compact rectangle rf -> the smaller rectangle rc (optionally truncated):
// one workgroup row per column, both sides contiguous.
__global__ void narrow_k(Phys ph, Rect rf, int kypf, const double2* __restrict__ src, Rect rc,
                         int kyp, double2* __restrict__ dst, int apply_trunc) {
  const int n = ph.n, ky = rc.ky(), c = blockIdx.y;
  const int r = blockIdx.x * blockDim.x + threadIdx.x;
  if (r >= ky) return;
  const int p = fft_of(r, rc, n);
  double2 v = src[(size_t)c * kypf + row_of(p, rf, n)];
  if (apply_trunc) {
    const double fkx = (double)c * ph.dkx, fky = (double)kyi_of(p, n) * ph.dky;
    if (cut_mode(ph, fkx * fkx, fky * fky) || (c == 0 && p == 0)) v = make_double2(0.0, 0.0);
  }
  dst[(size_t)c * kyp + r] = v;
}

// Flags a nonzero mode of compact rectangle rf outside rc.
__global__ void outside_cmp_k(Phys ph, Rect rf, int kypf, const double2* __restrict__ src,
                              Rect rc, int* flag) {
  const int n = ph.n, c = blockIdx.y;
  const int r = blockIdx.x * blockDim.x + threadIdx.x;
  if (r >= rf.ky() || (c <= rc.kx && row_of(fft_of(r, rf, n), rc, n) >= 0)) return;
  const double2 v = src[(size_t)c * kypf + r];
  if (v.x != 0.0 || v.y != 0.0) atomicOr(flag, 1);
}

// ka = k2**(alpv/2) over the compact rectangle, with kalpha's expressions.  Read
// by the batched passes, by f_pass and fj_pass (N <= 1024, 512) away from alpha
// = 2 and by c_pass for powers other than roots, so that a member and the same
// run alone use the same values.
__global__ void ka_table_k(Phys ph, Rect rc, int kyp, double* ka) {
  const int n = ph.n, ky = rc.ky();
  const size_t tot = (size_t)rc.kc() * ky;
  for (size_t e = blockIdx.x * (size_t)blockDim.x + threadIdx.x; e < tot;
       e += (size_t)gridDim.x * blockDim.x) {
    const int c = (int)(e / ky), r = (int)(e % ky);
    const double fkx = (double)c * ph.dkx;
    const double fkxs = fkx * fkx;
    const double fky = (double)kyi_of(fft_of(r, rc, n), n) * ph.dky;
    ka[(size_t)c * kyp + r] = (c == 0 && r == 0) ? 1.0 : kalpha(ph, fkxs + fky * fky);
  }
}

// Flags a nonzero reference mode outside the rectangle.
__global__ void outside_k(Phys ph, Rect rc, const double2* __restrict__ ref,
                          int* flag) {
  const int n = ph.n, nh = n / 2 + 1;
  const size_t tot = (size_t)nh * n;
  for (size_t e = blockIdx.x * (size_t)blockDim.x + threadIdx.x; e < tot;
       e += (size_t)gridDim.x * blockDim.x) {
    const int i = (int)(e % nh), p = (int)(e / nh);
    if (i > rc.kx || row_of(p, rc, n) < 0) {
      const double2 v = ref[e];
      if (v.x != 0.0 || v.y != 0.0) atomicOr(flag, 1);
    }
  }
}

// Compact rectangle -> reference half-spectrum (zeros outside).
__global__ void scatter_k(Phys ph, Rect rc, int kyp, const double2* __restrict__ cmp,
                          double2* ref) {
  const int n = ph.n, nh = n / 2 + 1;
  const size_t tot = (size_t)nh * n;
  for (size_t e = blockIdx.x * (size_t)blockDim.x + threadIdx.x; e < tot;
       e += (size_t)gridDim.x * blockDim.x) {
    const int i = (int)(e % nh), p = (int)(e / nh);
    const int r = row_of(p, rc, n);
    ref[e] = (i <= rc.kx && r >= 0) ? cmp[(size_t)i * kyp + r]
                                    : make_double2(0.0, 0.0);
  }
}

// The same if ref starts with kIoMark, else nothing: all but the element that the
// mark lies in, which one thread writes after that.  (A block counter in place of
// the second launch took 300 us at 4096^2: 65536 atomics on one address.)
__device__ __forceinline__ bool io_marked(const double2* ref) {
  return *reinterpret_cast<const unsigned long long*>(ref) == kIoMark;
}
__global__ void scatter_marked_k(Phys ph, Rect rc, int kyp, const double2* __restrict__ cmp,
                                 double2* ref) {
  if (!io_marked(ref)) return;
  const int n = ph.n, nh = n / 2 + 1;
  const size_t tot = (size_t)nh * n;
  for (size_t e = blockIdx.x * (size_t)blockDim.x + threadIdx.x; e < tot;
       e += (size_t)gridDim.x * blockDim.x) {
    const int i = (int)(e % nh), p = (int)(e / nh);
    const int r = row_of(p, rc, n);
    if (e > 0)
      ref[e] = (i <= rc.kx && r >= 0) ? cmp[(size_t)i * kyp + r]
                                      : make_double2(0.0, 0.0);
  }
}
__global__ void scatter_mark_k(const double2* __restrict__ cmp, double2* ref) {
  if (io_marked(ref)) ref[0] = cmp[0];  // mode (0, 0) lies in every rectangle
}

// src/forcing.f90:16-33.  One thread per forced mode: no two modes share an
// element, and a mode's own updates (itself, then its Hermitian partner) run
// in the reference's order.  amp = sdt*famp.
// z(i,j) += sdt*famp*(ff1 cos te, ff2 sin te) and the conjugate update of
// the Hermitian partner (src/forcing.f90:25-31).
__device__ __forceinline__ void force_one(const ForcedMode& f, double2 cs, double amp,
                                          double2* z) {
#pragma clang fp contract(off)
  const double a1 = amp * f.ff1 * cs.x, a2 = amp * f.ff2 * cs.y;
  double2 v = z[f.idx];
  v.x = v.x + a1;
  v.y = v.y + a2;
  z[f.idx] = v;
  if (f.pidx >= 0) {
    double2 w = z[f.pidx];
    w.x = w.x + a1;
    w.y = w.y - a2;
    z[f.pidx] = w;
  }
}

__global__ void forcing_k(int nf, const ForcedMode* __restrict__ fm,
                          const double2* __restrict__ ph, double amp,
                          double2* z) {
  const int k = blockIdx.x * blockDim.x + threadIdx.x;
  if (k >= nf) return;
  force_one(fm[k], ph[k], amp, z);
}

// Forcing of every ensemble member in one launch, one thread per forced
// mode; the phases of chunk step *step are used.
__global__ void ens_forcing_k(const EnsForce* __restrict__ f, int nmem, int total,
                              const int* __restrict__ step) {
  const int t = blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= total) return;
  int lo = 0, hi = nmem - 1;  // last member whose first mode is <= t
  while (lo < hi) {
    const int mid = (lo + hi + 1) >> 1;
    if (f[mid].first <= t) lo = mid;
    else hi = mid - 1;
  }
  const EnsForce& e = f[lo];
  const int k = t - e.first;
  if (k >= e.nf) return;
  force_one(e.modes[k], e.phases[(size_t)(*step) * e.nf + k], e.amp, e.z);
}

__global__ void ens_tick_k(int* step) { step[0] = step[0] + 1; }

// ---------------------------------------------------------------------------
// Diagnostics (src/diagnostics.f90), deterministic: the order of every sum is
// fixed, so the results do not change from run to run (the reference's
// accumulations on the GPU are unprotected, diagnostics.f90:25-39,84-101).
//
// Spectrum and fluxes: one workgroup (4 waves) per kx column bins the
// column's modes into LDS bins, one per shell.  In each half of a column
// (ky >= 0: rows 0..p; ky < 0: rows p+1..) the shell index is monotone in the
// row.  Each wave takes a quarter of the half in chunks of 64 rows, whose
// runs of equal shells a segmented wavefront scan sums (a fixed tree); a run
// that a chunk leaves open is carried in registers to the next.  A shell then
// belongs to one wave, except where a wave's first run continues the one
// before: first runs go to a slot per wave, added in wave order after the
// half.  One barrier per half instead of two per chunk, and the next chunk's
// loads are issued before this one is summed.  The column's bins go to
// part[c][b]; a second launch sums part[.][b] over the columns.  4096^2
// spectrum: bins 36 us (54 with a barrier pair per chunk and hypot, 42 with
// the scan through LDS and a double-precision root; 60 MB, bound by the some
// 300 instructions a chunk), columns 10 us (27 with one shell's column of
// part per wavefront).
// ---------------------------------------------------------------------------

__host__ __device__ __forceinline__ int shell_of(const Phys& ph, double fkxs, int p) {
  const double fky = (double)kyi_of(p, ph.n) * ph.dky;
  const double k = sqrt(fkxs + fky * fky);
  return (int)(k / ph.dkx) + 1;  // diagnostics.f90:32-34 (dk = dkx)
}

// Shells a column's kept rows fall in: [lo, hi], hi below NBIN
// (diagnostics.f90:35 bins only ib < NBIN).
__host__ __device__ __forceinline__ void column_shells(const Phys& ph, const Rect& rc, int c,
                                                       int& lo, int& hi) {
  const int n = ph.n;
  const double fkx = (double)c * ph.dkx, fkxs = fkx * fkx;
  lo = shell_of(ph, fkxs, 0);
  hi = shell_of(ph, fkxs, fft_of(rc.p, rc, n));
  if (rc.ky() > rc.p + 1) {
    const int h2 = shell_of(ph, fkxs, fft_of(rc.p + 1, rc, n));
    hi = h2 > hi ? h2 : hi;
  }
  hi = hi < n / 2 - 1 ? hi : n / 2 - 1;
}

constexpr int kDiagT = 256;  // threads of a diagnostics workgroup (4 waves)

// v of another lane of the wave, by a data-parallel move (0 where there is
// none): row_shr d within 16 lanes, the last lane of the row or half before.
template <int CTRL>
__device__ __forceinline__ double lane_dpp(double v) {
  const int lo = __builtin_amdgcn_update_dpp(0, __double2loint(v), CTRL, 0xf, 0xf, true);
  const int hi = __builtin_amdgcn_update_dpp(0, __double2hiint(v), CTRL, 0xf, 0xf, true);
  return __hiloint2double(hi, lo);
}
// Inclusive sums of v1, v2 over each run of equal keys in the wave (runs are
// contiguous, heads the ballot of their first lanes): a scan within the rows
// of 16 lanes, then the rows and halves a run crosses, without LDS traffic.
__device__ __forceinline__ void wave_runs(unsigned long long heads, int lane, double& v1,
                                          double& v2) {
  // lanes of the run before this one, in the wave and in the lane's row
  const int back = lane - (63 - __clzll((long long)(heads & (~0ull >> (63 - lane)))));
  const int rb = back < (lane & 15) ? back : (lane & 15);
  auto add = [&](bool c, double t1, double t2) {
    v1 = c ? v1 + t1 : v1;
    v2 = c ? v2 + t2 : v2;
  };
  add(rb >= 1, lane_dpp<0x111>(v1), lane_dpp<0x111>(v2));
  add(rb >= 2, lane_dpp<0x112>(v1), lane_dpp<0x112>(v2));
  add(rb >= 4, lane_dpp<0x114>(v1), lane_dpp<0x114>(v2));
  add(rb >= 8, lane_dpp<0x118>(v1), lane_dpp<0x118>(v2));
  // lane 15 to row 1, lane 47 to row 3; lane 31 to rows 2 and 3
  add((lane & 16) != 0 && back > (lane & 15), lane_dpp<0x142>(v1), lane_dpp<0x142>(v2));
  add((lane & 32) != 0 && back > (lane & 31), lane_dpp<0x143>(v1), lane_dpp<0x143>(v2));
}

__device__ __forceinline__ double lane_value(double v, int lane) {
  const int lo = __builtin_amdgcn_readlane(__double2loint(v), lane);
  const int hi = __builtin_amdgcn_readlane(__double2hiint(v), lane);
  return __hiloint2double(hi, lo);
}

// |v|^2.  As the square of the modulus (hypot): infinite where a part is, also
// beside a NaN.  The wave looks only if one of its sums is a NaN.
__device__ __forceinline__ double abs2(double2 v) {
  double a = v.x * v.x + v.y * v.y;
  if (__builtin_expect(__ballot(a != a) != 0, 0)) {
    if (isinf(v.x) || isinf(v.y)) a = __builtin_huge_val();
  }
  return a;
}

// int(sqrt(k2)) of a whole number up to 2^25: the single-precision root, off
// by at most one, put right.
__device__ __forceinline__ int isqrt_of(double k2) {
  const int m = (int)k2;
  int q = (int)__builtin_amdgcn_sqrtf((float)m);
  q += (q + 1) * (q + 1) <= m ? 1 : 0;
  return q * q > m ? q - 1 : q;
}

// WHICH = 0: spectrum (sp, sz);  WHICH = 1: fluxes (flzm, flem)
// nbl: the most shells of any column (LDS bins per sum).
template <int WHICH>
__global__ void __launch_bounds__(kDiagT) shell_bin_k(DiagArgs d, int nbl) {
  extern __shared__ double dsm[];
  constexpr int NW = kDiagT / 64;
  const Phys& ph = d.ph;
  const Rect rc = d.rc;
  const int n = ph.n, nbin = n / 2, c = blockIdx.x, tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  double* bin1 = dsm;         // shell b of the column in bin b - lo
  double* bin2 = bin1 + nbl;
  __shared__ double edge1[NW], edge2[NW];  // each wave's first run
  __shared__ int ekey[NW];
  const double fkx = (double)c * ph.dkx, fkxs = fkx * fkx;
  const double fac = (c == 0 || c == n / 2) ? (WHICH ? 1.0 : 0.5)   // diagnostics.f90:29-30
                                            : (WHICH ? 2.0 : 1.0);  // :89-90
  const size_t cq = (size_t)c * d.kyp;
  const bool unit = ph.dkx == 1.0 && ph.dky == 1.0;  // k2 a whole number
  int blo, bhi;
  column_shells(ph, rc, c, blo, bhi);
  if (bhi - blo + 1 > nbl) bhi = blo + nbl - 1;  // never: nbl is the maximum
  for (int b = blo + tid; b <= bhi; b += kDiagT) {
    bin1[b - blo] = 0.0;
    bin2[b - blo] = 0.0;
  }
  const int P = rc.p, Ky = rc.ky();
  for (int half = 0; half < 2; ++half) {
    const int h0 = half ? P + 1 : 0, h1 = half ? Ky : P + 1;  // rows [h0, h1)
    const int per = ((h1 - h0 + NW - 1) / NW + 63) & ~63;
    const int r0 = h0 + wave * per, r1 = r0 + per < h1 ? r0 + per : h1;
    __syncthreads();  // bins cleared; the half before added up
    if (lane == 0) ekey[wave] = -1;
    const double2 zero = make_double2(0.0, 0.0);
    double2 zn = r0 + lane < r1 ? d.z[cq + r0 + lane] : zero;
    double2 nn = WHICH && r0 + lane < r1 ? d.znl[cq + r0 + lane] : zero;
    int first = -2, ck = -1;       // the wave's first key; the carried run
    double c1 = 0.0, c2 = 0.0;
    // adds a finished run: the wave's first one to its slot
    auto put = [&](int key, double v1, double v2) {
      if (key == first) {
        ekey[wave] = key;
        edge1[wave] = v1;
        edge2[wave] = v2;
      } else {
        bin1[key - blo] = bin1[key - blo] + v1;
        bin2[key - blo] = bin2[key - blo] + v2;
      }
    };
    for (int base = r0; base < r1; base += 64) {
      const int r = base + lane, rn = r + 64;
      const double2 zv = zn, nv = nn;
      zn = rn < r1 ? d.z[cq + rn] : zero;
      if (WHICH) nn = rn < r1 ? d.znl[cq + rn] : zero;
      int key = -1;
      double v1 = 0.0, v2 = 0.0;
      if (r < r1 && !(c == 0 && r == 0)) {  // diagnostics.f90:28
        const int p = fft_of(r, rc, n);
        const double fky = (double)kyi_of(p, n) * ph.dky;
        const double k2 = fkxs + fky * fky;
        const int ib = unit ? isqrt_of(k2) + 1 : (int)(sqrt(k2) / ph.dkx) + 1;  // :34
        if (ib < nbin && ib >= blo && ib <= bhi) {
          key = ib;
          const double ka = kalpha(ph, k2);
          if (WHICH == 0) {
            const double a2 = abs2(zv);
            v1 = fac * a2 / ka;  // sp, diagnostics.f90:36
            v2 = fac * a2;       // sz, :37
          } else {
            const double fz = zv.x * nv.x + zv.y * nv.y;  // :93
            v1 = fac * fz;          // flzm, :98
            v2 = fac * (fz / ka);   // flem, :95,99
          }
        }
      }
      const int kprev = __shfl_up(key, 1);
      const bool head = lane == 0 || kprev != key;
      const unsigned long long heads = __ballot(head);
      wave_runs(heads, lane, v1, v2);
      const int k0 = __builtin_amdgcn_readfirstlane(key);
      if (base == r0) first = k0;
      if (ck == k0 && ck >= 0) {  // the carried run goes on in this chunk's first
        if ((heads & (~0ull >> (63 - lane))) == 1ull) {
          v1 = c1 + v1;
          v2 = c2 + v2;
        }
      } else if (ck >= 0 && lane == 0) {
        put(ck, c1, c2);
      }
      // runs that end inside the chunk (one lane each)
      if (lane < 63 && ((heads >> (lane + 1)) & 1ull) != 0 && key >= 0) put(key, v1, v2);
      ck = __builtin_amdgcn_readlane(key, 63);
      c1 = lane_value(v1, 63);
      c2 = lane_value(v2, 63);
    }
    if (ck >= 0 && lane == 0) put(ck, c1, c2);
    __syncthreads();
    if (tid == 0) {
      for (int w = 0; w < NW; ++w) {
        const int key = ekey[w];
        if (key >= 0) {
          bin1[key - blo] = bin1[key - blo] + edge1[w];
          bin2[key - blo] = bin2[key - blo] + edge2[w];
        }
      }
    }
  }
  __syncthreads();
  for (int b = blo + tid; b <= bhi; b += kDiagT) {
    d.part1[(size_t)c * nbin + (b - 1)] = bin1[b - blo];
    d.part2[(size_t)c * nbin + (b - 1)] = bin2[b - blo];
  }
  if (tid == 0) d.lohi[c] = make_int2(blo, bhi);
}

// Sum of a wavefront's values in a fixed tree order; lane 0 holds the total.
__device__ __forceinline__ double wave_sum(double v) {
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) v = v + __shfl_down(v, off);
  return v;
}

// The columns' bins summed over the columns: a workgroup takes 16 shells,
// its 64 rows of 16 threads the columns c = g, g + 64, ... in order (128
// contiguous bytes of part each), then a fixed tree over the rows.
constexpr int kSumT = 1024, kSumB = 16, kSumG = kSumT / kSumB;
__global__ void __launch_bounds__(kSumT) shell_sum_k(DiagArgs d, int which) {
  __shared__ double s1[kSumG][kSumB + 1], s2[kSumG][kSumB + 1];
  __shared__ int2 lh[8192 / 2 + 1];
  const Phys& ph = d.ph;
  const int nbin = ph.n / 2, kx = d.rc.kx;
  const int o = threadIdx.x % kSumB, g = threadIdx.x / kSumB;
  const int b = blockIdx.x * kSumB + o + 1;  // shell 1..NBIN
  for (int c = threadIdx.x; c <= kx; c += kSumT) lh[c] = d.lohi[c];
  __syncthreads();
  double a1 = 0.0, a2 = 0.0;
  for (int c0 = g; c0 <= kx; c0 += 8 * kSumG) {
    double t1[8], t2[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) {  // all in flight together
      const int c = c0 + i * kSumG;
      const bool in = c <= kx && b <= nbin && b >= lh[c].x && b <= lh[c].y;
      t1[i] = in ? d.part1[(size_t)c * nbin + (b - 1)] : 0.0;
      t2[i] = in ? d.part2[(size_t)c * nbin + (b - 1)] : 0.0;
    }
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      a1 = a1 + t1[i];
      a2 = a2 + t2[i];
    }
  }
  s1[g][o] = a1;
  s2[g][o] = a2;
  __syncthreads();
#pragma unroll
  for (int h = kSumG / 2; h > 0; h >>= 1) {
    if (g < h) {
      s1[g][o] = s1[g][o] + s1[g + h][o];
      s2[g][o] = s2[g][o] + s2[g + h][o];
    }
    __syncthreads();
  }
  if (g != 0 || b > nbin) return;
  if (which == 0) {  // diagnostics.f90:42-45
    d.out1[b - 1] = s1[0][o] / ph.dkx;
    d.out2[b - 1] = s2[0][o] / ph.dkx;
  } else {
    d.part1[(size_t)(kx + 1) * nbin + (b - 1)] = s1[0][o];  // flzm
    d.part2[(size_t)(kx + 1) * nbin + (b - 1)] = s2[0][o];  // flem
  }
}

// flz(i) = sum(flzm(i:NBIN)) and fle likewise (diagnostics.f90:104-109): a
// scan from the last shell down in one workgroup, four shells a thread, a
// fixed order (4.6 us at 4096^2; 36 with each thread adding its own suffix).
// NBIN <= 4096.
__global__ void __launch_bounds__(1024) suffix_k(DiagArgs d) {
  __shared__ double w1[16], w2[16];
  const int nbin = d.ph.n / 2, t = threadIdx.x, lane = t & 63, wave = t >> 6;
  const double* flzm = d.part1 + (size_t)(d.rc.kx + 1) * nbin;
  const double* flem = d.part2 + (size_t)(d.rc.kx + 1) * nbin;
  // thread t: the reversed positions 4t .. 4t+3, i.e. shells nbin-1-4t down
  double z[4], e[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int q = nbin - 1 - (4 * t + i);
    z[i] = q >= 0 ? flzm[q] : 0.0;
    e[i] = q >= 0 ? flem[q] : 0.0;
  }
#pragma unroll
  for (int i = 1; i < 4; ++i) {
    z[i] = z[i] + z[i - 1];
    e[i] = e[i] + e[i - 1];
  }
  double tz = z[3], te = e[3];  // inclusive scan of the threads' totals
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const double uz = __shfl_up(tz, o), ue = __shfl_up(te, o);
    if (lane >= o) {
      tz = tz + uz;
      te = te + ue;
    }
  }
  if (lane == 63) {
    w1[wave] = tz;
    w2[wave] = te;
  }
  __syncthreads();
  double bz = __shfl_up(tz, 1), be = __shfl_up(te, 1);
  if (lane == 0) bz = be = 0.0;
  double pz = 0.0, pe = 0.0;  // the waves before, in order
  for (int w = 0; w < wave; ++w) {
    pz = pz + w1[w];
    pe = pe + w2[w];
  }
  bz = pz + bz;
  be = pe + be;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int q = nbin - 1 - (4 * t + i);
    if (q >= 0) {
      d.out1[q] = be + e[i];  // fle
      d.out2[q] = bz + z[i];  // flz
    }
  }
}

// k2**a for the dissipation exponents of glob: repeated products for the
// small whole exponents the runs use (k^8 hyperviscosity is a = 4, linear
// drag a = 0), pow otherwise.
__device__ __forceinline__ double pow_k2(double k2, double a) {
  if (a == 0.0) return 1.0;
  if (a == 1.0) return k2;
  if (a == 2.0) return k2 * k2;
  if (a == 3.0) return (k2 * k2) * k2;
  if (a == 4.0) {
    const double t = k2 * k2;
    return t * t;
  }
  return pow(k2, a);
}

// src/diagnostics.f90:147-163: one workgroup per column; each thread sums
// its rows in order (four loads ahead), then a fixed wavefront tree and the
// four waves in order.  dise_* use k2**alpnu / ka for k2**(alpnu - alpv/2).
__global__ void __launch_bounds__(kDiagT) glob_col_k(DiagArgs d) {
  const Phys& ph = d.ph;
  const Rect rc = d.rc;
  const int n = ph.n, c = blockIdx.x, Ky = rc.ky();
  const double fkx = (double)c * ph.dkx, fkxs = fkx * fkx;
  const double fac = (c == 0 || c == n / 2) ? 0.5 : 1.0;
  const double2* z = d.z + (size_t)c * d.zcs;
  double acc[6] = {0, 0, 0, 0, 0, 0};
  for (int rb = threadIdx.x; rb < Ky; rb += 4 * kDiagT) {
    double2 zv[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int r = rb + i * kDiagT;
      zv[i] = r < Ky ? z[(size_t)r * d.zrs] : make_double2(0.0, 0.0);
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int r = rb + i * kDiagT;
      if (r >= Ky || (c == 0 && r == 0)) continue;
      const int p = fft_of(r, rc, n);
      const double fky = (double)kyi_of(p, n) * ph.dky;
      const double k2 = fkxs + fky * fky;
      const double ka = kalpha(ph, k2);
      const double a2 = fac * abs2(zv[i]), ae = a2 / ka;
      const double gnu = 2.0 * ph.nu * pow_k2(k2, ph.alpnu);
      const double gmu = 2.0 * ph.mu * pow_k2(k2, ph.alpmu);
      acc[0] = acc[0] + ae;        // ee
      acc[1] = acc[1] + a2;        // zz
      acc[2] = acc[2] + gnu * a2;  // disz_nu
      acc[3] = acc[3] + gmu * a2;  // disz_mu
      acc[4] = acc[4] + gnu * ae;  // dise_nu
      acc[5] = acc[5] + gmu * ae;  // dise_mu
    }
  }
  __shared__ double red[6][kDiagT / 64];
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
#pragma unroll
  for (int q = 0; q < 6; ++q) {
    const double v = wave_sum(acc[q]);
    if (lane == 0) red[q][wave] = v;
  }
  __syncthreads();
  if (threadIdx.x < 6) {
    const int q = threadIdx.x;
    double v = red[q][0];
    for (int w = 1; w < kDiagT / 64; ++w) v = v + red[q][w];
    d.gpart[(size_t)q * rc.kc() + c] = v;
  }
}

// Two wavefronts per quantity, over the columns in a fixed order.
__global__ void __launch_bounds__(12 * 64) glob_sum_k(DiagArgs d) {
  __shared__ double red[12];
  const int q = threadIdx.x / 128, t = threadIdx.x % 128, kc = d.rc.kc();
  const double* g = d.gpart + (size_t)q * kc;
  double s = 0.0;
  for (int c0 = t; c0 < kc; c0 += 8 * 128) {
    double v[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) v[i] = c0 + 128 * i < kc ? g[c0 + 128 * i] : 0.0;
#pragma unroll
    for (int i = 0; i < 8; ++i) s = s + v[i];
  }
  s = wave_sum(s);
  if (t % 64 == 0) red[threadIdx.x / 64] = s;
  __syncthreads();
  if (t == 0) d.gout[q] = red[2 * q] + red[2 * q + 1];
}

__global__ void shell_index_k(Phys ph, int* ib) {
  const int n = ph.n, nh = n / 2 + 1;
  const size_t tot = (size_t)nh * n;
  for (size_t e = blockIdx.x * (size_t)blockDim.x + threadIdx.x; e < tot;
       e += (size_t)gridDim.x * blockDim.x) {
    const int i = (int)(e % nh), p = (int)(e / nh);
    const double fkx = (double)i * ph.dkx;
    ib[e] = (e == 0) ? 0 : shell_of(ph, fkx * fkx, p);
  }
}

static inline unsigned grid_for(size_t tot, int block) {
  size_t g = (tot + block - 1) / block;
  return (unsigned)(g > 65536 ? 65536 : (g == 0 ? 1 : g));
}

#define GT_LOGN_CASE(V, ...) \
  case V: {                     \
    constexpr int L = V;        \
    __VA_ARGS__;                \
  } break;
#define GT_LOGN_SWITCH(LOGN_VAR, ...)                                     \
  switch (LOGN_VAR) {                                                     \
    GT_LOGN_CASE(4, __VA_ARGS__) GT_LOGN_CASE(5, __VA_ARGS__)             \
    GT_LOGN_CASE(6, __VA_ARGS__) GT_LOGN_CASE(7, __VA_ARGS__)             \
    GT_LOGN_CASE(8, __VA_ARGS__) GT_LOGN_CASE(9, __VA_ARGS__)             \
    GT_LOGN_CASE(10, __VA_ARGS__) GT_LOGN_CASE(11, __VA_ARGS__)           \
    GT_LOGN_CASE(12, __VA_ARGS__) GT_LOGN_CASE(13, __VA_ARGS__)           \
    default: return hipErrorInvalidValue;                                 \
  }

hipError_t launch_c_pass(int logn, int mode, const PassArgs& a, hipStream_t s) {
  GT_LOGN_SWITCH(logn, return c_pass_launch<L>(mode, a, s));
  return hipSuccess;
}

hipError_t launch_r_pass(int logn, const PassArgs& a, hipStream_t s) {
  GT_LOGN_SWITCH(logn, return r_pass_launch<L>(a, s));
  return hipSuccess;
}

hipError_t launch_j_pass(int logn, int mode, const AdjArgs& a, hipStream_t s) {
  GT_LOGN_SWITCH(logn, return j_pass_launch<L>(mode, a, s));
  return hipSuccess;
}

hipError_t launch_jr_pass(int logn, const AdjArgs& a, hipStream_t s) {
  GT_LOGN_SWITCH(logn, return jr_pass_launch<L>(a, s));
  return hipSuccess;
}

hipError_t launch_io(int logn, const IoArgs& a, hipStream_t s) {
  GT_LOGN_SWITCH(logn, return io_launch<L>(a, s));
  return hipSuccess;
}

hipError_t launch_produ(int n, const double* z, double* u, double* v,
                        hipStream_t s) {
  produ_k<<<grid_for(((size_t)n + 2) * n, 256), 256, 0, s>>>(n, z, u, v);
  return hipGetLastError();
}

hipError_t launch_trunc_cmp(const Phys& ph, const Rect& rc, int kyp, double2* z,
                            hipStream_t s) {
  trunc_cmp_k<<<grid_for((size_t)rc.kc() * rc.ky(), 256), 256, 0, s>>>(ph, rc, kyp, z);
  return hipGetLastError();
}

hipError_t launch_gather(const Phys& ph, const Rect& rc, int kyp, const double* ref,
                         double2* cmp, int apply_trunc, int* outside_flag,
                         hipStream_t s) {
  const double2* rc2 = reinterpret_cast<const double2*>(ref);
  gather_k<<<grid_for((size_t)rc.kc() * rc.ky(), 256), 256, 0, s>>>(
      ph, rc, kyp, rc2, cmp, apply_trunc);
  if (outside_flag)
    outside_k<<<grid_for((size_t)(ph.n / 2 + 1) * ph.n, 256), 256, 0, s>>>(
        ph, rc, rc2, outside_flag);
  return hipGetLastError();
}

hipError_t launch_narrow(const Phys& ph, const Rect& rf, int kypf, const double2* src,
                         const Rect& rc, int kyp, double2* dst, int apply_trunc,
                         int* outside_flag, hipStream_t s) {
  if (outside_flag)
    outside_cmp_k<<<dim3((rf.ky() + 255) / 256, rf.kc()), 256, 0, s>>>(ph, rf, kypf, src, rc,
                                                                      outside_flag);
  narrow_k<<<dim3((rc.ky() + 255) / 256, rc.kc()), 256, 0, s>>>(ph, rf, kypf, src, rc, kyp, dst,
                                                               apply_trunc);
  return hipGetLastError();
}

hipError_t launch_scatter(const Phys& ph, const Rect& rc, int kyp, const double2* cmp,
                          double* ref, hipStream_t s) {
  scatter_k<<<grid_for((size_t)(ph.n / 2 + 1) * ph.n, 256), 256, 0, s>>>(
      ph, rc, kyp, cmp, reinterpret_cast<double2*>(ref));
  return hipGetLastError();
}

hipError_t launch_scatter_marked(const Phys& ph, const Rect& rc, int kyp, const double2* cmp,
                                 double* ref, hipStream_t s) {
  double2* r = reinterpret_cast<double2*>(ref);
  scatter_marked_k<<<grid_for((size_t)(ph.n / 2 + 1) * ph.n, 256), 256, 0, s>>>(ph, rc, kyp, cmp,
                                                                               r);
  scatter_mark_k<<<1, 1, 0, s>>>(cmp, r);
  return hipGetLastError();
}

hipError_t launch_forcing(const Phys& ph, int nf, const ForcedMode* modes,
                          const double2* phases, double amp, double2* z,
                          hipStream_t s) {
  (void)ph;
  if (nf <= 0) return hipSuccess;
  forcing_k<<<(nf + 255) / 256, 256, 0, s>>>(nf, modes, phases, amp, z);
  return hipGetLastError();
}

hipError_t launch_ens_c_pass(int ty, int sched, int mode, const PassArgs* descs,
                             const uint32_t* items, int nitems, int grid,
                             hipStream_t s) {
  if (nitems <= 0) return hipSuccess;
  if (ty == 256) return sched ? ens_c_launch<256, 1>(mode, descs, items, nitems, grid, s)
                              : ens_c_launch<256, 0>(mode, descs, items, nitems, grid, s);
  if (ty == 512) return sched ? ens_c_launch<512, 1>(mode, descs, items, nitems, grid, s)
                              : ens_c_launch<512, 0>(mode, descs, items, nitems, grid, s);
  return hipErrorInvalidValue;
}

hipError_t launch_ens_r_pass(int tx, int ty, int sched, const PassArgs* descs,
                             const uint32_t* items, int nitems, int grid,
                             hipStream_t s) {
  if (nitems <= 0) return hipSuccess;
  if (tx == 256) return sched ? ens_r_launch<256, 1>(ty, descs, items, nitems, grid, s)
                              : ens_r_launch<256, 0>(ty, descs, items, nitems, grid, s);
  if (tx == 512) return sched ? ens_r_launch<512, 1>(ty, descs, items, nitems, grid, s)
                              : ens_r_launch<512, 0>(ty, descs, items, nitems, grid, s);
  return hipErrorInvalidValue;
}

hipError_t launch_ka_table(const Phys& ph, const Rect& rc, int kyp, double* ka,
                           hipStream_t s) {
  const size_t tot = (size_t)rc.kc() * rc.ky();
  ka_table_k<<<grid_for(tot, 256), 256, 0, s>>>(ph, rc, kyp, ka);
  return hipGetLastError();
}

hipError_t launch_ens_forcing(const EnsForce* f, int nmem, int total,
                              const int* step, hipStream_t s) {
  if (total <= 0) return hipSuccess;
  ens_forcing_k<<<(total + 255) / 256, 256, 0, s>>>(f, nmem, total, step);
  return hipGetLastError();
}

hipError_t launch_ens_tick(int* step, hipStream_t s) {
  ens_tick_k<<<1, 1, 0, s>>>(step);
  return hipGetLastError();
}

hipError_t launch_spectrum(const DiagArgs& d, int which, hipStream_t s) {
  const int nbin = d.ph.n / 2;
  int nbl = 1;  // the most shells of one column
  for (int c = 0; c <= d.rc.kx; ++c) {
    int lo, hi;
    column_shells(d.ph, d.rc, c, lo, hi);
    nbl = hi - lo + 1 > nbl ? hi - lo + 1 : nbl;
  }
  // LDS: two sums per shell of a column; 44 KB at N = 8192, 65,520 bytes (with
  // the static part above the 64 KB a launch gets by itself) untruncated
  const size_t lds = 2 * sizeof(double) * (size_t)nbl;
  if (lds > 60 * 1024) {
    const hipError_t e = hipFuncSetAttribute(
        which == 0 ? reinterpret_cast<const void*>(&shell_bin_k<0>)
                   : reinterpret_cast<const void*>(&shell_bin_k<1>),
        hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    if (e != hipSuccess) return e;
  }
  if (which == 0) shell_bin_k<0><<<d.rc.kc(), kDiagT, lds, s>>>(d, nbl);
  else shell_bin_k<1><<<d.rc.kc(), kDiagT, lds, s>>>(d, nbl);
  shell_sum_k<<<(nbin + kSumB - 1) / kSumB, kSumT, 0, s>>>(d, which);
  if (which == 1) suffix_k<<<1, 1024, 0, s>>>(d);
  return hipGetLastError();
}

hipError_t launch_glob(const DiagArgs& d, hipStream_t s) {
  glob_col_k<<<d.rc.kc(), kDiagT, 0, s>>>(d);
  glob_sum_k<<<1, 12 * 64, 0, s>>>(d);
  return hipGetLastError();
}

// Partial sums of the allocation-free glob: six per kx column (at most
// N/2 + 1 = 4097 columns, N <= 8192) and the six totals, 196,704 bytes per
// GPU for the life of the process.  Host code never uses the array's name
// as an address: glob_scratch resolves the device address once per device.
constexpr size_t kGlobScratch = 6 * (8192 / 2 + 1) + 6;
static __device__ __align__(256) double scratch[kGlobScratch];

hipError_t glob_scratch(double** ptr, size_t* count) {
  constexpr int kMaxDev = 64;
  static std::mutex mu;
  static double* addr[kMaxDev] = {};
  int dev = 0;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess) return e;
  if (dev < 0 || dev >= kMaxDev) return hipErrorInvalidDevice;
  std::lock_guard<std::mutex> lock(mu);
  if (addr[dev] == nullptr) {
    void* a = nullptr;
    e = hipGetSymbolAddress(&a, HIP_SYMBOL(scratch));
    if (e != hipSuccess) return e;
    addr[dev] = static_cast<double*>(a);
  }
  *ptr = addr[dev];
  *count = kGlobScratch;
  return hipSuccess;
}

hipError_t launch_shell_index(const Phys& ph, int* ib, hipStream_t s) {
  shell_index_k<<<grid_for((size_t)(ph.n / 2 + 1) * ph.n, 256), 256, 0, s>>>(ph, ib);
  return hipGetLastError();
}

#endif  // GT_INST_COMMON

}  // namespace gt
