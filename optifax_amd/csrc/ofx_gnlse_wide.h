// The fibre GNLSE solver for long grids: the integration of ofx_gnlse_impl.h
// (same equation, step control, sums per point and outputs) with 8 points of
// the field in each thread's registers.
//
// Thread t of n / 8 owns the points t + m n/8, m < 8, of every vector, so
//   * a transform runs as radix-8 steps (a radix-4 and a radix-2 pass) in
//     registers and meets LDS between them only: 4 exchanges for 2^13 points
//     instead of 6 (3 instead of 5 for 2^12), and LDS, whose bandwidth bounds
//     the passes, moves less;
//   * its input and output are the owner's points, so the stage combination
//     y + h sum_j b_j f_j feeds the first step directly (read: the stages that
//     weigh something; written: nothing but ynew), AT waits in registers for
//     the last product, and the phases exp(i B z) are formed once for both
//     ends of an evaluation;
//   * norms are summed where their terms pass through registers.
// The Raman convolution's half-length transforms run on half of the threads.
//
// Bound: vector instruction issue (65 % of the time at 2^13 points, 16 waves of
// about 2500 instructions an evaluation) with ~30 workgroup barriers between.
// us per evaluation with the Raman term against the general kernel, one fibre /
// 96 at once: FP32 2^13 31 / 38 (46 / 58), FP64 2^12 25 / 32 (34 / 42), FP64 2^11
// 17 / 18 (20 / 21).  With 16 points a thread (radix-16 steps, half the waves)
// the same took 33 / 45 at 2^13 and 32 / 43 at FP64 2^12: too few waves.
#pragma once
#include "ofx_gnlse_impl.h"

namespace ofx {

// points of a thread
#define GW_P 8

// Where this kernel runs: FP64 fields from 2^11 points (at 2^10 it measured
// 0.97-1.04 of the general kernel's speed) and FP32 fields at 2^13.  On shorter
// FP32 grids it is faster too (2^12: 1.6 times) and as accurate, but its passes
// round in another order, and soliton fission makes more of that on the coarser
// grids than a change of kernel is meant to move.  Error against FP64, general /
// this kernel, and their difference (2 cm, Raman and shock, 5, 7.5 and 10 kW, rtol
// 1e-6): 2^11 1.2e-5 / 9.6e-6, 1.5e-4 / 1.1e-4, 5.4e-4 / 4.3e-4 and 3.1e-6, 4.6e-5,
// 2.4e-4; 2^12 2.7e-6 / 3.7e-6, 8.2e-6 / 1.2e-5, 3.9e-5 / 1.3e-5 and 3.1e-6, 1.8e-5,
// 4.7e-5.
OFX_HD constexpr bool gw_runs(int lg, bool f64) { return f64 ? lg == 11 || lg == 12 : lg == 13; }

// LDS index of element i: one unused element after each 16
OFX_HD constexpr int gw_pad(int i) { return i + (i >> 4); }

// Twiddle tables (LDS) of 2^lg points: for the radix-8 steps of stride NS =
// 1, 8, 64, ... <= n / 8 the radix-4 pass's exp(-2 pi i k / (4 NS)), k < NS (none
// for NS = 1), and the radix-2 pass's exp(-2 pi i k / (8 NS)), k < 4 NS; then the
// quarter table exp(-2 pi i m / n), m < n / 4 (last passes of radix 4 and 2, and
// the Raman convolution).
OFX_HD constexpr int gw_r4_at(int ns) { return 5 * (ns - 1) / 7 - 1; }   // ns > 1
OFX_HD constexpr int gw_r2_at(int ns) { return ns > 1 ? gw_r4_at(ns) + ns : 0; }
OFX_HD constexpr int gw_top(int lg) { return 1 << (3 * ((lg - 3) / 3)); }  // largest NS
OFX_HD constexpr int gw_qt_at(int lg) { return gw_r2_at(gw_top(lg)) + 4 * gw_top(lg); }
OFX_HD constexpr int gw_table_size(int lg) { return gw_qt_at(lg) + (1 << lg) / 4; }

template <typename R>
std::vector<cpx<R>> gw_twiddles(int lg) {
  std::vector<cpx<R>> t((size_t)gw_table_size(lg));
  auto put = [&](int at, double k, double of) {
    const double ph = -2.0 * M_PI * k / of;
    t[(size_t)at].x = (R)cos(ph);
    t[(size_t)at].y = (R)sin(ph);
  };
  for (int ns = 1; ns <= gw_top(lg); ns <<= 3) {
    for (int k = 0; k < ns && ns > 1; k++) put(gw_r4_at(ns) + k, k, 4.0 * ns);
    for (int k = 0; k < 4 * ns; k++) put(gw_r2_at(ns) + k, k, 8.0 * ns);
  }
  for (int m = 0; m < (1 << lg) / 4; m++) put(gw_qt_at(lg) + m, m, (double)(1 << lg));
  return t;
}

// Ends a group of 4 points of an unrolled loop for the scheduler: with all the
// points' temporaries in flight at once the kernel spills more (as it is FP32 2^13
// keeps 320 and FP64 2^12 316 bytes of scratch a lane, FP64 2^11 none)
OFX_DEV void gw_group(int i) {
#ifndef OFX_EMU
  if ((i & 3) == 3) __builtin_amdgcn_sched_barrier(0);
#endif
}

template <typename R>
struct GwThread {
  cpx<R> v[GW_P];   // transform elements t + m L/8
  cpx<R> at[GW_P];  // AT at the owner's points
  cpx<R> ph[GW_P];  // exp(i B z) at the owner's points
};

// exp(i x) for an FP64 argument: quadrant reduction with a two-part pi / 2
// (Cody & Waite), Taylor polynomials to r^9 and r^10 in FP32 (expi's, with a
// cheaper quadrant) and to r^17 and r^16 in FP64
OFX_DEV cpx<float> gw_expi(double x, float) {
#ifdef OFX_EMU
  return expi(x, 0.0f);
#else
  const double PIO2_HI = 1.5707963267948966, PIO2_LO = 6.123233995736766e-17;
  // q = rint(2 x / pi) and q mod 4 from the sum with 1.5 2^52, whose low
  // mantissa bits are q
  const double MAGIC = 6755399441055744.0;
  const double qm = x * 0.63661977236758134 + MAGIC;
  const double q = qm - MAGIC;
  const unsigned k = (unsigned)__builtin_bit_cast(u64, qm);
  const float r = (float)fma(-q, PIO2_LO, fma(-q, PIO2_HI, x));
  const float r2 = r * r;
  const float s =
      r * fmaf(r2, fmaf(r2, fmaf(r2, fmaf(r2, 1.0f / 362880.0f, -1.0f / 5040.0f), 1.0f / 120.0f),
                        -1.0f / 6.0f),
               1.0f);
  const float c = fmaf(
      r2,
      fmaf(r2, fmaf(r2, fmaf(r2, fmaf(r2, -1.0f / 3628800.0f, 1.0f / 40320.0f), -1.0f / 720.0f),
                    1.0f / 24.0f),
           -0.5f),
      1.0f);
  const float a = (k & 1) ? s : c, b = (k & 1) ? c : s;
  const unsigned sa = ((k + 1) & 2) << 30, sb = (k & 2) << 30;
  return mkc<float>(__builtin_bit_cast(float, __builtin_bit_cast(unsigned, a) ^ sa),
                    __builtin_bit_cast(float, __builtin_bit_cast(unsigned, b) ^ sb));
#endif
}
OFX_DEV cpx<double> gw_expi(double x, double) {
#ifdef OFX_EMU
  return expi(x, 0.0);
#else
  const double PIO2_HI = 1.5707963267948966, PIO2_LO = 6.123233995736766e-17;
  const double q = rint(x * 0.63661977236758134);
  const double r = fma(-q, PIO2_LO, fma(-q, PIO2_HI, x)), z = r * r;
  double p = 1.0 / 355687428096000.0;
  p = fma(p, z, -1.0 / 1307674368000.0);
  p = fma(p, z, 1.0 / 6227020800.0);
  p = fma(p, z, -1.0 / 39916800.0);
  p = fma(p, z, 1.0 / 362880.0);
  p = fma(p, z, -1.0 / 5040.0);
  p = fma(p, z, 1.0 / 120.0);
  p = fma(p, z, -1.0 / 6.0);
  const double sr = fma(p * z, r, r);
  double u = 1.0 / 20922789888000.0;
  u = fma(u, z, -1.0 / 87178291200.0);
  u = fma(u, z, 1.0 / 479001600.0);
  u = fma(u, z, -1.0 / 3628800.0);
  u = fma(u, z, 1.0 / 40320.0);
  u = fma(u, z, -1.0 / 720.0);
  u = fma(u, z, 1.0 / 24.0);
  u = fma(u, z, -0.5);
  const double cr = fma(u, z, 1.0);
  const int k = (int)fma(-4.0, floor(0.25 * q), q);   // q mod 4
  const double a = (k & 1) ? cr : sr, b = (k & 1) ? sr : cr;
  return mkc<double>((k == 1 || k == 2) ? -b : b, (k & 2) ? -a : a);
#endif
}

template <typename R, int LG>
struct GwRun {
  typedef cpx<R> C;
  typedef GwThread<R> T;
  static constexpr int N = 1 << LG, NT = N / GW_P, H = N / 2, NH = NT / 2;
  T* thr;
  C* buf;          // gw_pad(N) elements
  const C* tw;     // the steps' twiddles (LDS)
  const C* qt;     // quarter table exp(-2 pi i m / N) (LDS)
  double* red;
  const OFX_GLOBAL double* B;
  const OFX_GLOBAL R* W;
  const OFX_GLOBAL C* RW;
  double lre, gamma, fr, dT;
  C *ws, *f0, *f6;  // stage vectors: f1..f5 = ws + j N; f0 and f6 swap after a step

  OFX_DEV C* stage(int j) const { return j == 0 ? f0 : (j == 6 ? f6 : ws + (size_t)j * N); }

  int tid;         // the thread's index, its origin hidden (refresh)

  // Hides where the index comes from, so that addresses are formed where they
  // are used instead of being kept in registers throughout (kept, more spills)
  OFX_DEV void refresh() {
#ifndef OFX_EMU
    asm volatile("" : "+v"(tid));
#endif
  }
  template <typename F>
  OFX_DEV void each(F f) {
#ifdef OFX_EMU
    for (int t = 0; t < NT; t++) f(t, thr[t]);
#else
    f(tid, *thr);
#endif
  }

  static OFX_DEV void bfly2(C& a, C& b) {
    const C x = a, y = b;
    a = cadd(x, y);
    b = csub(x, y);
  }
  template <int SIGN>
  static OFX_DEV C turn(C v, C w) {
    return SIGN > 0 ? cmulc(v, w) : cmul(v, w);
  }

  // The passes from stride NS on (radix 8, or what is left of L) on v;
  // afterwards v[i] is element 8 (t - k) + k + NS i of the next step (k = t mod
  // NS), or element t + i L/8 of the result.
  template <int SIGN, int LGL, int NS>
  OFX_DEV void step(int t, C* v) {
    constexpr int L = 1 << LGL, TL = L / GW_P, LEFT = L / NS;
    const C one = mkc<R>(R(1), R(0));
    if constexpr (LEFT >= 8) {
      const int k = t & (NS - 1);
      const C w = NS > 1 ? tw[gw_r4_at(NS) + k] : one;
#pragma unroll
      for (int u = 0; u < 2; u++) bfly4<R, SIGN, (NS > 1)>(v[u], v[u + 2], v[u + 4], v[u + 6], w);
#pragma unroll
      for (int m = 0; m < 4; m++) {
        if (NS > 1 || m > 0)
          v[2 * m + 1] = turn<SIGN>(v[2 * m + 1], tw[gw_r2_at(NS) + k + NS * m]);
        bfly2(v[2 * m], v[2 * m + 1]);
      }
      // (m, b) from place 2 m + b to m + 4 b
      const C x[8] = {v[0], v[2], v[4], v[6], v[1], v[3], v[5], v[7]};
#pragma unroll
      for (int i = 0; i < 8; i++) v[i] = x[i];
    } else if constexpr (LEFT == 4) {
#pragma unroll
      for (int u = 0; u < 2; u++)
        bfly4<R, SIGN, true>(v[u], v[u + 2], v[u + 4], v[u + 6], qt[(t + TL * u) * (N / L)]);
    } else {
#pragma unroll
      for (int u = 0; u < 4; u++) {
        v[u + 4] = turn<SIGN>(v[u + 4], tw_half(qt, N, N / L, t + TL * u));
        bfly2(v[u], v[u + 4]);
      }
    }
  }

  // v[i] of the first L / 8 threads transformed in place (element t + i L/8)
  template <int SIGN, int LGL, int NS = 1>
  OFX_DEV void transform() {
    constexpr int L = 1 << LGL, TL = L / GW_P;
    each([&](int t, T& s) {
      if (t < TL) step<SIGN, LGL, NS>(t, s.v);
    });
    if constexpr (L / NS > GW_P) {
      OFX_SYNC();   // (everyone has read the exchange before this one)
      each([&](int t, T& s) {
        if (t >= TL) return;
        const int k = t & (NS - 1);
        C* p = buf + gw_pad(GW_P * (t - k) + k);
#pragma unroll
        for (int i = 0; i < GW_P; i++) p[gw_pad(NS * i)] = s.v[i];
      });
      OFX_SYNC();
      each([&](int t, T& s) {
        if (t >= TL) return;
        const C* p = buf + gw_pad(t);
#pragma unroll
        for (int i = 0; i < GW_P; i++) s.v[i] = p[gw_pad(TL * i)];
      });
      transform<SIGN, LGL, NS * GW_P>();
    }
  }

  // dT fr fft(ifft(IT) RW) at the owner's points, IT = |AT|^2, into the real
  // parts of v: the real convolution at half length on packed data, as in
  // gnlse_rhs
  OFX_DEV void raman() {
    const R inv_n = (R)(1.0 / (double)N);
    R* rb = reinterpret_cast<R*>(buf);
    OFX_SYNC();
    each([&](int t, T& s) {
#pragma unroll
      for (int i = 0; i < GW_P; i++)
        rb[t + NT * i] = s.at[i].x * s.at[i].x + s.at[i].y * s.at[i].y;
    });
    OFX_SYNC();
    each([&](int t, T& s) {
      if (t >= NH) return;
#pragma unroll
      for (int i = 0; i < GW_P; i++) s.v[i] = mkc<R>(rb[2 * (t + NH * i)], rb[2 * (t + NH * i) + 1]);
    });
    refresh();
    transform<1, LG - 1>();
    refresh();
    // Zi[k] and Zi[H - k] meet through LDS
    OFX_SYNC();
    each([&](int t, T& s) {
      if (t >= NH) return;
#pragma unroll
      for (int i = 0; i < GW_P; i++) buf[t + NH * i] = s.v[i];
    });
    OFX_SYNC();
    each([&](int t, T& s) {
      if (t >= NH) return;
#pragma unroll
      for (int i = 0; i < GW_P; i++) {
        const int k = t + NH * i;
        const C a = s.v[i], b = buf[k == 0 ? 0 : H - k];
        const C bc = mkc<R>(b.x, -b.y);
        const C E = cscale(cadd(a, bc), R(0.5));
        const C d = csub(a, bc);
        const C O = mkc<R>(R(0.5) * d.y, R(-0.5) * d.x);   // d / 2i
        const C w = tw_half(qt, N, 1, k);                    // exp(-2 pi i k / N)
        const C wO = cmulc(O, w);
        const C x0 = cscale(cmul(cadd(E, wO), ldg(RW, k)), inv_n);
        const C x1 = cscale(cmul(csub(E, wO), ldg(RW, k + H)), inv_n);
        const C P = cadd(x0, x1), Q = cmul(csub(x0, x1), w);
        s.v[i] = mkc<R>(P.x - Q.y, P.y + Q.x);   // P + i Q
        gw_group(i);
      }
    });
    refresh();
    transform<-1, LG - 1>();
    refresh();
    OFX_SYNC();
    each([&](int t, T& s) {
      if (t >= NH) return;
#pragma unroll
      for (int i = 0; i < GW_P; i++) {
        rb[2 * (t + NH * i)] = s.v[i].x;
        rb[2 * (t + NH * i) + 1] = s.v[i].y;
      }
    });
    OFX_SYNC();
    each([&](int t, T& s) {
#pragma unroll
      for (int i = 0; i < GW_P; i++) s.v[i].x = rb[t + NT * i];
    });
  }

  // f = rhs(z, y + h sum_{j <= k} DP_B[j][k] f_j) (gnlsefib.m:49-61; k < 0:
  // rhs(z, y)).  keep (the last stage): the argument is stored there, *norm
  // gets its squared norm and *err ||sum_j DP_E[j] f_j||^2, j < 7, with f the
  // seventh.
  OFX_DEV void rhs(double z, const C* y, double h, int k, C* f, C* keep, double* norm,
                   double* err) {
    const R gf = (R)exp(lre * z), gb = (R)(exp(-lre * z) / (double)N);
    const OFX_GLOBAL C* yg = gl(y);
    double sn = 0.0, se = 0.0;
    refresh();
    each([&](int t, T& s) {
#pragma unroll
      for (int i = 0; i < GW_P; i++) s.v[i] = mkc<R>(R(0), R(0));
      C y0[GW_P];
#pragma unroll
      for (int i = 0; i < GW_P; i++) y0[i] = ldg(yg, t + NT * i);
#pragma unroll 2
      for (int j = 0; j <= k; j++) {
        const double b = DP_B[j][k];
        const R c = (R)(h * b);
        const OFX_GLOBAL C* fg = gl(stage(j));
#pragma unroll
        for (int i = 0; i < GW_P; i++) {
          const C x = ldg(fg, t + NT * i);
          s.v[i].x = s.v[i].x + c * x.x;
          s.v[i].y = s.v[i].y + c * x.y;
        }
      }
#pragma unroll
      for (int i = 0; i < GW_P; i++) s.v[i] = cadd(y0[i], s.v[i]);
      if (keep) {
        OFX_GLOBAL C* kg = gl(keep);
#pragma unroll
        for (int i = 0; i < GW_P; i++) {
          stg(kg, t + NT * i, s.v[i]);
          const double x = (double)s.v[i].x, w = (double)s.v[i].y;
          sn += x * x + w * w;
          gw_group(i);
        }
      }
#pragma unroll
      for (int i = 0; i < GW_P; i++) {
        s.ph[i] = gw_expi(B[t + NT * i] * z, R(0));
        s.v[i] = cscale(cmul(s.v[i], s.ph[i]), gf);
        gw_group(i);
      }
    });
    transform<-1, LG>();
    refresh();
    if (RW) {
      each([&](int, T& s) {
#pragma unroll
        for (int i = 0; i < GW_P; i++) s.at[i] = s.v[i];
      });
      raman();
      const R dfr = (R)(dT * fr), one_fr = (R)(1.0 - fr);
      each([&](int, T& s) {
#pragma unroll
        for (int i = 0; i < GW_P; i++) {
          const C a = s.at[i];
          s.v[i] = cscale(a, one_fr * (a.x * a.x + a.y * a.y) + dfr * s.v[i].x);
        }
      });
    } else {
      each([&](int, T& s) {
#pragma unroll
        for (int i = 0; i < GW_P; i++)
          s.v[i] = cscale(s.v[i], s.v[i].x * s.v[i].x + s.v[i].y * s.v[i].y);
      });
    }
    refresh();
    transform<1, LG>();
    refresh();
    // rhs = i gamma W (M / n) exp(-L z), M = n ifft(.)
    const R gW = (R)gamma;
    OFX_GLOBAL C* fo = gl(f);
    each([&](int t, T& s) {
#pragma unroll
      for (int i = 0; i < GW_P; i++) {
        const C m = cscale(cmulc(s.v[i], s.ph[i]), gb);
        const R g = gW * W[t + NT * i];
        s.v[i] = mkc<R>(-g * m.y, g * m.x);
        stg(fo, t + NT * i, s.v[i]);
        gw_group(i);
      }
      if (keep) {
        double ax[GW_P], ay[GW_P];
#pragma unroll
        for (int i = 0; i < GW_P; i++) ax[i] = ay[i] = 0.0;
#pragma unroll 1
        for (int j = 0; j < 6; j++) {
          const double e = DP_E[j];
          if (e == 0.0) continue;
          const OFX_GLOBAL C* fg = gl(stage(j));
#pragma unroll
          for (int i = 0; i < GW_P; i++) {
            const C x = ldg(fg, t + NT * i);
            ax[i] += e * (double)x.x;
            ay[i] += e * (double)x.y;
          }
        }
#pragma unroll
        for (int i = 0; i < GW_P; i++) {
          const double x = ax[i] + DP_E[6] * (double)s.v[i].x;
          const double w = ay[i] + DP_E[6] * (double)s.v[i].y;
          se += x * x + w * w;
        }
      }
    });
    if (keep) {
      *norm = wg_sum(sn, red);
      *err = wg_sum(se, red);
    }
  }

  // o = y + sum_j cs[j] f_j over the seven stages (y itself without cs)
  OFX_DEV void write_out(const C* y, const double* cs, double* o) {
    const OFX_GLOBAL C* yg = gl(y);
    each([&](int t, T&) {
#pragma unroll 2
      for (int i = 0; i < GW_P; i++) {
        const int at = t + NT * i;
        C v = ldg(yg, at);
        if (cs) {
          R ax = R(0), ay = R(0);
#pragma unroll
          for (int j = 0; j < 7; j++) {
            const C x = ldg(gl(stage(j)), at);
            ax += (R)cs[j] * x.x;
            ay += (R)cs[j] * x.y;
          }
          v = mkc<R>(v.x + ax, v.y + ay);
        }
        gl(o)[2 * at] = (double)v.x;
        gl(o)[2 * at + 1] = (double)v.y;
      }
    });
  }

  // squared norm of v; *finite: no entry is infinite or NaN
  OFX_DEV double norm2_of(const C* v, bool* finite) {
    double s = 0.0, bad = 0.0;
    each([&](int t, T&) {
      for (int i = 0; i < GW_P; i++) {
        const C x = ldg(gl(v), t + NT * i);
        const double a = (double)x.x, b = (double)x.y;
        if (!(fabs(a) <= 1.7976931348623157e308) || !(fabs(b) <= 1.7976931348623157e308)) bad = 1.0;
        s += a * a + b * b;
      }
    });
    if (finite) *finite = wg_sum(bad, red) == 0.0;
    return wg_sum(s, red);
  }

  // ode45 over zs[0] .. zs[nsaves - 1] (the control of gnlse_instance)
  OFX_DEV void integrate(const GnlseArgs& a, int inst, C* lbuf, C* ltw) {
    buf = lbuf;
#ifdef OFX_EMU
    tid = 0;
#else
    tid = (int)threadIdx.x;
#endif
    each([&](int t, T&) {
      for (int i = t; i < gw_table_size(LG); i += NT) ltw[i] = ((const C*)a.tw)[i];
    });
    tw = ltw;
    qt = ltw + gw_qt_at(LG);
    B = gl(a.B + (size_t)inst * N);
    W = gl((const R*)a.W + (size_t)inst * N);
    RW = a.RW ? gl((const C*)a.RW + (size_t)inst * N) : nullptr;
    lre = a.lre[inst];
    gamma = a.gamma[inst];
    fr = a.fr[inst];
    dT = a.dT[inst];
    ws = (C*)a.ws + (size_t)inst * 11 * N;
    f0 = ws;
    f6 = ws + (size_t)6 * N;
    C* y = ws + (size_t)7 * N;
    C* ynew = ws + (size_t)8 * N;
    double* out = a.out + (size_t)inst * a.nsaves * 2 * N;
    each([&](int t, T&) {
      for (int i = 0; i < GW_P; i++) {
        const double* p = a.y0 + ((size_t)inst * N + t + NT * i) * 2;
        y[t + NT * i] = mkc<R>((R)p[0], (R)p[1]);
      }
    });
    write_out(y, nullptr, out);
    const double t0 = a.zs[0], tfinal = a.zs[a.nsaves - 1];
    const double tdir = tfinal >= t0 ? 1.0 : -1.0;
    const double rtol = a.rtol, pw = 1.0 / 5.0;
    const double threshold = a.atol / rtol;
    const double hmax = 0.1 * fabs(tfinal - t0);
    double t = t0;
    OFX_SYNC();
    rhs(t, y, 0.0, -1, f0, nullptr, nullptr, nullptr);
    long long nfev = 1, acc = 0, rej = 0;
    int status = GNLSE_OK;
    double normy = sqrt(norm2_of(y, nullptr));
    double hmin = 16.0 * eps_of(t);
    double absh = fmin(hmax, fabs(a.zs[1] - a.zs[0]));
    const double rh =
        (sqrt(norm2_of(f0, nullptr)) / fmax(normy, threshold)) / (0.8 * pow(rtol, pw));
    if (absh * rh > 1.0) absh = 1.0 / rh;
    absh = fmax(absh, hmin);
    int nxt = 1;
    bool done = false;
    while (!done) {
      hmin = 16.0 * eps_of(t);
      absh = fmin(hmax, fmax(hmin, absh));
      double h = tdir * absh;
      if (1.1 * absh >= fabs(tfinal - t)) {
        h = tfinal - t;
        absh = fabs(h);
        done = true;
      }
      bool nofailed = true;
      double err = 0.0, normynew = 0.0, tnew = t;
      for (;;) {
#pragma unroll 1
        for (int k = 0; k < 6; k++) {
          const double hk = h;
          double tk;
          if (k < 5) {
            tk = t + h * DP_A[k];
          } else {
            tnew = t + h * DP_A[5];
            if (done) tnew = tfinal;
            h = tnew - t;
            tk = tnew;
          }
          rhs(tk, y, hk, k, stage(k + 1), k == 5 ? ynew : nullptr, &normynew, &err);
        }
        nfev += 6;
        normynew = sqrt(normynew);
        err = sqrt(err);
        const double errwt = fmax(fmax(normy, normynew), threshold);
        err = absh * (err / errwt);
        if (!(err == err)) {  // NaN: the field is not finite
          status = GNLSE_NONFINITE;
          break;
        }
        if (acc + rej + 1 > a.max_steps) {
          status = GNLSE_CAP;
          break;
        }
        if (!(err > rtol)) break;
        rej++;
        if (absh <= hmin) {
          status = GNLSE_HMIN;
          break;
        }
        if (nofailed) {
          nofailed = false;
          absh = fmax(hmin, absh * fmax(0.1, 0.8 * pow(rtol / err, pw)));
        } else {
          absh = fmax(hmin, 0.5 * absh);
        }
        h = tdir * absh;
        done = false;
      }
      if (status != GNLSE_OK) break;
      acc++;
      while (nxt < a.nsaves && tdir * (tnew - a.zs[nxt]) >= 0.0) {
        double* o = out + (size_t)nxt * 2 * N;
        if (a.zs[nxt] == tnew) {
          write_out(ynew, nullptr, o);
        } else {
          const double s = (a.zs[nxt] - t) / h;
          const double sv[4] = {s, s * s, s * s * s, s * s * s * s};
          double cs[7];
          for (int j = 0; j < 7; j++)
            cs[j] = h * (((DP_BI[j][0] * sv[0] + DP_BI[j][1] * sv[1]) + DP_BI[j][2] * sv[2]) +
                         DP_BI[j][3] * sv[3]);
          write_out(y, cs, o);
        }
        nxt++;
      }
      if (done) break;
      if (nofailed) {
        const double temp = 1.25 * pow(err / rtol, pw);
        absh = temp > 0.2 ? absh / temp : 5.0 * absh;
      }
      t = tnew;
      C* sw = y;
      y = ynew;
      ynew = sw;
      normy = normynew;
      sw = f0;
      f0 = f6;
      f6 = sw;
    }
    bool finite = true;
    if (status == GNLSE_OK) norm2_of(y, &finite);
    if (!finite) status = GNLSE_NONFINITE;
    if (OFX_TID == 0) {
      long long* st = a.stats + 4 * (size_t)inst;
      st[0] = acc;
      st[1] = rej;
      st[2] = nfev;
      st[3] = status;
    }
  }
};

}  // namespace ofx
