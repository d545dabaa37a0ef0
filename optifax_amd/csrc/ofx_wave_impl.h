// Body of the wave kernel: the adaptive Heun pass (RK23: ofx_wave_rk23.h) and the
// round trip of ofx_pass_impl.h for clusters whose members hold a small share of the field
// (at most 4 points a thread), where a step is a chain of latencies.
//
// The decomposition, the exchange buffers, the tags and the arithmetic of
// every sample are those of ofx_pass_impl.h (results are the same bits); what
// differs is who does the work and how often the workgroup meets:
//   * Nonlinear stages: one thread takes S consecutive columns of one row
//     with two neighbours on each side and runs both stages, the corrector
//     and the error quotient in registers, so the workgroup meets once
//     instead of three times, and 3 S + 6 evaluations of the nonlinear term
//     (8 for S = 1) replace 6 S + 6.
//   * Transforms: one wave runs 256 / L transforms of length L <= 256 with 4
//     elements a lane.  The passes exchange through the wave's own LDS slot
//     (LDS accesses of a wave are ordered), so a transform has no workgroup
//     barrier; the passes' twiddles and the four-step factors stay in
//     registers.  Forward rows, dispersion and inverse rows share the element
//     distribution (j + m L/4), so nothing moves between them; rows are
//     polled straight into the first pass's registers, and the last pass
//     stores straight to t2.
//   * The dispersion phasors are kept while the step length stays the same,
//     and the next step's exp(-i bdwz) is formed while t2 is in flight.
//   * A cluster of one workgroup transposes through LDS: no exchange at all.
// A step of the multi-wave form has 4 workgroup barriers, of the single-wave
// form none.
//
// Bound: the latency of the step's dependent chain, not arithmetic or memory: two
// exchanges (one tagged word takes about 0.5 us from one XCD to another), about 20
// LDS round trips, and 5 to 8 cycles for each instruction of a wave that is alone on
// its SIMD.  At 2^15 points the waves wait in 69 % of their cycles and issue
// vector instructions in 18 %.  A step of the same share without exchange (2^8
// points) takes 2.6 us of the 8.0; how much of the rest the polls of whole
// columns, the threefold inverse columns (2 own, 4 halo) and the members' spread
// take has not been measured apart.
// With the geometry a compile-time constant (WvGeoCt) index arithmetic, address
// registers and the branches on it go.  One instance, us per adaptive step,
// FP32, against the general kernel at its best geometry: 2^9 points 3.4 (7.9),
// 2^11 4.7 (9.0), 2^13 6.2 (11.0), 2^15 8.0 (12.7), 2^16 10.2 (15.4); FP64 2^14
// 9.9 (14.5).
#pragma once
#include "ofx_pass_impl.h"

namespace ofx {

// One wave transform's LDS slot: 256 elements, one unused element after each
// 16 (the Stockham passes' stores then spread over the banks).
#define WV_SLOT 272
OFX_DEV int wv_pad(int f) { return f + (f >> 4); }

// Orders the LDS accesses of one wave around an exchange within it (no
// instruction: the hardware keeps a wave's LDS accesses in order)
OFX_DEV void wv_order() {
#ifndef OFX_EMU
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
#endif
}

// State of one thread.  On the device one object per thread, in registers; in
// the emulation an array that each phase walks.
template <typename R, int S, int HW = 2>
struct WvThread {
  typedef cpx<R> C;
  C v[4];                  // transform elements j + m L/4
  C wt[S + 2 * HW];        // exp(i w0 t) of the stage window
  C twr[3][3], twc[3][3];  // twiddles of the passes after each exchange (rows, columns)
  C fc[4], fr[4];          // four-step factors of the own column / row elements
  C ph[4];                 // dispersion phasors for the step length held
  double beta[4];
  R alpha[4], am[4], ab[S];
  int jr, qr, jc, qc;      // element and sequence of the lane, rows and columns
  int tk2, tlc;            // first t2 entry: row, local column
};

// In-register radix-4 butterfly (ofx_pass_impl.h's arithmetic)
template <typename R, int SIGN, bool TW>
OFX_DEV void wv_r4(cpx<R>* v, const cpx<R>* w) {
  typedef cpx<R> C;
  C v0 = v[0], v1 = v[1], v2 = v[2], v3 = v[3];
  if (TW) {
    if (SIGN > 0) {
      v1 = wv_mulc(v1, w[0]);
      v2 = wv_mulc(v2, w[1]);
      v3 = wv_mulc(v3, w[2]);
    } else {
      v1 = wv_mulq(v1, w[0]);
      v2 = wv_mulq(v2, w[1]);
      v3 = wv_mulq(v3, w[2]);
    }
  }
  C s02 = cadd(v0, v2), d02 = csub(v0, v2), s13 = cadd(v1, v3), d13 = csub(v1, v3);
  C rd = (SIGN < 0) ? mkc<R>(d13.y, -d13.x) : mkc<R>(-d13.y, d13.x);
  v[0] = cadd(s02, s13);
  v[1] = cadd(d02, rd);
  v[2] = csub(s02, s13);
  v[3] = csub(d02, rd);
}

// Exchanges of a length-2^lg transform and the stride of the pass after
// exchange e (a radix-2 pass comes first for odd lg)
OFX_DEV int wv_exchanges(int lg) { return (lg & 1) ? (lg - 1) >> 1 : (lg >> 1) - 1; }
OFX_DEV int wv_stride(int lg, int e) { return (lg & 1) ? 2 << (2 * e) : 4 << (2 * e); }

// A tagged element's place: words at base + i ws (uniform) plus a 32-bit byte
// offset of the lane, so that an access needs no 64-bit lane address.
struct WvAt {
  const u64* base;
  size_t ws;
  unsigned off;
};
template <typename T>
OFX_DEV void wv_load(const WvAt& t, u64* w) {
#pragma unroll
  for (int i = 0; i < Tagged<T>::NW; i++)
    w[i] = tag_load((const u64*)((const char*)(t.base + i * t.ws) + t.off));
}
template <typename T>
OFX_DEV void wv_put(const WvAt& t, T v, unsigned tag) {
  typedef Tagged<T> TT;
  const typename TT::Words x = __builtin_bit_cast(typename TT::Words, v);
  const u64 hi = (u64)tag << 32;
#pragma unroll
  for (int i = 0; i < TT::NW; i++)
    tag_store((u64*)((char*)const_cast<u64*>(t.base + i * t.ws) + t.off), hi | (u64)x.w[i]);
}

// Poll `N` tagged elements of this thread (those of `mask`): loads are issued
// together, repeated for the words that are still old, and the clock and the
// abort flag are looked at while a repeat is in flight.
template <typename T, int N, typename Src, typename Commit>
OFX_DEV bool wv_poll(unsigned mask, unsigned tag, Src src, Commit commit, Spin& sp) {
  typedef Tagged<T> TT;
  u64 w[N][TT::NW];
  unsigned pend = mask;
#pragma unroll
  for (int j = 0; j < N; j++)
    if ((pend >> j) & 1u) {
      wv_load<T>(src(j), w[j]);
    }
  for (;;) {
#pragma unroll
    for (int j = 0; j < N; j++)
      if (((pend >> j) & 1u) && TT::check(w[j], tag)) {
        commit(j, TT::value(w[j]));
        pend &= ~(1u << j);
      }
    if (!pend) return true;
#pragma unroll
    for (int j = 0; j < N; j++)
      if ((pend >> j) & 1u) {
        wv_load<T>(src(j), w[j]);
      }
#ifdef OFX_EMU
    sched_yield();
    const unsigned long long now = emu_clock();
#else
    const unsigned long long now = wall_clock64();
#endif
    if (sp.n == 0) sp.t0 = now;
    if ((++sp.n & 7) == 0 && flag_load(sp.abort_flag)) return false;
    if (now - sp.t0 > sp.limit) {
      flag_set(sp.abort_flag);
      return false;
    }
  }
}

// max over the wave's lanes of a value that is never NaN, in every lane:
// DPP shifts within rows of 16, then across rows; lane 63 holds the result.
// (Six ds_bpermute pairs cost about 600 cycles here.)
#ifndef OFX_EMU
template <int CTRL>
OFX_DEV double wv_dpp_max(double v) {
  const u64 u = __builtin_bit_cast(u64, v);
  const int lo = (int)(unsigned)u, hi = (int)(unsigned)(u >> 32);
  const unsigned plo = (unsigned)__builtin_amdgcn_update_dpp(lo, lo, CTRL, 0xf, 0xf, false);
  const unsigned phi = (unsigned)__builtin_amdgcn_update_dpp(hi, hi, CTRL, 0xf, 0xf, false);
  const double o = __builtin_bit_cast(double, ((u64)phi << 32) | plo);
  return o > v ? o : v;
}
OFX_DEV double wv_wave_max(double v) {
  v = wv_dpp_max<0x111>(v);  // row_shr:1
  v = wv_dpp_max<0x112>(v);  // row_shr:2
  v = wv_dpp_max<0x114>(v);  // row_shr:4
  v = wv_dpp_max<0x118>(v);  // row_shr:8
  v = wv_dpp_max<0x142>(v);  // row_bcast:15
  v = wv_dpp_max<0x143>(v);  // row_bcast:31
  const u64 u = __builtin_bit_cast(u64, v);
  const unsigned lo = (unsigned)__builtin_amdgcn_readlane((int)(unsigned)u, 63);
  const unsigned hi = (unsigned)__builtin_amdgcn_readlane((int)(unsigned)(u >> 32), 63);
  return __builtin_bit_cast(double, ((u64)hi << 32) | lo);
}
#endif

// Launch geometry of a member (HW: halo columns on each side): read from the
// instance and the launch ...
template <int HW_ = 2>
struct WvGeoRt {
  static constexpr bool FIXED = false;
  static constexpr int HW = HW_;
  int n, n1, n2, lg1, lg2, lgW, Cn, W, Rr, LC, sT, NT, nw;
  OFX_DEV void set(const InstDesc& d, int C, int block) {
    n = d.n;
    n1 = d.n1;
    n2 = d.n2;
    lg1 = d.lg1;
    lg2 = d.lg2;
    Cn = C;
    int lgC = 0;
    while ((1 << lgC) < C) lgC++;
    W = n1 >> lgC;
    lgW = lg1 - lgC;
    Rr = n2 >> lgC;
    LC = W + 2 * HW;
    sT = n2 + 1;
    NT = block;
    nw = NT >> 6;
  }
};
// ... or fixed for a grid size's default geometry: shifts, strides, slot and
// wave counts are then constants (about half of a step's instructions form
// indices otherwise).
template <int LG, int LGC, int NT_, int HW_ = 2>
struct WvGeoCt {
  static constexpr bool FIXED = true;
  static constexpr int n = 1 << LG, lg1 = (LG + 1) / 2, lg2 = LG - lg1, n1 = 1 << lg1, n2 = 1 << lg2,
                       Cn = 1 << LGC, W = n1 >> LGC, lgW = lg1 - LGC, Rr = n2 >> LGC, HW = HW_,
                       LC = W + 2 * HW, sT = n2 + 1, NT = NT_, nw = NT >> 6;
  OFX_DEV void set(const InstDesc&, int, int) {}
};

// One member's share of one instance.
template <typename R, int S, typename GEO, bool REFRESH>
struct WvRun : GEO {
  typedef cpx<R> C;
  typedef Tagged<C> TT;
  typedef WvThread<R, S, GEO::HW> T;
  using GEO::n; using GEO::n1; using GEO::n2; using GEO::lg1; using GEO::lg2; using GEO::lgW;
  using GEO::Cn; using GEO::W; using GEO::Rr; using GEO::LC; using GEO::sT; using GEO::NT;
  using GEO::nw; using GEO::HW;
  const LaunchArgs& a;
  const ClusterDesc& cd;
  const InstDesc& d;
  SyncState& sy;
  double* red;   // [0, 16) wave maxima, [32] the cluster's maximum
  int* sflag;    // [0] barrier verdict, [1] a poll gave up
  T* thr;
  int rank, wv, tid, c0, k20;
  C *A0, *X, *Tb, *K1;   // (K1: RK23 only, two buffers of A0's layout)
  u64 *t1b, *t2b, *slots;
  int* abort_flag;

  OFX_DEV WvRun(const LaunchArgs& a_, const ClusterDesc& cd_, const InstDesc& d_, SyncState& sy_,
                double* red_, int* sflag_, T* thr_)
      : a(a_), cd(cd_), d(d_), sy(sy_), red(red_), sflag(sflag_), thr(thr_) {}

  // f(thread id, wave, state) for every thread of the workgroup
  template <typename F>
  OFX_DEV void each(F f) {
#ifdef OFX_EMU
    for (int t = 0; t < NT; t++) f(t, t >> 6, thr[t]);
#else
    f(tid, wv, *thr);
#endif
  }
  // Hides where the lane's indices come from, so that the addresses formed
  // from them are formed again in every step instead of being kept in
  // registers across it.  Kept they are 10 % faster with a fixed geometry (2^15
  // points 8.0 against 8.6 us per step) and, where they fit, with a run-time one
  // (FP32 fields in workgroups of 256: 9.0 against 10.0); elsewhere they spill
  // (FP64 14.6 against 13.4, 512 threads 18.9 against 11.9).  The fixed geometries
  // in FP64 and FP32 2^10 and 2^16 keep them too, though from FP64 2^11 on (but
  // 2^12) and at FP32 2^16 they use 68 to 368 bytes of scratch a lane for it.
  // us per step, kept / formed again: FP64 2^8 3.15 / 3.44, 2^10 6.1 / 6.3, 2^11 7.4
  // / 7.1, 2^12 7.9 / 8.5, 2^13 10.6 / 10.6, 2^14 10.5 / 10.0, 2^15 11.2 / 11.4, 2^16
  // 16.4 / 15.8; FP32 2^10 4.3 / 5.0, 2^16 10.7 / 10.2.
  OFX_DEV void refresh() {
#ifndef OFX_EMU
    if constexpr (REFRESH)
      asm volatile("" : "+v"(tid), "+v"(thr->jr), "+v"(thr->qr), "+v"(thr->jc), "+v"(thr->qc));
#endif
  }
  // workgroup barrier (one wave needs none: only the order of its accesses)
  OFX_DEV void meet() {
#ifndef OFX_EMU
    if (nw > 1)
      __syncthreads();
    else
      wv_order();
#endif
  }

  // 256 / 2^lg transforms in each of the first `act` waves, element j + m L/4
  // of sequence q in v[m]; slot: the waves' slots.
  template <int SIGN, bool ROWS>
  OFX_DEV void fft(int lg, int act, C* slots) {
#ifndef OFX_EMU
    if (wv >= act) return;
#endif
    const int L = 1 << lg, l4 = L >> 2, odd = lg & 1, ne = wv_exchanges(lg);
    const C one = mkc<R>(R(1), R(0));
    each([&](int, int w, T& t) {
      if (w >= act) return;
      if (odd) {
        const C a0 = cadd(t.v[0], t.v[2]), a1 = csub(t.v[0], t.v[2]);
        const C b0 = cadd(t.v[1], t.v[3]), b1 = csub(t.v[1], t.v[3]);
        t.v[0] = a0;
        t.v[1] = a1;
        t.v[2] = b0;
        t.v[3] = b1;
      } else {
        wv_r4<R, SIGN, false>(t.v, &one);
      }
    });
#pragma unroll
    for (int e = 0; e < 3; e++) {
      if (e >= ne) break;
      each([&](int, int w, T& t) {
        if (w >= act) return;
        const int q = ROWS ? t.qr : t.qc, j = ROWS ? t.jr : t.jc;
        C* b = slots + w * WV_SLOT;
        if (odd) {
          if (e == 0) {
            C* p = b + wv_pad(q * L + 2 * j);
            const int o = wv_pad(L >> 1);
            p[0] = t.v[0];
            p[1] = t.v[1];
            p[o] = t.v[2];
            p[o + 1] = t.v[3];
          } else {
            const int ns = e == 1 ? 2 : 8, k = j & (ns - 1);
            C* p = b + wv_pad(q * L + ((j - k) << 2) + k);
#pragma unroll
            for (int m = 0; m < 4; m++) p[wv_pad(ns * m)] = t.v[m];
          }
        } else {
          const int ns = e == 0 ? 1 : (e == 1 ? 4 : 16), k = j & (ns - 1);
          C* p = b + wv_pad(q * L + ((j - k) << 2) + k);
#pragma unroll
          for (int m = 0; m < 4; m++) p[wv_pad(ns * m)] = t.v[m];
        }
      });
      wv_order();
      each([&](int, int w, T& t) {
        if (w >= act) return;
        const int q = ROWS ? t.qr : t.qc, j = ROWS ? t.jr : t.jc;
        const C* p = slots + w * WV_SLOT + wv_pad(q * L + j);
#pragma unroll
        for (int m = 0; m < 4; m++) t.v[m] = p[wv_pad(l4 * m)];
        wv_r4<R, SIGN, true>(t.v, ROWS ? t.twr[e] : t.twc[e]);
      });
      wv_order();
    }
  }

  OFX_DEV u64* t1_of(unsigned x) { return t1b + (size_t)(x & 1u) * n * TT::NW; }
  OFX_DEV u64* t2_of(unsigned x) { return t2b + (size_t)(x & 1u) * n * TT::NW; }
  // member `q`'s error record of exchange x (slot_at's wave 0, value 0)
  OFX_DEV u64* record_of(unsigned x, int q) {
    return slots + ((size_t)(x & 1u) * OFX_SLOT_WAVES * 4 * Cn + q) * TT::NW;
  }
  OFX_DEV Spin spin() { return Spin{abort_flag, a.timeout_ticks, 0, 0}; }
  // entry of sample (column c, row k2) in t1 (member-blocked, see ofx_pass_impl.h)
  OFX_DEV unsigned t1_at(int c, int k2) {
    return ((((unsigned)(c >> lgW) << lg2) + (unsigned)k2) << lgW) + (unsigned)(c & (W - 1));
  }
  OFX_DEV int col_waves() { return (W * n2 + 255) >> 8; }
  OFX_DEV int row_waves() { return (Rr * n1 + 255) >> 8; }

  // per-thread constants of the instance
  OFX_DEV void setup() {
    const C* twg = (const C*)a.twiddle;
    const C* wtg = (const C*)d.wt;
    const R* abg = (const R*)d.absorb;
    each([&](int tid, int w, T& t) {
      const int lane = tid & 63;
      t.qr = lane >> (lg1 - 2);
      t.jr = lane & ((n1 >> 2) - 1);
      t.qc = lane >> (lg2 - 2);
      t.jc = lane & ((n2 >> 2) - 1);
#pragma unroll
      for (int e = 0; e < 3; e++) {
#pragma unroll
        for (int c = 0; c < 3; c++) {
          t.twr[e][c] = mkc<R>(R(1), R(0));
          t.twc[e][c] = mkc<R>(R(1), R(0));
        }
        if (e < wv_exchanges(lg1)) {
          const int ns = wv_stride(lg1, e), k = t.jr & (ns - 1);
#pragma unroll
          for (int c = 0; c < 3; c++) t.twr[e][c] = twg[(c + 1) * k * (a.nmax / (4 * ns))];
        }
        if (e < wv_exchanges(lg2)) {
          const int ns = wv_stride(lg2, e), k = t.jc & (ns - 1);
#pragma unroll
          for (int c = 0; c < 3; c++) t.twc[e][c] = twg[(c + 1) * k * (a.nmax / (4 * ns))];
        }
      }
      const int cl = w * (256 >> lg2) + t.qc, rl = w * (256 >> lg1) + t.qr;
      const double TWO_PI = 6.283185307179586232;
      // the four-step factor exp(-2 pi i c k2 / n) as the FP64 product of two
      // unit phasors, rounded once (element i: columns 0..3, rows 4..7)
#pragma unroll 1
      for (int i = 0; i < 8; i++) {
        const int c = i < 4 ? c0 + cl : t.jr + (i & 3) * (n1 >> 2);
        const int k2 = i < 4 ? t.jc + (i & 3) * (n2 >> 2) : k20 + rl;
        const int m = (c * k2) & (n - 1), q = m >> lg1, r = m & (n1 - 1);
        const double aq = -TWO_PI * (double)q / (double)n2;
        const double ar = -TWO_PI * (double)r / (double)n;
        const double qx = cos(aq), qy = sin(aq), rx = cos(ar), ry = sin(ar);
        const C f = mkc<R>((R)wv_fma(qx, rx, -(qy * ry)), (R)wv_fma(qy, rx, qx * ry));
#pragma unroll
        for (int u = 0; u < 4; u++) {
          if (i == u) t.fc[u] = f;
          if (i == u + 4) t.fr[u] = f;
        }
      }
#pragma unroll
      for (int m = 0; m < 4; m++) {
        t.beta[m] = 0.0;
        t.alpha[m] = R(0);
        t.ph[m] = mkc<R>(R(1), R(0));
        t.am[m] = R(1);
        if (rl < Rr) {
          const int kk = (k20 + rl) + n2 * (t.jr + m * (n1 >> 2));
          t.beta[m] = gl(d.beta)[kk];
          t.alpha[m] = (R)gl(d.alpha)[kk];
        }
      }
      const int r = tid & (n2 - 1), s0 = (tid >> lg2) * S;
#pragma unroll
      for (int i = 0; i < S + 2 * HW; i++) {
        const int lc = s0 + i < LC ? s0 + i : LC - 1;
        const int j = (c0 - HW + lc + n1 * r) & (n - 1);
        t.wt[i] = wv_mulq(wtg[(j >> lg1) * n1], wtg[j & (n1 - 1)]);
      }
#pragma unroll
      for (int i = 0; i < S; i++)
        t.ab[i] = s0 + i < W ? abg[(c0 + s0 + i + n1 * r) & (n - 1)] : R(1);
      t.tk2 = tid / LC;
      t.tlc = tid - t.tk2 * LC;
    });
  }

  // Forward transforms of the own columns, elements from src(column, row),
  // twiddled, to t1 (or to LDS in a cluster of one)
  template <typename Src>
  OFX_DEV void columns_forward(Src src, unsigned x, unsigned tag) {
    const int act = col_waves(), l4 = n2 >> 2, qn = 256 >> lg2;
    each([&](int, int w, T& t) {
      if (w >= act) return;
      const int cl = w * qn + t.qc;
#pragma unroll
      for (int m = 0; m < 4; m++) t.v[m] = src(cl < W ? cl : W - 1, t.jc + l4 * m);
    });
    wv_order();
    fft<-1, false>(lg2, act, X);
    u64* const t1 = t1_of(x);
    each([&](int, int w, T& t) {
      const int cl = w * qn + t.qc;
      if (w >= act || cl >= W) return;
#pragma unroll
      for (int m = 0; m < 4; m++) {
        const int k2 = t.jc + l4 * m;
        const C v = wv_mul(t.v[m], t.fc[m]);
        if (Cn == 1)
          Tb[wv_pad((k2 << lg1) + cl)] = v;
        else
          wv_put<C>(WvAt{t1, (size_t)n, t1_at(c0 + cl, k2) * 8u}, v, tag);
      }
    });
  }

  // Inverse transforms of the own rows (elements in v), twiddled, to t2 (or
  // to LDS in a cluster of one)
  OFX_DEV void rows_inverse(unsigned x, unsigned tag) {
    const int act = row_waves(), l4 = n1 >> 2, qn = 256 >> lg1;
    fft<1, true>(lg1, act, Tb);
    u64* const t2 = t2_of(x);
    each([&](int, int w, T& t) {
      const int rl = w * qn + t.qr;
      if (w >= act || rl >= Rr) return;
#pragma unroll
      for (int m = 0; m < 4; m++) {
        const int c = t.jr + l4 * m;
        const C v = wv_mulc(t.v[m], t.fr[m]);
        if (Cn == 1)
          X[wv_pad((c << lg2) + rl)] = v;
        else
          wv_put<C>(WvAt{t2, (size_t)n, (unsigned)(((k20 + rl) << lg1) + c) * 8u}, v, tag);
      }
    });
  }

  // The own rows of t1 (and, for an attempt of the pass, the cluster's error
  // records) into the first row pass's elements.  With records in a cluster of
  // several workgroups the caller meets before it reads the cluster's error
  // maximum in red[32] and whether a poll gave up in sflag[1]; otherwise this
  // meets, and only sflag[1] is set.
  OFX_DEV void rows_in(unsigned x, unsigned tag, bool records) {
    const int act = row_waves(), l4 = n1 >> 2, qn = 256 >> lg1;
    if (Cn == 1) {
      meet();
      each([&](int, int w, T& t) {
        if (w >= act) return;
        const C* p = Tb + w * WV_SLOT;
#pragma unroll
        for (int m = 0; m < 4; m++) t.v[m] = p[wv_pad((t.qr << lg1) + t.jr + l4 * m)];
      });
      wv_order();
      return;
    }
    const u64* t1 = t1_of(x);
    bool ok = true;
    double v = -1.0;
    each([&](int tid, int w, T& t) {
      const int rl = w * qn + t.qr, lane = tid & 63;
      unsigned mask = w < act && rl < Rr ? 0xfu : 0u;
      if (records && w == nw - 1)
        mask |= (lane < Cn ? 0x10u : 0u) | (lane + 64 < Cn ? 0x20u : 0u);
      Spin sp = spin();
      ok = wv_poll<C, 6>(
               mask, tag,
               [&](int j) -> WvAt {
                 if (j < 4) return WvAt{t1, (size_t)n, t1_at(t.jr + l4 * j, k20 + rl) * 8u};
                 return WvAt{record_of(x, 0), 1, (unsigned)((lane + 64 * (j - 4)) * TT::NW) * 8u};
               },
               [&](int j, C c) {
                 if (j < 4)
                   t.v[j] = c;
                 else
                   v = red_op(v, unpack_d<R>(c), 0);
               },
               sp) &&
           ok;
      if (!ok) sflag[1] = 1;
    });
#ifdef OFX_EMU
    red[32] = v;
#else
    if (records && wv == nw - 1) {
      v = wv_wave_max(v);
      red[32] = v;
    }
#endif
    if (!records) meet();
  }

  // Own and halo columns of the inverse transform, scaled, into A0.  Meets
  // twice; false (uniform) when the cluster gave up.
  OFX_DEV bool columns_inverse(unsigned x, unsigned tag) {
    const int l4 = n2 >> 2, qn = 256 >> lg2;
    const R inv = R(1) / R(n);
    if (Cn == 1) {
      meet();
      const int act = col_waves();
      each([&](int, int w, T& t) {
        if (w >= act) return;
        const C* p = X + w * WV_SLOT;
#pragma unroll
        for (int m = 0; m < 4; m++) t.v[m] = p[wv_pad((t.qc << lg2) + t.jc + l4 * m)];
      });
      wv_order();
      fft<1, false>(lg2, act, X);
      each([&](int, int w, T& t) {
        const int c = w * qn + t.qc;
        if (w >= act || c >= W) return;
#pragma unroll
        for (int m = 0; m < 4; m++) {
          const int r = t.jc + l4 * m;
          const C v = cscale(t.v[m], inv);
          A0[(HW + c) * sT + r] = v;
          // the wrapped copies carry a row shift
          if (c < HW) A0[(HW + W + c) * sT + ((r - 1) & (n2 - 1))] = v;
          if (c >= W - HW) A0[(c - (W - HW)) * sT + ((r + 1) & (n2 - 1))] = v;
        }
      });
      meet();
      return true;
    }
    const u64* t2 = t2_of(x);
    const int tot = LC * n2, dk = NT / LC, dl = NT - dk * LC;
    bool ok = true;
    each([&](int tid, int, T& t) {
      int k2 = t.tk2, lc = t.tlc;
      Spin sp = spin();
      for (int base = tid; base < tot && ok; base += 4 * NT) {
        unsigned src[4];
        int dst[4];
        unsigned mask = 0;
#pragma unroll
        for (int b = 0; b < 4; b++) {
          const int gc = (c0 - HW + lc) & (n1 - 1);
          src[b] = (unsigned)((k2 << lg1) + gc);
          dst[b] = wv_pad((lc << lg2) + k2);
          if (base + b * NT < tot) mask |= 1u << b;
          k2 += dk;
          lc += dl;
          if (lc >= LC) {
            lc -= LC;
            k2++;
          }
        }
        ok = wv_poll<C, 4>(
            mask, tag, [&](int b) { return WvAt{t2, (size_t)n, src[b] * 8u}; },
            [&](int b, C v) { X[dst[b]] = v; }, sp);
      }
      if (!ok) sflag[1] = 1;
    });
    meet();
    const int slots = (tot + 255) >> 8;
    for (int s = 0; s < slots; s += nw) {
      const int act = slots - s < nw ? slots - s : nw;
      each([&](int, int w, T& t) {
        if (w >= act) return;
        const C* p = X + (s + w) * WV_SLOT;
#pragma unroll
        for (int m = 0; m < 4; m++) t.v[m] = p[wv_pad((t.qc << lg2) + t.jc + l4 * m)];
      });
      wv_order();
      fft<1, false>(lg2, act, X + s * WV_SLOT);
      each([&](int, int w, T& t) {
        const int lc = (s + w) * qn + t.qc;
        if (w >= act || lc >= LC) return;
        const int gc = c0 - HW + lc;
        const int sh = gc < 0 ? 1 : (gc >= n1 ? -1 : 0);
#pragma unroll
        for (int m = 0; m < 4; m++) {
          const int r = (t.jc + l4 * m + sh) & (n2 - 1);
          A0[lc * sT + r] = cscale(t.v[m], inv);
        }
      });
    }
    const bool fail = sflag[1] != 0;
    meet();
    return !fail;
  }

  // one adaptive RK23 pass (ofx_wave_rk23.h)
  OFX_DEV int rk23(R cc, long long& att, long long& acc, double& s_held);
  OFX_DEV void boundary_in(unsigned x, unsigned tag, C* dst);

  OFX_DEV void run(int rank_, C* lds);
};

template <typename R, int S, typename GEO, bool REFRESH>
OFX_DEV void WvRun<R, S, GEO, REFRESH>::run(int rank_, C* lds) {
  // converged in an earlier launch (and not rewritten since): nothing to do
  if (a.conv_tol > 0.0 && a.trips > 0 && d.status[0] == ST_CONVERGED) return;
  rank = rank_;
#ifdef OFX_EMU
  wv = tid = 0;
#else
  tid = (int)threadIdx.x;
  wv = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
#endif
  GEO::set(d, cd.C, a.block);
  c0 = rank * W;
  k20 = rank * Rr;
  t1b = (u64*)uniform(cd.t1);
  t2b = (u64*)uniform(cd.t2);
  slots = (u64*)uniform(cd.slots);
  abort_flag = uniform(cd.abort_flag);
  A0 = lds;
  X = A0 + LC * sT;
  Tb = X + ((LC * n2 + 255) >> 8) * WV_SLOT;
  K1 = Tb + ((Rr * n1 + 255) >> 8) * WV_SLOT;
  C* field = (C*)d.field;
  const double dt = d.dt;
  const R cc = (R)(0.5 / dt / d.w0);
  const int nsteps = uniform(d.nsteps);
  const double sel = uniform(d.sel);
  const double nChunks = (double)nsteps / sel;
  const bool cavity = a.trips > 0 && d.cav != nullptr;
  const int trips = a.trips > 0 ? a.trips : 1;
  int status = ST_RUNNING;
  long long attempts = 0, accepted = 0;
  const int trip_base = d.trips_done[0];
  const bool fresh = d.fresh[0] != 0;
  const double* const Gd = uniform(d.G);
  const double bdiffw0 = uniform(d.bdiffw0), hmin = uniform(d.h);
  const double max_err = uniform(d.max_err), min_err = uniform(d.min_err);
  float* const stepmods = uniform(d.stepmods);
  C* const apft = uniform((C*)d.apft);
  const int n_cols = uniform(d.n_cols);

  setup();
  each([&](int tid, int, T&) {
    for (int idx = tid; idx < LC * n2; idx += NT) {
      const int lc = idx >> lg2, r = idx & (n2 - 1);
      A0[lc * sT + r] = field[(c0 - HW + lc + n1 * r) & (n - 1)];
    }
    if (tid == 0) sflag[1] = 0;
  });
  meet();
  double s_held = 0.0;  // step length of the phasors in ph / am

  int trip = 0;
  for (; trip < trips && status == ST_RUNNING; trip++) {
    long long trip_att = 0, trip_acc = 0;
    double k = 1.0, stepmod = 4.0;
    int chunk = 1;
    // step multipliers start each trip from a zero row; entry j belongs to
    // thread j mod NT, so program order orders its clear, writes and copy
    if (a.trips > 0 && rank == 0 && stepmods)
      each([&](int tid, int, T&) {
        for (int j = tid; j < nsteps; j += NT) gl(stepmods)[j] = 0.0f;
      });
    if constexpr (HW == 4) {
      status = rk23(cc, trip_att, trip_acc, s_held);
      attempts += trip_att;
      accepted += trip_acc;
      chunk = (int)nChunks + 1;  // (no Heun loop)
    }
    double Gk = (double)chunk <= nChunks ? uniform(gl(Gd)[(int)k - 1]) : 0.0;
    // exp(-i bdwz) at both ends of the step
    C eb0 = expi(-(bdiffw0 * (k - 1.0) * hmin), R(0));
    C eb1 = expi(-(bdiffw0 * (k - 1.0 + stepmod) * hmin), R(0));
    if constexpr (HW == 2) while ((double)chunk <= nChunks) {
      refresh();
      const R gk = (R)(hmin * stepmod * Gk);
      // ---- both stages, corrector, error quotient, absorber ----
      double lmax = -1.0;
      int bad = 0;
      each([&](int tid, int, T& t) {
        const int r = tid & (n2 - 1), s0 = (tid >> lg2) * S;
        if (s0 >= W) return;
        C x[S + 4], f[S + 4], k1[S + 4];
#pragma unroll
        for (int i = 0; i < S + 4; i++) x[i] = A0[(s0 + i < LC ? s0 + i : LC - 1) * sT + r];
#pragma unroll
        for (int i = 0; i < S + 4; i++) f[i] = wv_nl(x[i], wv_mul(t.wt[i], eb0));
#pragma unroll
        for (int i = 1; i < S + 3; i++) 
          k1[i] = wv_rounded(k_term<R>(f[i], f[i + 1], f[i - 1], gk, cc));
#pragma unroll
        for (int i = 1; i < S + 3; i++)
          if (i <= S || i >= 3) f[i] = wv_nl(cadd(x[i], k1[i]), wv_mul(t.wt[i], eb1));
#pragma unroll
        for (int i = 2; i < S + 2; i++) {
          if (s0 + i - 2 >= W) break;
          if (!(isfinite((double)x[i].x) && isfinite((double)x[i].y))) bad = 1;
          const C a1 = cadd(x[i], k1[i]);
          // (the term of a column itself has the other rounding of exp(i th))
          const C fi = wv_nl(a1, wv_mulq(t.wt[i], eb1));
          const C k2 = k_term<R>(fi, f[i + 1], f[i - 1], gk, cc);
          C e = cadd(cadd(x[i], cscale(k1[i], R(0.5))), cscale(k2, R(0.5)));
          const double ex = (double)e.x - (double)a1.x, ey = (double)e.y - (double)a1.y;
          const double err = sqrt(ex * ex + ey * ey) /
                             (sqrt((double)e.x * (double)e.x + (double)e.y * (double)e.y) + 1.0);
          if (err > lmax) lmax = err;
          if (t.ab[i - 2] != R(1)) e = cscale(e, t.ab[i - 2]);
          X[wv_pad(((s0 + i - 2) << lg2) + r)] = e;
        }
      });
      double wmax = bad ? INFINITY : fmin(lmax, DBL_MAX);
#ifdef OFX_EMU
      red[0] = wmax;
      const int nred = 1;
#else
      const int nred = nw;
      wmax = wv_wave_max(wmax);
      if (nw > 1) red[wv] = wmax;
#endif
      meet();
      unsigned x1 = 0, tag1 = 0;
      double gmax = wmax;
      if (nw > 1 || OFX_NT == 1) {
        gmax = red[0];
        for (int w = 1; w < nred; w++) gmax = red_op(gmax, red[w], 0);
      }
      if (Cn > 1) {
        // the last wave publishes the member's error maximum
        x1 = ++sy.nx;
        tag1 = sy.base + x1;
        each([&](int tid, int, T&) {
          if (tid == NT - 1)
            wv_put<C>(WvAt{record_of(x1, rank), 1, 0u}, pack_d<R>(gmax), tag1);
        });
      }
      const bool early = Cn == 1;  // the decision needs no exchange
      auto decide = [&]() -> int {  // 0 accept, 1 reject, 2 leave
        attempts++;
        trip_att++;
        if (isinf(gmax)) {
          status = ST_NONFINITE;
          return 2;
        }
        if (100.0 * gmax > max_err && stepmod > 1.0) {
          stepmod -= 1.0;
          eb1 = expi(-(bdiffw0 * (k - 1.0 + stepmod) * hmin), R(0));
          return 1;  // A0 is untouched
        }
        return 0;
      };
      int dec = 0;
      if (early) {
        dec = decide();
        if (dec == 2) break;
        if (dec == 1) {
          meet();  // (red and X are written again)
          continue;
        }
      }
      columns_forward([&](int cl, int r) { return X[wv_pad((cl << lg2) + r)]; }, x1, tag1);
      rows_in(x1, tag1, true);
      fft<-1, true>(lg1, row_waves(), Tb);
      if (!early) {
        meet();
        if (sflag[1]) {
          status = ST_BARRIER_TIMEOUT;
          break;
        }
        gmax = red[32];
        dec = decide();
        if (dec == 2) break;
        if (dec == 1) continue;
      }
      // ---------------- accept ----------------
      const double pcterr = 100.0 * gmax;
      accepted++;
      trip_acc++;
      if (rank == 0 && stepmods)
        each([&](int tid, int, T&) {
          const int e = (int)k - 1;
          if (tid == (e & (NT - 1))) gl(stepmods)[e] = (float)stepmod;
        });
      const double s_used = stepmod;
      double ns = stepmod;
      if (pcterr < min_err) ns += 1.0;
      if (k < nsteps && (k + ns) > nsteps) ns = (double)nsteps - k;
      const double knew = k + ns;
      const double Gnext = gl(Gd)[((int)knew < nsteps ? (int)knew : nsteps) - 1];
      int cend = chunk;
      while ((double)cend <= nChunks && !(knew < cend * sel && knew <= nsteps)) cend++;
      // dispersion in the rows' registers; the phasors of an unchanged step
      // length are those of the last step
      if (s_used != s_held) {
        each([&](int, int w, T& t) {
          if (w >= row_waves()) return;
#pragma unroll
          for (int m = 0; m < 4; m++) {
            t.ph[m] = expi(-t.beta[m] * s_used, R(0));
            const R al = t.alpha[m];
            t.am[m] = al == R(1) ? R(1) : (al == R(0) ? R(0) : (R)pow(al, (R)s_used));
          }
        });
        s_held = s_used;
      }
      each([&](int, int w, T& t) {
        if (w >= row_waves()) return;
#pragma unroll
        for (int m = 0; m < 4; m++) 
          t.v[m] = wv_rounded(cscale(wv_mul(t.v[m], t.ph[m]), t.am[m]));
      });
      if (apft && cend > chunk)
        each([&](int, int w, T& t) {
          const int rl = w * (256 >> lg1) + t.qr;
          if (w >= row_waves() || rl >= Rr) return;
          OFX_GLOBAL C* ap = gl(apft);
          for (int c2 = chunk; c2 < cend; c2++)
            if (c2 - 1 < n_cols)
#pragma unroll
              for (int m = 0; m < 4; m++)
                stg(ap, (size_t)(c2 - 1) * n + (k20 + rl) + n2 * (t.jr + m * (n1 >> 2)), t.v[m]);
        });
      unsigned x2 = 0, tag2 = 0;
      if (Cn > 1) {
        x2 = ++sy.nx;
        tag2 = sy.base + x2;
      }
      rows_inverse(x2, tag2);
      // the next step's exp(-i bdwz) while t2 is in flight (both ends move on
      // by the step when its length is kept)
      k = knew;
      stepmod = ns;
      chunk = cend;
      eb0 = ns == s_used ? eb1 : expi(-(bdiffw0 * (k - 1.0) * hmin), R(0));
      eb1 = expi(-(bdiffw0 * (k - 1.0 + stepmod) * hmin), R(0));
      if (!columns_inverse(x2, tag2)) {
        status = ST_BARRIER_TIMEOUT;
        break;
      }
      Gk = uniform(Gnext);
    }
    if (status != ST_RUNNING) break;
    if (a.trips > 0 && rank == 0 && d.sm_hist && stepmods) {
      float* row = d.sm_hist + (size_t)((trip_base + trip) % d.hist_cap) * (size_t)nsteps;
      each([&](int tid, int, T&) {
        for (int j = tid; j < nsteps; j += NT) gl(row)[j] = gl(stepmods)[j];
      });
    }
    if (a.trips > 0 && rank == 0 && d.trip_log && trip_base + trip < d.trip_cap) {
      double* tl = d.trip_log + 4 * (size_t)(trip_base + trip);
      tl[2] = (double)trip_att;
      tl[3] = (double)trip_acc;
    }
    if (!cavity) continue;
    // ---------------- cavity: OC split, detuning, pump (one FFT pair) ----------------
    {
      const unsigned xc1 = ++sy.nx, tagc1 = sy.base + xc1;
      columns_forward([&](int cl, int r) { return A0[(HW + cl) * sT + r]; }, xc1, tagc1);
      rows_in(xc1, tagc1, false);
      if (sflag[1]) {
        status = ST_BARRIER_TIMEOUT;
        break;
      }
      fft<-1, true>(lg1, row_waves(), Tb);
      const C* pump = (const C*)d.pump;
      const C* cav = (const C*)d.cav;
      const C* ocm = (const C*)d.ocm;
      C* ocs = (C*)d.oc_spec;
      double* esd = d.esd_sum;
      double* xesd = d.xesd_sum;
      C* hist = d.hist ? (C*)d.hist + (size_t)((trip_base + trip) % d.hist_cap) * (size_t)n : nullptr;
      const bool have_prev = (trip_base + trip) > 0 && !(fresh && trip == 0);
      double acc[3] = {0.0, 0.0, 0.0};  // sum (S-Sp)^2, sum S^2, sum S
      each([&](int, int w, T& t) {
        const int rl = w * (256 >> lg1) + t.qr;
        if (w >= row_waves() || rl >= Rr) return;
#pragma unroll
        for (int m = 0; m < 4; m++) {
          const int kk = (k20 + rl) + n2 * (t.jr + m * (n1 >> 2));
          const C v = t.v[m];
          xesd[kk] += wv_abs2(v);
          if (hist) hist[kk] = v;
          const C o = wv_mulq(v, ocm[kk]);
          const double So = wv_abs2(o);
          if (have_prev) {
            const C op = ocs[kk];
            const double Sp = wv_abs2(op);
            acc[0] = wv_fma(So - Sp, So - Sp, acc[0]);
          }
          acc[1] = wv_fma(So, So, acc[1]);
          acc[2] += So;
          ocs[kk] = o;
          esd[kk] += So;
          const C mm = wv_mul(cav[kk], expi(-d.delay * dw_of(kk, n, dt), R(0)));
          t.v[m] = cadd(wv_mul(v, mm), pump ? pump[kk] : mkc<R>(R(0), R(0)));
        }
      });
      const unsigned xc2 = ++sy.nx, tagc2 = sy.base + xc2;
      const int par = (int)(xc2 & 1u);
      publish_slots<R>(cd, par, rank, 1, acc[0], acc[1], acc[2], tagc2);
      rows_inverse(xc2, tagc2);
      double tot[3];
      if (!columns_inverse(xc2, tagc2) ||
          !gather_sums<R>(cd, par, tagc2, tot, red, a.timeout_ticks)) {
        status = ST_BARRIER_TIMEOUT;
        break;
      }
      const double conv = have_prev ? (tot[1] > 0.0 ? sqrt(tot[0] / tot[1]) : 0.0) : INFINITY;
      if (rank == 0 && d.trip_log && trip_base + trip < d.trip_cap) {
        double* tl = d.trip_log + 4 * (size_t)(trip_base + trip);
        tl[0] = conv;
        tl[1] = tot[2];
      }
      meet();  // (red is written again)
      if (a.conv_tol > 0.0 && conv < a.conv_tol) {
        status = ST_CONVERGED;
        trip++;
        break;
      }
    }
  }
  if (status == ST_RUNNING) status = ST_DONE;
  // store own columns (after a barrier so no member still reads the input halo)
  if (status != ST_BARRIER_TIMEOUT) {
    sy.nreal++;
    if (!cluster_barrier(cd, sy.nreal * (unsigned)Cn, a.timeout_ticks, sflag))
      status = ST_BARRIER_TIMEOUT;
  }
  if (status != ST_BARRIER_TIMEOUT)
    each([&](int tid, int, T&) {
      for (int idx = tid; idx < W * n2; idx += NT) {
        const int lc = HW + (idx >> lg2), r = idx & (n2 - 1);
        field[(c0 - HW + lc + n1 * r) & (n - 1)] = A0[lc * sT + r];
      }
    });
  if (rank == 0 && OFX_TID == 0) {
    d.status[0] = status;
    if (a.trips > 0) {
      if (trip > 0) d.fresh[0] = 0;
      d.trips_done[0] += trip;
    }
    d.counters[0] += attempts;
    d.counters[1] += accepted;
  }
  meet();  // (the next instance writes A0)
}

template <typename R, int S, typename GEO, bool REFRESH>
OFX_DEV void wave_main(const LaunchArgs& a, int wg, cpx<R>* lds, double* red, int* sflag,
                       WvThread<R, S, GEO::HW>* thr) {
  const int ci = a.wg_cluster[wg];
  if (ci < 0) return;
  const ClusterDesc& cd = a.clusters[ci];
  const int rank = a.wg_rank[wg];
  SyncState sy;
  member_begin(a, cd, wg, rank, sflag, sy);
  for (int ii = 0; ii < cd.n_inst; ii++) {
    const int id = a.inst_order[cd.first_inst + ii];
    WvRun<R, S, GEO, REFRESH> run(a, cd, a.inst[id], sy, red, sflag, thr);
    run.run(rank, lds);
    if (flag_load(cd.abort_flag)) break;
  }
  member_end(cd, sy);
}

}  // namespace ofx
