// The RK23 pass of the wave kernel (ofx_wave_impl.h): the Bogacki-Shampine
// 3(2) step and the step control of ofx_pass_impl.h's rk23_pass, with the same
// roundings.
//
// Bound: as for Heun, the latency of a step's dependent chain.  The general
// kernel runs a step in five LDS phases with a workgroup barrier each and three
// evaluations of the nonlinear term a point and stage, then exchanges.  Here a
// thread holds S own columns of one row and 4 neighbours on each side and
// forms K2, K3, the solution, K4 and the error quotient in registers: S + 6,
// S + 4 and S + 2 evaluations, no barrier.  K4 (the next step's K1) goes to
// the other of two LDS buffers; its three boundary columns on each side reach
// the neighbours with the attempt's exchange, read by waves that have no row
// to transform where there are any.  After a rejection K1 is formed again from
// the window's own samples.  One instance, us per adaptive step, FP32 (general
// kernel): 2^9 points 3.5 (8.8), 2^11 5.8 (10.0), 2^13 6.8 (11.3), 2^15 9.3
// (18.1); FP64 2^13 10.0 (14.7).  A pass of 8192 points: 28.8 -> 15.2 ms.
#pragma once
#include "ofx_wave_impl.h"

namespace ofx {

// The neighbours' K4 boundary columns of exchange x (kx, see rk23_pass) into
// the halo columns 1..3 and HW + W.. of dst.  The caller meets before it reads dst
// or sflag[1], which a poll that gave up sets.
template <typename R, int S, typename GEO, bool REFRESH>
OFX_DEV void WvRun<R, S, GEO, REFRESH>::boundary_in(unsigned x, unsigned tag, C* dst) {
  const int act = row_waves(), w0 = act < nw ? act : 0, stride = (nw - w0) * 64;
  const u64* kx = (const u64*)uniform(cd.kx) + (size_t)(x & 1u) * Cn * 6 * n2 * TT::NW;
  const int left = (rank + Cn - 1) & (Cn - 1), right = (rank + 1) & (Cn - 1);
  bool ok = true;
  each([&](int tid, int w, T&) {
    if (w < w0) return;
    Spin sp = spin();
    for (int base = tid - w0 * 64; base < 6 * n2 && ok; base += 4 * stride) {
      unsigned src[4];
      int to[4];
      unsigned mask = 0;
#pragma unroll
      for (int b = 0; b < 4; b++) {
        const int e = base + b * stride, col6 = e >> lg2, r = e & (n2 - 1);
        const int side = col6 >= 3 ? 1 : 0, col = col6 - 3 * side;
        // (columns across the wrap carry a row shift)
        int rr = r;
        if (side == 0 && c0 - 3 + col < 0) rr = (r - 1) & (n2 - 1);
        if (side == 1 && c0 + W + col >= n1) rr = (r + 1) & (n2 - 1);
        src[b] = (unsigned)(((side ? right * 2 : left * 2 + 1) * 3 + col) * n2 + rr);
        to[b] = (side ? HW + W + col : 1 + col) * sT + r;
        if (e < 6 * n2) mask |= 1u << b;
      }
      ok = wv_poll<C, 4>(
          mask, tag, [&](int b) { return WvAt{kx, (size_t)Cn * 6 * n2, src[b] * 8u}; },
          [&](int b, C v) { dst[to[b]] = v; }, sp);
    }
    if (!ok) sflag[1] = 1;
  });
}

template <typename R, int S, typename GEO, bool REFRESH>
OFX_DEV int WvRun<R, S, GEO, REFRESH>::rk23(R cc, long long& att, long long& acc, double& s_held) {
  const int Ns = uniform(d.nsteps), sel = (int)uniform(d.sel), nchunks = Ns / sel;
  const double A1c = 1.0 / 2.0, A2c = 3.0 / 4.0;
  const R a1 = (R)A1c, a2 = (R)A2c, a3 = (R)(4.0 / 9.0), a4 = (R)(1.0 / 3.0),
          a5 = (R)(2.0 / 9.0);
  const R b1 = (R)(1.0 / 8.0), b2 = (R)(1.0 / 3.0), b3 = (R)(1.0 / 4.0), b4 = (R)(7.0 / 24.0);
  const double* const Gd = uniform(d.G);
  const double bdw = uniform(d.bdiffw0), h = uniform(d.h);
  const double max_err = uniform(d.max_err), min_err = uniform(d.min_err);
  float* const stepmods = uniform(d.stepmods);
  C* const apft = uniform((C*)d.apft);
  const int n_cols = uniform(d.n_cols);
  u64* const kxb = (u64*)uniform(cd.kx);

  double k = 0.0, stepprev = 4.0, stepmod = 4.0, cend = sel;
  int chunk = 0, cur = 0;          // cur: the LDS buffer that holds K1
  bool k1_new = true;              // K1 is to be formed from A0 ...
  double k1_at = 0.0;              // ... at this z, with this g
  R k1_g = (R)(stepmod * h * gl(Gd)[0]);
  C e2, e3, e4;                    // exp(-i bdwz) of the stages
  R gk;
  bool more;
  // the next attempt's chunk, phasors and g
  auto next = [&] {
    while (chunk < nchunks && !(k < cend)) {
      chunk++;
      cend = (double)(chunk + 1) * (double)sel;
      stepmod = stepprev;
    }
    more = chunk < nchunks;
    const int g = (int)k < Ns ? (int)k : Ns - 1;
    gk = (R)(stepmod * h * gl(Gd)[g]);
    e2 = expi(-(bdw * (k + A1c * stepmod) * h), R(0));
    e3 = expi(-(bdw * (k + A2c * stepmod) * h), R(0));
    e4 = expi(-(bdw * (k + stepmod) * h), R(0));
  };
  next();
  while (more) {
    if ((int)k >= Ns) return ST_BAD_ARG;
    refresh();
    unsigned x1 = 0, tag1 = 0;
    if (Cn > 1) {
      x1 = ++sy.nx;
      tag1 = sy.base + x1;
    }
    C* const Kc = K1 + cur * (LC * sT);
    C* const Kn = K1 + (cur ^ 1) * (LC * sT);
    cur ^= 1;
    u64* const kx = kxb + (size_t)(x1 & 1u) * Cn * 6 * n2 * TT::NW;
    const C e1 = k1_new ? expi(-(bdw * k1_at * h), R(0)) : mkc<R>(R(1), R(0));
    // ---- all stages, the solution, the error quotient, absorber ----
    double lmax = -1.0;
    int bad = 0;
    each([&](int tid, int, T& t) {
      const int r = tid & (n2 - 1), s0 = (tid >> lg2) * S;
      if (s0 >= W) return;
      C x[S + 8], f[S + 8], k1[S + 8], k2[S + 8], e[S + 8];
#pragma unroll
      for (int i = 0; i < S + 8; i++) x[i] = A0[(s0 + i) * sT + r];
      if (k1_new) {
#pragma unroll
        for (int i = 0; i < S + 8; i++) f[i] = wv_nl(x[i], wv_mul(t.wt[i], e1));
#pragma unroll
        for (int i = 1; i < S + 7; i++) k1[i] = k_term<R>(f[i], f[i + 1], f[i - 1], k1_g, cc);
      } else {
#pragma unroll
        for (int i = 1; i < S + 7; i++) k1[i] = Kc[(s0 + i) * sT + r];
      }
#pragma unroll
      for (int i = 1; i < S + 7; i++)
        f[i] = wv_nl(cadd(x[i], cscale(k1[i], a1)), wv_mul(t.wt[i], e2));
#pragma unroll
      for (int i = 2; i < S + 6; i++) k2[i] = k_term<R>(f[i], f[i + 1], f[i - 1], gk, cc);
#pragma unroll
      for (int i = 2; i < S + 6; i++)
        f[i] = wv_nl(cadd(x[i], cscale(k2[i], a2)), wv_mul(t.wt[i], e3));
      C k3[S + 8];
#pragma unroll
      for (int i = 3; i < S + 5; i++) {
        k3[i] = k_term<R>(f[i], f[i + 1], f[i - 1], gk, cc);
        const C u = mkc<R>(wv_fma(k2[i].x, a4, k3[i].x * a3), wv_fma(k2[i].y, a4, k3[i].y * a3));
        e[i] = cadd(cadd(x[i], u), cscale(k1[i], a5));
      }
#pragma unroll
      for (int i = 3; i < S + 5; i++) f[i] = wv_nl(e[i], wv_mul(t.wt[i], e4));
#pragma unroll
      for (int i = 4; i < S + 4; i++) {
        const C k4 = k_term<R>(f[i], f[i + 1], f[i - 1], gk, cc);
        const C u = mkc<R>(wv_fma(k4.x, b1, k3[i].x * b2), wv_fma(k4.y, b1, k3[i].y * b2));
        const C as = cadd(cadd(cadd(x[i], u), cscale(k2[i], b3)), cscale(k1[i], b4));
        const double aE = sqrt(wv_abs2(e[i]));
        if (aE > 0.0) {
          const double dx = (double)as.x - (double)e[i].x, dy = (double)as.y - (double)e[i].y;
          const double q = 0.5 * sqrt(wv_fma(dy, dy, dx * dx)) / (aE + 1.0);
          if (q > lmax) lmax = q;
        }
        if (isnan((double)e[i].x) || isnan((double)e[i].y)) bad = 1;
        const int c = s0 + i - 4;  // own column
        Kn[(HW + c) * sT + r] = k4;
        if (Cn == 1) {
          // the wrapped copies carry a row shift
          if (c < 3) Kn[(HW + W + c) * sT + ((r - 1) & (n2 - 1))] = k4;
          if (c >= W - 3) Kn[(c - (W - HW)) * sT + ((r + 1) & (n2 - 1))] = k4;
        } else {
          const size_t ws = (size_t)Cn * 6 * n2;
          if (c < 3) wv_put<C>(WvAt{kx, ws, (unsigned)((rank * 6 + c) * n2 + r) * 8u}, k4, tag1);
          if (c >= W - 3)
            wv_put<C>(WvAt{kx, ws, (unsigned)((rank * 6 + 3 + c - (W - 3)) * n2 + r) * 8u}, k4,
                      tag1);
        }
        C v = e[i];
        if (t.ab[i - 4] != R(1)) v = cscale(v, t.ab[i - 4]);
        X[wv_pad((c << lg2) + r)] = v;
      }
    });
    k1_new = false;
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
    double gmax = wmax;
    if (nw > 1 || OFX_NT == 1) {
      gmax = red[0];
      for (int w = 1; w < nred; w++) gmax = red_op(gmax, red[w], 0);
    }
    if (Cn > 1)
      // the last wave publishes the member's error maximum
      each([&](int tid, int, T&) {
        if (tid == NT - 1) wv_put<C>(WvAt{record_of(x1, rank), 1, 0u}, pack_d<R>(gmax), tag1);
      });
    double pmax = 0.0;
    auto decide = [&]() -> int {  // 0 accept, 1 reject, 2 leave
      att++;
      if (isinf(gmax)) return 2;
      pmax = gmax < 0.0 ? -1.0 : 4.0 * 100.0 * gmax;
      if (!(pmax >= max_err && stepmod > 1.0 && (k - stepmod) > 0.0)) return 0;
      // back by the failed step, one minimal step smaller, K1 from A0
      k = k - stepmod;
      stepmod = stepmod - 1.0;
      stepprev = stepmod;
      k1_new = true;
      k1_at = k + stepmod;
      k1_g = (R)(stepmod * h * gl(Gd)[(int)k]);
      k = k + stepmod;
      next();
      return 1;
    };
    const bool early = Cn == 1;  // the decision needs no exchange
    if (early) {
      const int dec = decide();
      if (dec == 2) return ST_NONFINITE;
      if (dec == 1) {
        meet();  // (red, X and K1 are written again)
        continue;
      }
    }
    columns_forward([&](int cl, int r) { return X[wv_pad((cl << lg2) + r)]; }, x1, tag1);
    rows_in(x1, tag1, true);
    if (!early) boundary_in(x1, tag1, Kn);
    fft<-1, true>(lg1, row_waves(), Tb);
    if (!early) {
      meet();
      if (sflag[1]) return ST_BARRIER_TIMEOUT;
      gmax = red[32];
      const int dec = decide();
      if (dec == 2) return ST_NONFINITE;
      if (dec == 1) continue;
    }
    // ---------------- accept ----------------
    acc++;
    if (rank == 0 && stepmods && (int)k < Ns)
      each([&](int tid, int, T&) {
        const int e = (int)k;
        if (tid == (e & (NT - 1))) gl(stepmods)[e] = (float)stepmod;
      });
    const double s_used = stepmod;
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
      const int rl = w * (256 >> lg1) + t.qr;
      if (w >= row_waves()) return;
#pragma unroll
      for (int m = 0; m < 4; m++)
        t.v[m] = wv_rounded(cscale(wv_mul(t.v[m], t.ph[m]), t.am[m]));
      if (apft && chunk < n_cols && rl < Rr)
#pragma unroll
        for (int m = 0; m < 4; m++)
          stg(gl(apft), (size_t)chunk * n + (k20 + rl) + n2 * (t.jr + m * (n1 >> 2)), t.v[m]);
    });
    unsigned x2 = 0, tag2 = 0;
    if (Cn > 1) {
      x2 = ++sy.nx;
      tag2 = sy.base + x2;
    }
    rows_inverse(x2, tag2);
    // step control (rk23_pass's order) while t2 is in flight
    if (k + stepmod >= cend && k < cend - 1.0) {
      const double stepend = (cend - k) - 1.0;
      stepprev = stepmod;
      stepmod = stepend;
    } else {
      if (!(pmax >= max_err) && !(pmax >= min_err) && (k + stepmod + stepmod) < cend - 1.0)
        stepmod = stepmod * 2.0;
      stepprev = stepmod;
    }
    k = k + stepmod;
    next();
    if (!columns_inverse(x2, tag2)) return ST_BARRIER_TIMEOUT;
  }
  return ST_RUNNING;
}

}  // namespace ofx
