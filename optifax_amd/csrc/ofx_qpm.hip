// QPM gain maps on gfx950: the two sums behind the reference's GPU phase-
// matching analysis.
//
// 1. qpmgain.m:140-149 evaluates, for every (signal, pump) pair o of the map,
//        As[o] = g[o] * sum_k P(z_k) dz_k exp(i dk[o] z_k)
//    over the crystal's sampled poling P (about 10^6 samples per metre) as a
//    3-D gpuArray [signals x pumps x z] summed over z.  Here the z axis
//    arrives as runs: r = (z0, len, weight) stands for `len` samples z0, z0 + dz, ..., with one weight (the poling sign
//    times the sample spacing).  A run's sum is a geometric series,
//        sum_q exp(i dk (z0 + q dz)) = exp(i (dk z0 + th (len-1)/2))
//                                      sin(len th / 2) / sin(th / 2),
//    th = dk dz reduced to (-pi, pi], so a grating of constant domains costs
//    two sines per domain instead of one complex exponential per sample.
//    Runs of one sample give the literal sum for any z.  Few outputs are
//    shared out further, each summed by 4 or 16 threads.  Phases are formed
//    and reduced mod 2 pi in FP64; everything is FP64.
//
// 2. sincgain.m / sincgain_sparse.m:55-70 evaluate the narrowband mismatch
//    factor gain[g][o] = sum_j (sinc((dk0[o] - m_j kc[g]) L / 2) / m_j)^2 over
//    grating periods g and QPM orders m_j, with MATLAB's normalized sinc
//    sin(pi x)/(pi x).  One thread per (o, g), the argument reduced in FP64.
//
// Both maps are independent per output; the z runs are staged through LDS in
// chunks shared by the workgroup.
#include <hip/hip_runtime.h>
#include <math.h>
#include <stdio.h>
#include <string.h>

#include <algorithm>

#include "../../include/optifax_hip.h"

namespace ofxq {

constexpr int ZS_THREADS = 256;
constexpr int ZS_CHUNK = 512;  // runs staged in LDS at a time (24 KB)

__device__ __forceinline__ double reduce_2pi(double x) {
  // x - 2 pi round(x / 2 pi), two-term (Cody-Waite) split of 2 pi; the fma
  // makes q * TWO_PI_HI exact for |q| < 2^26
  const double TWO_PI_HI = 6.283185307179586232;
  const double TWO_PI_LO = 2.4492935982947064e-16;
  const double q = rint(x * 0.15915494309189533577);
  return fma(-q, TWO_PI_LO, fma(-q, TWO_PI_HI, x));
}

// sin x and cos x: x reduced to r in [-pi/4, pi/4] with its quadrant (the
// two-part pi / 2 of Cody & Waite; the fma keeps q * hi exact), then the
// Taylor polynomials of sin r (to r^17) and cos r (to r^16), whose truncation
// is below 2^-53 of the result.  Half the instructions of the general sincos,
// which brings arguments of any size and so reduces a second time.
__device__ __forceinline__ void sincos_cw(double x, double& s, double& c) {
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
  s = (k & 2) ? -a : a;
  c = (k == 1 || k == 2) ? -b : b;
}

// 256 threads: 256 / PARTS outputs, each summed in PARTS shares of the runs
// that meet in LDS in share order.  Bound by FP64 instruction issue (a sincos
// per output and run, and a sine where the run length changes); one share per
// output left a SIMD with at most one or two waves, too few to cover the
// polynomials' dependent chains.  Device time of a map before (general sincos,
// a division a run, one share) and now: 120000 outputs x 802 chirped runs 0.515
// -> 0.312 ms, uniform 0.367 -> 0.223; 2000 x 401 0.157 -> 0.014.  The error
// against the literal sum is unchanged (9.4e-14 there).
template <int PARTS>
__global__ void __launch_bounds__(ZS_THREADS)
zsum_kernel(int n_out, const double* __restrict__ dk, int n_run, const double* __restrict__ z0,
            const int* __restrict__ len, const double* __restrict__ wgt, double dz,
            double* __restrict__ out) {
  constexpr int OUTS = ZS_THREADS / PARTS;
  __shared__ double s_z0[ZS_CHUNK];
  __shared__ double s_w[ZS_CHUNK];
  __shared__ double s_m[ZS_CHUNK];
  const int part = threadIdx.x / OUTS;
  const int o = blockIdx.x * OUTS + threadIdx.x % OUTS;
  const double k = o < n_out ? dk[o] : 0.0;
  // per output: the reduced step phase and the series' denominator, by which
  // the whole sum is divided at the end (a run of one sample adds it as it is)
  const double th = reduce_2pi(k * dz);
  double s_half, c_half;
  sincos_cw(0.5 * th, s_half, c_half);
  // Below 1e-18 the series factor of a run of m < 2^31 samples is m to
  // rounding; formed with that sine, terms of very small dk would underflow.
  if (fabs(s_half) < 1e-18) s_half = 0.0;
  double ar = 0.0, ai = 0.0;
  // the series factor depends on the run length only: kept while consecutive
  // runs share it (a uniform grating has one or two lengths)
  double m_prev = 1.0, d_prev = s_half == 0.0 ? 1.0 : s_half;
  for (int base = 0; base < n_run; base += ZS_CHUNK) {
    const int cnt = min(ZS_CHUNK, n_run - base);
    __syncthreads();
    for (int i = threadIdx.x; i < cnt; i += ZS_THREADS) {
      s_z0[i] = z0[base + i];
      s_w[i] = wgt[base + i];
      s_m[i] = (double)len[base + i];
    }
    __syncthreads();
    const int end = cnt * (part + 1) / PARTS;
    for (int i = cnt * part / PARTS; i < end; i++) {
      const double m = s_m[i];   // the same for every thread of the share
      if (m != m_prev) {
        double c_m;
        if (s_half == 0.0)
          d_prev = m;  // every sample of the run has the same phase
        else if (m == 1.0)
          d_prev = s_half;
        else
          sincos_cw(0.5 * m * th, d_prev, c_m);
        m_prev = m;
      }
      double s, c;
      sincos_cw(fma(k, s_z0[i], 0.5 * (m - 1.0) * th), s, c);
      const double a = s_w[i] * d_prev;
      ar = fma(a, c, ar);
      ai = fma(a, s, ai);
    }
  }
  if (PARTS > 1) {
    // (the staging arrays hold 512 values each: 256 of either sum)
    __syncthreads();
    s_z0[threadIdx.x] = ar;
    s_w[threadIdx.x] = ai;
    __syncthreads();
    if (part) return;
    for (int p = 1; p < PARTS; p++) {
      ar += s_z0[p * OUTS + threadIdx.x];
      ai += s_w[p * OUTS + threadIdx.x];
    }
  }
  if (o < n_out) {
    const double d = s_half == 0.0 ? 1.0 : s_half;
    out[2 * (size_t)o] = ar / d;
    out[2 * (size_t)o + 1] = ai / d;
  }
}

template <int PARTS>
static void launch_zsum(int n_out, const double* dk, int n_run, const double* z0, const int* len,
                        const double* wgt, double dz, double* out) {
  const int outs = ZS_THREADS / PARTS;
  hipLaunchKernelGGL(zsum_kernel<PARTS>, dim3((n_out + outs - 1) / outs), dim3(ZS_THREADS), 0, 0,
                     n_out, dk, n_run, z0, len, wgt, dz, out);
}

__global__ void sinc_gain_kernel(int n_out, const double* __restrict__ dk0, int n_g,
                                 const double* __restrict__ kc, int n_m,
                                 const double* __restrict__ m, double half_len,
                                 double* __restrict__ gain) {
  const size_t idx = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (idx >= (size_t)n_out * (size_t)n_g) return;
  const int o = (int)(idx % (size_t)n_out);
  const int g = (int)(idx / (size_t)n_out);
  const double PI = 3.141592653589793116;
  double acc = 0.0;
  for (int j = 0; j < n_m; j++) {
    const double x = (dk0[o] - m[j] * kc[g]) * half_len;  // sinc argument
    double v;
    if (x == 0.0) {
      v = 1.0;
    } else {
      // sin(pi x) with pi x reduced mod 2 pi in FP64
      v = sin(reduce_2pi(PI * x)) / (PI * x);
    }
    v /= m[j];
    acc = fma(v, v, acc);
  }
  gain[idx] = acc;
}

struct Buf {
  void* p = nullptr;
  ~Buf() {
    if (p) hipFree(p);
  }
};

static int hip_ok(hipError_t e) { return e == hipSuccess ? OFX_OK : OFX_E_HIP; }

template <typename T>
static int up(Buf& b, const T* src, size_t n) {
  if (hipMalloc(&b.p, std::max<size_t>(n, 1) * sizeof(T)) != hipSuccess) return OFX_E_NOMEM;
  if (n) return hip_ok(hipMemcpy(b.p, src, n * sizeof(T), hipMemcpyHostToDevice));
  return OFX_OK;
}

}  // namespace ofxq

using namespace ofxq;

extern "C" int ofx_qpm_zsum(int device, int n_out, const double* dk, int n_run, const double* z0,
                            const int* len, const double* wgt, double dz, double* out,
                            double* ms) {
  if (n_out < 0 || n_run < 0 || !(dz > 0.0) || (n_out && (!dk || !out)) ||
      (n_run && (!z0 || !len || !wgt)))
    return OFX_E_ARG;
  for (int r = 0; r < n_run; r++)
    if (len[r] < 1) return OFX_E_ARG;
  if (n_out == 0) return OFX_OK;
  if (hipSetDevice(device) != hipSuccess) return OFX_E_NODEVICE;
  Buf b_dk, b_z, b_l, b_w, b_o;
  int st = up(b_dk, dk, (size_t)n_out);
  if (!st) st = up(b_z, z0, (size_t)n_run);
  if (!st) st = up(b_l, len, (size_t)n_run);
  if (!st) st = up(b_w, wgt, (size_t)n_run);
  if (!st && hipMalloc(&b_o.p, 16 * (size_t)n_out) != hipSuccess) st = OFX_E_NOMEM;
  if (st) return st;
  hipEvent_t e0, e1;
  hipEventCreate(&e0);
  hipEventCreate(&e1);
  hipEventRecord(e0, 0);
  // Shares per output: 16 while that is at most 8 waves on each of the device's
  // 1024 SIMDs, 4 up to 32 waves, then 1 (8 and more).  Device us of 802 runs on
  // either side of the lines: 2^15 - 1 outputs 66 (16 shares), 2^15 74 (4); 2^19 - 1
  // 890 (4), 2^19 917 (1).  The first line could lie higher (45000 outputs 99 with 4
  // shares, 91 at the rate of 16).  Maps of few runs gain nothing from shares: 2^19
  // outputs x 1 run 17 with 4 shares, 10 with 1, of a 1 ms call.  30000 outputs x 602
  // runs: 80 with 16 shares, 260 before.
  (n_out < (1 << 15)   ? launch_zsum<16>
   : n_out < (1 << 19) ? launch_zsum<4>
                       : launch_zsum<1>)(n_out, (const double*)b_dk.p, n_run,
                                         (const double*)b_z.p, (const int*)b_l.p,
                                         (const double*)b_w.p, dz, (double*)b_o.p);
  st = hip_ok(hipGetLastError());
  hipEventRecord(e1, 0);
  if (!st) st = hip_ok(hipMemcpy(out, b_o.p, 16 * (size_t)n_out, hipMemcpyDeviceToHost));
  if (!st && ms) {
    float f = 0.f;
    hipEventElapsedTime(&f, e0, e1);
    *ms = f;
  }
  hipEventDestroy(e0);
  hipEventDestroy(e1);
  return st;
}

extern "C" int ofx_sinc_gain(int device, int n_out, const double* dk0, int n_g, const double* kc,
                             int n_m, const double* m, double length, double* gain, double* ms) {
  if (n_out < 0 || n_g < 0 || n_m < 1 || !m || (n_out && (!dk0 || !gain)) || (n_g && !kc))
    return OFX_E_ARG;
  for (int j = 0; j < n_m; j++)
    if (!(m[j] != 0.0)) return OFX_E_ARG;
  const size_t tot = (size_t)n_out * (size_t)n_g;
  if (tot == 0) return OFX_OK;
  if (hipSetDevice(device) != hipSuccess) return OFX_E_NODEVICE;
  Buf b_dk, b_kc, b_m, b_g;
  int st = up(b_dk, dk0, (size_t)n_out);
  if (!st) st = up(b_kc, kc, (size_t)n_g);
  if (!st) st = up(b_m, m, (size_t)n_m);
  if (!st && hipMalloc(&b_g.p, 8 * tot) != hipSuccess) st = OFX_E_NOMEM;
  if (st) return st;
  hipEvent_t e0, e1;
  hipEventCreate(&e0);
  hipEventCreate(&e1);
  hipEventRecord(e0, 0);
  const size_t blocks = (tot + 255) / 256;
  hipLaunchKernelGGL(sinc_gain_kernel, dim3((unsigned)blocks), dim3(256), 0, 0, n_out,
                     (const double*)b_dk.p, n_g, (const double*)b_kc.p, n_m, (const double*)b_m.p,
                     0.5 * length, (double*)b_g.p);
  st = hip_ok(hipGetLastError());
  hipEventRecord(e1, 0);
  if (!st) st = hip_ok(hipMemcpy(gain, b_g.p, 8 * tot, hipMemcpyDeviceToHost));
  if (!st && ms) {
    float f = 0.f;
    hipEventElapsedTime(&f, e0, e1);
    *ms = f;
  }
  hipEventDestroy(e0);
  hipEventDestroy(e1);
  return st;
}
