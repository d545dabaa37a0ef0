// Internal types shared by the HIP kernels and the host runtime of libofx_hip.
// Not part of the public C ABI (include/optifax_hip.h is).
#pragma once
#ifndef OFX_EMU
#include <hip/hip_runtime.h>
#endif
#include <stdint.h>

namespace ofx {

// Method codes (match OFX_METHOD_* in optifax_hip.h).
enum { METHOD_HEUN = 0, METHOD_RK23 = 1 };

// Instance status codes written by the kernel (match OFX_STATUS_* values).
enum {
  ST_RUNNING = 0,
  ST_DONE = 1,
  ST_CONVERGED = 2,
  ST_NONFINITE = 3,
  ST_BARRIER_TIMEOUT = 4,
  ST_BAD_ARG = 5,
};

// Default geometry of the wave kernel (ofx_wave_impl.h) on a grid of 2^lg
// points, lg <= 16: log2 of the workgroups an instance and the threads of each.
// For lg >= WAVE_FIXED_LG a kernel with this geometry fixed exists; smaller
// grids are not used in earnest.  us per adaptive step, FP32 / FP64, of one
// instance by workgroups (each with its best thread count, all with the
// geometry fixed); the general kernel at its best geometry after the colon:
//   2^8   1 workgroup 2.6 / 3.0, 4: 4.3 / 6.0
//   2^9   1: 3.4 / 4.0, 8: 4.8 / 6.8                      : 7.9 / 8.9
//   2^10  1: 4.1 / 6.0, 8: 4.9 / 6.8, 32: 5.3 / 7.9       : 8.7 / -
//   2^11  8: 5.1 / 8.0, 16: 4.7 / 7.2, 32: 5.1 / 7.1      : 9.0 / 10.6
//   2^12  16: 5.3 / 7.5, 32: 5.9 / 8.3                    : 10.2 / 11.7
//   2^13  16: 6.8 / 10.7, 32: 6.2 / 9.9, 64: 7.3 / 11.3   : 11.0 / 12.8
//   2^14  32: 8.1 / 12.6, 64: 7.2 / 9.9, 128: 7.3 / 10.5  : 12.2 / 14.5
//   2^15  64: 8.1 / 11.9, 128: 8.0 / 11.1                 : 12.7 / 16.1
//   2^16  64: 12.2 / 17.3, 128: 10.2 / 15.5               : 15.4 / -
// Threads: 4 transform elements each where that leaves the stages at most 2
// points a thread (2^12 FP32 at 16 workgroups: 128 threads 6.3, 256 5.3; 2^15
// at 128: 128 threads 9.9, 256 8.0, 512 10.2).
// RK23 (a member owns 4 columns or more; FP64 2^16 does not fit LDS):
//   2^8   1: 2.9 / 3.4, 2: 6.2 / 7.8                      : 8.1 / 9.5
//   2^9   1: 3.5 / 4.3, 4: 6.5 / 8.1                      : 8.8 / 10.5
//   2^10  1: 4.5 / 6.4, 4: 6.2 / 7.8, 8: 7.0 / 8.9        : 9.5 / 11.0
//   2^11  8: 5.8 / 8.1, 16: 7.2 / 10.2                    : 10.0 / 11.7
//   2^12  8: 8.4 / 11.1, 16: 6.7 / 8.3                    : 11.4 / 13.1
//   2^13  16: 8.1 / 12.0, 32: 6.8 / 10.0                  : 11.3 / 14.7
//   2^14  16: 11.8 / -, 32: 10.0 / 17.1                   : 16.1 / 20.0
//   2^15  32: 14.9 / -, 64: 9.3 / 16.7                    : 18.1 / 22.4
//   2^16  64: 13.4 / -                                    : 23.6 / -
// (FP32 2^14 at 32 workgroups: 256 threads 11.7, 512 10.0; FP64's 512-thread
// form spills.)
enum { WAVE_FIXED_LG = 8 };
struct WaveGeometry {
  int lgC, block;
};
constexpr WaveGeometry wave_geometry(int lg, bool f64, bool rk23) {
  if (rk23)
    return lg <= 10   ? WaveGeometry{0, lg < 6 ? 64 : lg < 8 ? 1 << lg : 256}
           : lg <= 13 ? WaveGeometry{lg == 11 ? 3 : lg - 8, 256}
                      : WaveGeometry{lg == 14 ? 5 : 6, f64 ? 256 : 512};
  return lg <= 10   ? WaveGeometry{0, lg < 6 ? 64 : lg < 8 ? 1 << lg : lg < 10 || f64 ? 256 : 512}
         : lg == 11 ? WaveGeometry{4, 128}
         : lg == 12 ? WaveGeometry{4, 256}
         : lg <= 14 ? WaveGeometry{lg - 8, 256}
                    : WaveGeometry{7, lg == 16 && !f64 ? 512 : 256};
}

// Everything one instance needs on the device.  One array entry per instance,
// uploaded once per run; pointers are device pointers.
struct InstDesc {
  // grid: N = n1 * n2 points, time index j = c + n1 * r (c column, r row)
  int n, n1, n2, lg1, lg2;
  int nsteps;      // NSteps (number of minimal steps h)
  int n_cols;      // ApFT columns written (0 = none)
  int method;      // METHOD_HEUN or METHOD_RK23
  double w0;       // reference angular frequency [rad/s]
  double bdiffw0;  // beta0 - beta1*w0 [1/m]
  double h;        // minimal step [m]
  double dt;       // time step [s]
  double max_err;  // percent
  double min_err;  // percent
  double sel;      // steps per ApFT chunk
  double delay;    // cavity detuning [s] (round-trip mode)
  // read-only tables (FFT order)
  const double* beta;   // N: per-minimal-step phase phi_rel/L*h
  const double* alpha;  // N: T^(1/NSteps)
  const double* G;      // nsteps: poling-signed coupling
  const void* wt;       // N complex: exp(i*w0*t_j), phase reduced in FP64 (fftshifted time)
  const void* absorb;   // N real: absorbing-boundary factor of t_j (1 outside the zone)
  // in/out
  void* field;          // N complex: fftshifted time field (crystal input / output)
  void* apft;           // n_cols*N complex or null
  float* stepmods;      // nsteps or null
  // round-trip mode (all null in single-pass mode)
  const void* pump;     // N complex: pump spectrum in the crystal (FFT order)
  const void* cav;      // N complex: crystal output -> next crystal input transfer
  const void* ocm;      // N complex: crystal output -> output-coupled spectrum
  void* oc_spec;        // N complex: last output-coupled spectrum (in/out)
  double* esd_sum;      // N: sum over trips of |output-coupled spectrum|^2 (FFT order)
  double* xesd_sum;     // N: sum over trips of |crystal-output spectrum|^2 (FFT order)
  void* hist;           // [hist_cap][N] complex: crystal-output spectra of recent trips, or null
  float* sm_hist;       // [hist_cap][nsteps]: step multipliers of those trips (0 = not accepted)
  int hist_cap;         // trips held; trip t (cumulative, 0-based) sits in slot t % hist_cap
  int pad2;
  double* trip_log;     // [trip_cap][4]: conv metric, oc energy, attempts, accepted
  int trip_cap;
  int pad1;
  int* status;          // ST_* per instance
  int* trips_done;      // per instance, cumulative (also the trip-log base)
  int* fresh;           // per instance: 1 after a field rewrite (no previous spectrum yet)
  long long* counters;  // [0] attempts, [1] accepted (cumulative over the launch)
};

// One cluster = C workgroups cooperating on one instance at a time.
struct ClusterDesc {
  int C;           // workgroups in this cluster
  int first_inst;  // offset into the instance-order list
  int n_inst;      // instances processed in sequence
  int halo;        // halo columns each side
  // Exchange buffers hold tagged elements: every 32-bit word of a complex
  // sample as one 64-bit word (word | tag << 32), two parity halves each.
  void* t1;          // [2][N] tagged complex: forward transpose, N of the cluster
  void* t2;          // [2][N] tagged complex: inverse transpose
  void* slots;       // [2][C][8 waves][4] tagged complex-sized records (doubles)
  unsigned* bar;     // counter barrier (zeroed before every launch)
  int* abort_flag;   // set when a member gives up waiting
  int* xcc;          // C ints: hardware XCC id of each member (placement diagnostic)
  void* kx;          // RK23 only: [2][C][2 sides][3 columns][n2] tagged complex, K4 boundary
  unsigned* epoch;   // [0] tag base of this launch, [1] largest exchange count used by it
};

struct LaunchArgs {
  const InstDesc* inst;
  const ClusterDesc* clusters;
  const int* inst_order;   // instance indices, grouped per cluster
  const int* wg_cluster;   // per workgroup: cluster index or -1 (idle slot)
  const int* wg_rank;      // per workgroup: rank within its cluster
  const void* twiddle;     // NMAX complex: exp(-2 pi i m / NMAX)
  int nmax;                // twiddle table size (largest N in the launch)
  int trips;               // 0: single pass (MEX mode); >0: round trips
  double conv_tol;         // stop an instance when conv metric < tol (<=0 never)
  unsigned long long timeout_ticks;  // barrier spin limit in wall-clock ticks
  int* xcc_ids;            // optional: per workgroup hardware XCC id (diagnostic)
  int block;               // threads per workgroup
};

}  // namespace ofx
