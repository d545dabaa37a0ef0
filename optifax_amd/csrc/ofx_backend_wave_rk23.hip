// The wave kernels' RK23 forms (ofx_wave_rk23.h): by precision and points a
// thread for any geometry, and with a grid size's default geometry fixed.
#include <hip/hip_runtime.h>

#include "../../include/optifax_hip.h"
#include "ofx_backend.h"
#include "ofx_wave_rk23.h"

namespace ofx {

template <typename R, int S, int MAXT>
__global__ void __launch_bounds__(MAXT) wave_rk23(LaunchArgs a) {
  extern __shared__ __align__(16) unsigned char ofx_lds_raw[];
  __shared__ double red[64];
  __shared__ int sflag[4];
  WvThread<R, S, 4> thr;
  wave_main<R, S, WvGeoRt<4>, sizeof(R) == 8 || (MAXT > 256)>(
      a, (int)blockIdx.x, reinterpret_cast<cpx<R>*>(ofx_lds_raw), red, sflag, &thr);
}

template <typename R, int MAXT>
static const void* by_points(int points) {
  return points == 4   ? (const void*)wave_rk23<R, 4, MAXT>
         : points == 2 ? (const void*)wave_rk23<R, 2, MAXT>
                       : (const void*)wave_rk23<R, 1, MAXT>;
}

const void* wave_rk23_fn(int precision, int points, bool wide) {
  if (precision == OFX_F64)
    return wide ? by_points<double, 512>(points) : by_points<double, 256>(points);
  return wide ? by_points<float, 512>(points) : by_points<float, 256>(points);
}

template <typename R, int LG>
struct FixedGeometry {
  static constexpr WaveGeometry g = wave_geometry(LG, sizeof(R) == 8, true);
  static constexpr int share = (1 << LG) >> g.lgC, S = share > g.block ? share / g.block : 1;
  typedef WvGeoCt<LG, g.lgC, g.block, 4> Geo;
};

template <typename R, int LG>
__global__ void __launch_bounds__((FixedGeometry<R, LG>::g.block)) wave_rk23_fixed(LaunchArgs a) {
  extern __shared__ __align__(16) unsigned char ofx_lds_raw[];
  __shared__ double red[64];
  __shared__ int sflag[4];
  typedef FixedGeometry<R, LG> F;
  // (512 threads form their addresses again each step: kept they spill, 2^15
  // points 12.1 against 9.3 us per step, and still use 152 to 356 bytes of scratch
  // a lane.  FP64 keeps them, with 68 to 536 bytes of scratch from 2^10 on; kept /
  // formed again: 2^8 4.0 / 4.2, 2^10 7.7 / 7.4, 2^11 9.0 / 8.6, 2^12 8.9 / 9.9, 2^13
  // 11.5 / 12.5, 2^14 17.4 / 16.2, 2^15 15.4 / 13.8)
  WvThread<R, F::S, 4> thr;
  wave_main<R, F::S, typename F::Geo, (F::g.block > 256)>(a, (int)blockIdx.x,
                                             reinterpret_cast<cpx<R>*>(ofx_lds_raw), red, sflag,
                                             &thr);
}

template <typename R>
static const void* by_size(int lg) {
  switch (lg) {
    case 8: return (const void*)wave_rk23_fixed<R, 8>;
    case 9: return (const void*)wave_rk23_fixed<R, 9>;
    case 10: return (const void*)wave_rk23_fixed<R, 10>;
    case 11: return (const void*)wave_rk23_fixed<R, 11>;
    case 12: return (const void*)wave_rk23_fixed<R, 12>;
    case 13: return (const void*)wave_rk23_fixed<R, 13>;
    case 14: return (const void*)wave_rk23_fixed<R, 14>;
    case 15: return (const void*)wave_rk23_fixed<R, 15>;
    default:   // (FP64 fields of 2^16 points do not fit LDS on 64 workgroups)
      if constexpr (sizeof(R) == 4) return (const void*)wave_rk23_fixed<R, 16>;
      return nullptr;
  }
}

const void* wave_rk23_fixed_fn(int precision, int lg) {
  return precision == OFX_F64 ? by_size<double>(lg) : by_size<float>(lg);
}

}  // namespace ofx
