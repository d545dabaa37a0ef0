// The wave kernels (ofx_wave_impl.h) with a grid size's default geometry fixed
// at compile time (wave_geometry), 2^8 to 2^16 points in either precision.
// Scratch bytes a lane (addresses kept, see refresh()): FP32 2^10 16, 2^16 368; FP64
// 2^11 156, 2^13 256, 2^14 140, 2^15 296, 2^16 68; none at the other sizes.
#include <hip/hip_runtime.h>

#include "../../include/optifax_hip.h"
#include "ofx_backend.h"
#include "ofx_wave_impl.h"

namespace ofx {

template <typename R, int LG>
struct FixedGeometry {
  static constexpr WaveGeometry g = wave_geometry(LG, sizeof(R) == 8, false);
  static constexpr int share = (1 << LG) >> g.lgC, S = share > g.block ? share / g.block : 1;
  typedef WvGeoCt<LG, g.lgC, g.block> Geo;
};

template <typename R, int LG>
__global__ void __launch_bounds__((FixedGeometry<R, LG>::g.block)) wave_kernel_fixed(LaunchArgs a) {
  extern __shared__ __align__(16) unsigned char ofx_lds_raw[];
  __shared__ double red[64];
  __shared__ int sflag[4];
  typedef FixedGeometry<R, LG> F;
  WvThread<R, F::S> thr;
  wave_main<R, F::S, typename F::Geo, false>(a, (int)blockIdx.x,
                                             reinterpret_cast<cpx<R>*>(ofx_lds_raw), red, sflag,
                                             &thr);
}

template <typename R>
static const void* by_size(int lg) {
  switch (lg) {
    case 8: return (const void*)wave_kernel_fixed<R, 8>;
    case 9: return (const void*)wave_kernel_fixed<R, 9>;
    case 10: return (const void*)wave_kernel_fixed<R, 10>;
    case 11: return (const void*)wave_kernel_fixed<R, 11>;
    case 12: return (const void*)wave_kernel_fixed<R, 12>;
    case 13: return (const void*)wave_kernel_fixed<R, 13>;
    case 14: return (const void*)wave_kernel_fixed<R, 14>;
    case 15: return (const void*)wave_kernel_fixed<R, 15>;
    default: return (const void*)wave_kernel_fixed<R, 16>;
  }
}

const void* wave_fixed_fn(int precision, int lg) {
  return precision == OFX_F64 ? by_size<double>(lg) : by_size<float>(lg);
}

}  // namespace ofx
