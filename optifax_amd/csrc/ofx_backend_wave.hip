// The wave kernels (ofx_wave_impl.h): the Heun pass and round trip with small
// shares per workgroup, by precision and points a thread, for any geometry
// (default geometries: ofx_backend_wave_fixed.hip).
#include <hip/hip_runtime.h>

#include "../../include/optifax_hip.h"
#include "ofx_backend.h"
#include "ofx_wave_impl.h"

namespace ofx {

// MAXT: workgroups of up to 256 threads have 512 registers a lane (half of them
// accumulation registers), which hold a lane's twiddles, factors and phasors
// without scratch memory, in FP64 with the addresses formed again each step.  With
// 512 threads 256, and part of them spills: FP32 132 to 168 bytes of scratch a
// lane, FP64 888 to 968 (by default only FP32 fields have 512 threads).
template <typename R, int S, int MAXT>
__global__ void __launch_bounds__(MAXT) wave_kernel(LaunchArgs a) {
  extern __shared__ __align__(16) unsigned char ofx_lds_raw[];
  __shared__ double red[64];
  __shared__ int sflag[4];
  WvThread<R, S> thr;
  wave_main<R, S, WvGeoRt<>, sizeof(R) == 8 || (MAXT > 256)>(
      a, (int)blockIdx.x, reinterpret_cast<cpx<R>*>(ofx_lds_raw), red, sflag, &thr);
}

template <typename R, int MAXT>
static const void* by_points(int points) {
  return points == 4   ? (const void*)wave_kernel<R, 4, MAXT>
         : points == 2 ? (const void*)wave_kernel<R, 2, MAXT>
                       : (const void*)wave_kernel<R, 1, MAXT>;
}

const void* wave_kernel_fn(int precision, int points, bool wide) {
  if (precision == OFX_F64)
    return wide ? by_points<double, 512>(points) : by_points<double, 256>(points);
  return wide ? by_points<float, 512>(points) : by_points<float, 256>(points);
}

}  // namespace ofx
