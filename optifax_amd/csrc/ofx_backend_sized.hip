// The general pass kernel for Heun instances at a counter barrier, 512 threads,
// with the splits of 2^12 to 2^16 points fixed at compile time (SIZED in
// ofx_pass_impl.h) and both nonlinear stages in one pass.
//
// It runs where the shares are large (2048 to 4096 points a workgroup, the device
// full) and is bound by instruction issue with two waves a SIMD (LDS holds one
// workgroup a CU).  32 cavities of 2^14 to 2^16 points, one round trip: 87.8 ms
// with the geometry read at run time, 82.7 fixed, 76.9 with the stages in one
// pass.  1024 threads have 128 registers each and spill more: 83.2 (against 82.7).
// The six inlined bodies share one allocation of 256 registers and spill: FP32 103
// vector and 689 scalar registers (400 bytes of scratch a lane), FP64 324 and 1153
// (604 bytes); how much time that takes has not been measured.
#define OFX_NT 512
#define OFX_SIZED
#include <hip/hip_runtime.h>

#include "../../include/optifax_hip.h"
#include "ofx_backend.h"
#include "ofx_pass_impl.h"

namespace ofx {

static_assert(OFX_NT == XMODE_SIZED_BLOCK, "the launch has this many threads");

template <typename R>
__global__ void __launch_bounds__(OFX_NT) pass_kernel_sized(LaunchArgs a) {
  extern __shared__ __align__(16) unsigned char ofx_lds_raw[];
  __shared__ double red[64];
  __shared__ int sflag[4];
  cluster_main<R, XM_BARRIER, true>(a, (int)blockIdx.x, reinterpret_cast<cpx<R>*>(ofx_lds_raw), red,
                                    sflag);
}

const void* sized_kernel(int precision) {
  return precision == OFX_F64 ? (const void*)pass_kernel_sized<double>
                              : (const void*)pass_kernel_sized<float>;
}

}  // namespace ofx
