// The wide fibre kernels (ofx_gnlse_wide.h), in a file of their own: beside them
// the compiler shares code of the general kernel (ofx_gnlse.hip) that it inlines
// otherwise, which cost that one 3 to 4 % (FP32 fields, 2^8 to 2^12 points).
#include <hip/hip_runtime.h>
#include <math.h>

#include "../../include/optifax_hip.h"
#include "ofx_gnlse_impl.h"
#include "ofx_gnlse_wide.h"

namespace ofx {

// n = 2^LG points, n / 8 threads (ofx_gnlse_wide.h)
template <typename R, int LG>
__global__ void __launch_bounds__((1 << LG) / GW_P) gnlse_wide_kernel(GnlseArgs a) {
  extern __shared__ __align__(16) unsigned char gnlse_smem[];
  cpx<R>* buf = reinterpret_cast<cpx<R>*>(gnlse_smem);
  cpx<R>* tw = buf + gw_pad(1 << LG);
  __shared__ double red[16];
  GwThread<R> thr;
  GwRun<R, LG> run;
  run.thr = &thr;
  run.red = red;
  run.integrate(a, blockIdx.x, buf, tw);
}

const void* gnlse_wide_fn(int precision, int lg) {
  if (precision == OFX_F32) return (const void*)gnlse_wide_kernel<float, 13>;
  return lg == 11 ? (const void*)gnlse_wide_kernel<double, 11>
                  : (const void*)gnlse_wide_kernel<double, 12>;
}

}  // namespace ofx
