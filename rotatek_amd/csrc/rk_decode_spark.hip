// rk_decode_spark.hip -- the decode kernels over SparK-pruned visual Keys
// (both 16-bit types) and their launcher (declared in rk_decode.h).
#include "rk_decode_dev.h"

namespace rk {

template <class TT, int KB, int HMAX>
hipError_t launch_spark(const DecodeArgs& a, dim3 grid, hipStream_t s) {
  if (a.fused)
    hipLaunchKernelGGL((decode_kernel<TT, KB, true, HMAX, true, false, false, true, true>), grid, dim3(kThreads), 0,
                       s, a);
  else
    hipLaunchKernelGGL((decode_kernel<TT, KB, true, HMAX, true, false, false, false, true>), grid, dim3(kThreads), 0,
                       s, a);
  const hipError_t e = hipGetLastError();
  if (e != hipSuccess || a.fused) return e;
  hipLaunchKernelGGL((merge_kernel<TT>), dim3(merge_grid(a)), dim3(kThreads), 0, s, a);
  return hipGetLastError();
}

template <class TT>
hipError_t launch_spark_any(int kb, int hmax, const DecodeArgs& a, dim3 grid, hipStream_t s) {
  if (kb == 1) return hmax > 1 ? launch_spark<TT, 1, 16>(a, grid, s) : launch_spark<TT, 1, 1>(a, grid, s);
  if (kb == 2) return hmax > 1 ? launch_spark<TT, 2, 16>(a, grid, s) : launch_spark<TT, 2, 1>(a, grid, s);
  return hipErrorInvalidValue;
}

hipError_t decode_launch_spark(int dtype, int kb, int hmax, const DecodeArgs& a, dim3 grid, hipStream_t s) {
  return dtype == RK_F16 ? launch_spark_any<F16>(kb, hmax, a, grid, s) : launch_spark_any<BF16>(kb, hmax, a, grid, s);
}

}  // namespace rk
