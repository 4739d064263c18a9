// rk_decode_think_f16.hip -- the F16 decode kernels over ThinK-pruned visual
// Keys and their launcher (declared in rk_decode.h).
#include "rk_decode_dev.h"

namespace rk {

hipError_t decode_launch_think_f16(int dkb, bool vec, int hmax, const DecodeArgs& a, dim3 grid, hipStream_t s) {
  return launch_sel_dk<F16>(dkb, vec, hmax, a, grid, s);
}

}  // namespace rk
