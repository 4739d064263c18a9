// rk_decode_think_bf16.hip -- the BF16 decode kernels over ThinK-pruned visual
// Keys and their launcher (declared in rk_decode.h).
#include "rk_decode_dev.h"

namespace rk {

hipError_t decode_launch_think_bf16(int dkb, bool vec, int hmax, const DecodeArgs& a, dim3 grid, hipStream_t s) {
  return launch_sel_dk<BF16>(dkb, vec, hmax, a, grid, s);
}

}  // namespace rk
