// gemm_q8_width_i8.hip -- the 256 x 224 / 192 / 160 tiles of the int8 GEMM.
#include "gemm_q8_kernel.hpp"

namespace psq {

int q8_width_i8(int width, int out, int act, const Q8Args &x) { return launch_width<false, 0>(width, out, act, x); }

}  // namespace psq
