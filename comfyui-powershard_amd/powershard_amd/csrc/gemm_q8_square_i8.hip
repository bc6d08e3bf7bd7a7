// gemm_q8_square_i8.hip -- the 256 x 256 tiles of the int8 GEMM.
#include "gemm_q8_kernel.hpp"

namespace psq {

int q8_square_i8(int out, int act, const Q8Args &x) { return launch_square<false>(out, act, x); }

}  // namespace psq
