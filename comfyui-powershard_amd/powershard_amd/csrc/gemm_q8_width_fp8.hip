// gemm_q8_width_fp8.hip -- the 256 x 224 / 192 / 160 tiles of the fp8 GEMM.
#include "gemm_q8_kernel.hpp"

namespace psq {

int q8_width_fp8(int kind, int width, int out, int act, const Q8Args &x)
{
    return kind == Q8_E4M3 ? launch_width<true, 0>(width, out, act, x) : launch_width<true, 1>(width, out, act, x);
}

}  // namespace psq
