// gemm_q8_square_fp8.hip -- the 256 x 256 tiles of the fp8 GEMM, e4m3fn or e5m2 weights.
#include "gemm_q8_kernel.hpp"

namespace psq {

int q8_square_fp8(int kind, int out, int act, const Q8Args &x)
{
    if (kind == Q8_E4M3) return launch_square<true>(out, act, x);
    using L = Lay<2, 4, 4>;   // e5m2 weights take no activation
    switch (out) {
    case OUT_BF16: return launch_layout<true, OUT_BF16, ACT_NONE, 1, L>(x);
    case OUT_F16: return launch_layout<true, OUT_F16, ACT_NONE, 1, L>(x);
    default: return launch_layout<true, OUT_F32, ACT_NONE, 1, L>(x);
    }
}

}  // namespace psq
