// gemm_q8.hpp -- what the translation units of the W8A8 / FP8 GEMM share.
#pragma once

#include "psq_common.hpp"

namespace psq {

// Epilogue operands and output of a W8A8 / FP8 GEMM.
struct Q8Epi {
    const float *a_scale;
    const float *w_scale;
    int w_per_row;
    const void *bias;
    int bias_dtype;
    void *y;
    int64_t ldy;
    int vec;          // rows of y are 16-byte aligned: 4-element vector stores allowed
};

// One checked call.
struct Q8Args {
    const uint8_t *a;
    int64_t lda;
    const uint8_t *w;
    int64_t ldw, M, N, K;
    Q8Epi ep;
    hipStream_t st;
    const char *name;
};

// Operand kinds: int8 x int8, e4m3 x e4m3, e4m3 activations x e5m2 weights.
enum { Q8_I8 = 0, Q8_E4M3 = 1, Q8_E5M2W = 2 };

// Output types of the tiles: enum psq_dtype, 3 = int32 (256 x 256 int8 tiles only), and the bf16 / f16
// outputs stored as fp32 (no activation; int8 and e4m3 weights).
enum { Q8_OUT_I32 = 3, Q8_WIDE_BF16 = 4, Q8_WIDE_F16 = 5 };

// Runs the problem on the small tiles (gemm_q8_small.hip) when they are the faster ones: true and its
// status, or false and nothing launched.
bool q8_small(int kind, int out, int act, const Q8Args &x, int &status);

// Quantizes one or two rows x itself (gemm_q8_vec.hip) where q8_vec_fits: a checked call whose operand
// `a` and row scales are not used.  wide: y is fp32.
bool q8_vec_fits(int64_t M, int64_t K, int act);
int q8_vec(int kind, const void *x, int x_dtype, int64_t ldx, int rotk, int wide, int act, const Q8Args &a);

// The large tiles: 256 x 256 (every output and activation of its kind), and 256 x width, width 224, 192
// or 160 (bf16 / f16 outputs, also stored as fp32; no gate).
int q8_square_i8(int out, int act, const Q8Args &x);
int q8_square_fp8(int kind, int out, int act, const Q8Args &x);
int q8_width_i8(int width, int out, int act, const Q8Args &x);
int q8_width_fp8(int kind, int width, int out, int act, const Q8Args &x);

// A bias word (the bias element zero-extended, or the fp32 bits) to fp32.
__device__ __forceinline__ float bias_word(uint32_t w, int dt)
{
    if (dt == PSQ_BF16) return __uint_as_float(w << 16);
    if (dt == PSQ_F16) return f16_to_f32(w);
    return __uint_as_float(w);
}

}  // namespace psq
