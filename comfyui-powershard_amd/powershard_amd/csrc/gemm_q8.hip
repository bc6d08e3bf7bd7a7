// gemm_q8.hip -- entry points of the W8A8 int8 and fp8 GEMMs: argument checks and the choice of tiles.
// The kernels: gemm_q8_kernel.hpp (large tiles), gemm_q8_small.hip (small tiles, split K).
#include "gemm_q8.hpp"
#include "quantize.hpp"

namespace psq {
namespace {

// Vector stores need 16-byte-aligned rows; the staged stores also address a 32-row block with a
// 32-bit lane offset, which holds for rows below 2^27 bytes.  Other outputs take the element-store path.
int vec_ok(const void *y, int64_t ldy, int elem)
{
    return (((uintptr_t)y & 15) == 0 && (ldy * elem) % 16 == 0 && ldy * elem < (1LL << 27)) ? 1 : 0;
}

int check_shapes(const char *name, const void *a, int64_t lda, const void *w, int64_t ldw, int64_t M, int64_t N,
                 int64_t K)
{
    if (M < 0 || N < 0 || K < 0) return set_error(PSQ_E_ARG, "%s: negative size", name);
    // an empty problem reads nothing: empty tensors may come with null data pointers
    if (M > 0 && N > 0 && (!a || !w)) return set_error(PSQ_E_ARG, "%s: null operand", name);
    if (K == 0 || K % 128)
        return set_error(PSQ_E_SHAPE, "%s: K=%lld must be a positive multiple of 128", name, (long long)K);
    if (lda < K || ldw < K || lda % 16 || ldw % 16)
        return set_error(PSQ_E_SHAPE, "%s: lda=%lld ldw=%lld must be multiples of 16 covering K", name,
                         (long long)lda, (long long)ldw);
    if (((uintptr_t)a & 15) || ((uintptr_t)w & 15)) return set_error(PSQ_E_SHAPE, "%s: operands must be 16-byte aligned", name);
    if (M > (1LL << 30) || N > (1LL << 30) || K > (1LL << 30))
        return set_error(PSQ_E_SHAPE, "%s: size too large", name);
    if (lda > (1LL << 23) || ldw > (1LL << 23))   // a tile's row offsets (256 rows) fit in 31 bits
        return set_error(PSQ_E_SHAPE, "%s: lda/ldw above 2^23", name);
    return PSQ_OK;
}

// Activation codes, and the gate's shape rules: N = 2 H rows with H a multiple of 64, an output of
// H columns, and every W row offset (row ldw, 32-bit lane offsets from the weight's first row)
// plus the k offset below 2^32.
int check_act(const char *name, int activation, int64_t N, int64_t ldw, int64_t K, int64_t ldy)
{
    if (activation != ACT_NONE && activation != ACT_GELU_TANH && activation != ACT_SILU_GATE)
        return set_error(PSQ_E_ARG, "%s: bad activation %d", name, activation);
    if (activation == ACT_SILU_GATE) {
        if (N % 128) return set_error(PSQ_E_SHAPE, "%s: the SiLU gate needs N a multiple of 128, got %lld", name, (long long)N);
        if (N * ldw + K >= (1LL << 32)) return set_error(PSQ_E_SHAPE, "%s: the SiLU gate needs N ldw + K < 2^32", name);
        if (ldy < N / 2) return set_error(PSQ_E_SHAPE, "%s: ldy < N / 2", name);
    } else if (ldy < N) {
        return set_error(PSQ_E_SHAPE, "%s: ldy < N", name);
    }
    return PSQ_OK;
}

// The tile width (256, 224, 192 or 160 columns by 256 rows) with the least time for a problem that the
// small tiles leave.
//
// Whole rounds of workgroups cost the tile's own time c, a last round that fills the fraction f of the
// CUs 0.65 + 0.25 f of it (the clock rises with idle CUs).  c, relative to the 256 x 256 tile, from
// 32760 x 13824 x 5120 (31 and 36 rounds against 27) and 8192 x 15360 x 5120 (12 rounds): narrower tiles
// read more LDS per MFMA.  Measured, 256 against the width taken (us, int8): 4095 x 5120 x 5120 114 ->
// 94.9 (160), 4095 x 5120 x 13824 317 -> 260 (160), 2048 x 5120 x 5120 52.5 -> 50.7 (192), 1560 x 13824 x
// 5120 134 -> 117 (192), 4095 x 13824 x 5120 273 -> 259 (224), 8192 x 5376 x 14336 516 -> 497 (224; fp8
// 449 -> 455, left at 256).
int pick_width(bool fp8, int64_t M, int64_t N, int cus)
{
    const struct {
        int width;
        double c;
    } ways[] = {{256, 1.0}, {224, fp8 ? 0.94 : 0.925}, {192, 0.80}, {160, 0.71}};
    int best = 256;
    double least = 1e30;
    for (const auto &w : ways) {
        const int64_t tiles = ((M + 255) / 256) * ((N + w.width - 1) / w.width);
        const double f = (double)(tiles % cus) / cus;
        const double t = w.c * ((double)(tiles / cus) + (f > 0 ? 0.65 + 0.25 * f : 0.0));
        if (t < least) {
            least = t;
            best = w.width;
        }
    }
    return best;
}

// The kernel of a checked call.
int run(int kind, int out, int act, const Q8Args &x)
{
    if (int e = require_device()) return e;
    int status, dev = 0;
    if (q8_small(kind, out, act, x, status)) return status;
    if (hipGetDevice(&dev) != hipSuccess) return set_error(PSQ_E_DEVICE, "%s: no device", x.name);
    const bool fp8 = kind != Q8_I8;
    const int width = out != PSQ_F32 && act != ACT_SILU_GATE ? pick_width(fp8, x.M, x.N, cu_count(dev)) : 256;
    if (width == 256) return fp8 ? q8_square_fp8(kind, out, act, x) : q8_square_i8(out, act, x);
    return fp8 ? q8_width_fp8(kind, width, out, act, x) : q8_width_i8(width, out, act, x);
}

}  // namespace
}  // namespace psq

extern "C" {

int psq_gemm_i8_act(const int8_t *a, int64_t lda, const float *a_scale, const int8_t *w, int64_t ldw,
                    const float *w_scale, const void *bias, int bias_dtype, int activation, void *y, int y_dtype,
                    int64_t ldy, int64_t M, int64_t N, int64_t K, void *stream)
{
    using namespace psq;
    if (int e = check_shapes("gemm_i8", a, lda, w, ldw, M, N, K)) return e;
    if (int e = check_act("gemm_i8", activation, N, ldw, K, ldy)) return e;
    if (M == 0 || N == 0) return PSQ_OK;
    if (!a_scale || !w_scale || !y) return set_error(PSQ_E_ARG, "gemm_i8: null scale or output");
    if (!valid_dtype(y_dtype) || (bias && !valid_dtype(bias_dtype))) return set_error(PSQ_E_ARG, "gemm_i8: bad dtype");
    Q8Epi ep{a_scale, w_scale, 1, bias, bias_dtype, y, ldy, vec_ok(y, ldy, y_dtype == PSQ_F32 ? 4 : 2)};
    return run(Q8_I8, y_dtype, activation,
               {(const uint8_t *)a, lda, (const uint8_t *)w, ldw, M, N, K, ep, (hipStream_t)stream, "gemm_i8"});
}

int psq_gemm_i8(const int8_t *a, int64_t lda, const float *a_scale, const int8_t *w, int64_t ldw,
                const float *w_scale, const void *bias, int bias_dtype, void *y, int y_dtype, int64_t ldy,
                int64_t M, int64_t N, int64_t K, void *stream)
{
    return psq_gemm_i8_act(a, lda, a_scale, w, ldw, w_scale, bias, bias_dtype, PSQ_ACT_NONE, y, y_dtype, ldy, M, N,
                           K, stream);
}

int psq_gemm_i8_i32(const int8_t *a, int64_t lda, const int8_t *w, int64_t ldw, int32_t *c, int64_t ldc,
                    int64_t M, int64_t N, int64_t K, void *stream)
{
    using namespace psq;
    if (int e = check_shapes("gemm_i8_i32", a, lda, w, ldw, M, N, K)) return e;
    if (M == 0 || N == 0) return PSQ_OK;
    if (!c) return set_error(PSQ_E_ARG, "gemm_i8_i32: null output");
    if (ldc < N) return set_error(PSQ_E_SHAPE, "gemm_i8_i32: ldc < N");
    if (int e = require_device()) return e;
    Q8Epi ep{nullptr, nullptr, 0, nullptr, 0, c, ldc, vec_ok(c, ldc, 4)};
    return q8_square_i8(Q8_OUT_I32, ACT_NONE, {(const uint8_t *)a, lda, (const uint8_t *)w, ldw, M, N, K, ep,
                                      (hipStream_t)stream, "gemm_i8_i32"});
}

int psq_gemm_fp8_act(const uint8_t *a, int64_t lda, const float *a_scale, const uint8_t *w, int64_t ldw,
                     const float *w_scale, int w_scale_per_row, const void *bias, int bias_dtype, int activation,
                     void *y, int y_dtype, int64_t ldy, int64_t M, int64_t N, int64_t K, void *stream)
{
    using namespace psq;
    if (int e = check_shapes("gemm_fp8", a, lda, w, ldw, M, N, K)) return e;
    if (int e = check_act("gemm_fp8", activation, N, ldw, K, ldy)) return e;
    if (M == 0 || N == 0) return PSQ_OK;
    if (!a_scale || !w_scale || !y) return set_error(PSQ_E_ARG, "gemm_fp8: null scale or output");
    if (!valid_dtype(y_dtype) || (bias && !valid_dtype(bias_dtype))) return set_error(PSQ_E_ARG, "gemm_fp8: bad dtype");
    Q8Epi ep{a_scale, w_scale, w_scale_per_row ? 1 : 0, bias, bias_dtype, y, ldy, vec_ok(y, ldy, y_dtype == PSQ_F32 ? 4 : 2)};
    return run(Q8_E4M3, y_dtype, activation, {a, lda, w, ldw, M, N, K, ep, (hipStream_t)stream, "gemm_fp8"});
}

int psq_gemm_fp8(const uint8_t *a, int64_t lda, const float *a_scale, const uint8_t *w, int64_t ldw,
                 const float *w_scale, int w_scale_per_row, const void *bias, int bias_dtype, void *y, int y_dtype,
                 int64_t ldy, int64_t M, int64_t N, int64_t K, void *stream)
{
    return psq_gemm_fp8_act(a, lda, a_scale, w, ldw, w_scale, w_scale_per_row, bias, bias_dtype, PSQ_ACT_NONE, y,
                            y_dtype, ldy, M, N, K, stream);
}

int psq_gemm_fp8_e5m2w(const uint8_t *a, int64_t lda, const float *a_scale, const uint8_t *w, int64_t ldw,
                       const float *w_scale, int w_scale_per_row, const void *bias, int bias_dtype, void *y,
                       int y_dtype, int64_t ldy, int64_t M, int64_t N, int64_t K, void *stream)
{
    using namespace psq;
    if (int e = check_shapes("gemm_fp8_e5m2w", a, lda, w, ldw, M, N, K)) return e;
    if (int e = check_act("gemm_fp8_e5m2w", PSQ_ACT_NONE, N, ldw, K, ldy)) return e;
    if (M == 0 || N == 0) return PSQ_OK;
    if (!a_scale || !w_scale || !y) return set_error(PSQ_E_ARG, "gemm_fp8_e5m2w: null scale or output");
    if (!valid_dtype(y_dtype) || (bias && !valid_dtype(bias_dtype)))
        return set_error(PSQ_E_ARG, "gemm_fp8_e5m2w: bad dtype");
    Q8Epi ep{a_scale, w_scale, w_scale_per_row ? 1 : 0, bias, bias_dtype, y, ldy, vec_ok(y, ldy, y_dtype == PSQ_F32 ? 4 : 2)};
    return run(Q8_E5M2W, y_dtype, ACT_NONE, {a, lda, w, ldw, M, N, K, ep, (hipStream_t)stream, "gemm_fp8_e5m2w"});
}

// The codes, rounded up to a 16-byte line, then the row scales.
int64_t psq_linear_q8_scratch_bytes(int64_t M, int64_t K) { return M <= 0 || K <= 0 ? 0 : ((M * K + 15) & ~15LL) + 4 * M; }

int psq_linear_q8(int weights, const void *x, int x_dtype, int64_t ldx, int rot_group, const void *w, int64_t ldw,
                  const float *w_scale, int w_scale_per_row, const void *bias, int bias_dtype, int activation, void *y,
                  int y_f32, int64_t ldy, int64_t M, int64_t N, int64_t K, void *scratch, void *stream)
{
    using namespace psq;
    const char *name = "linear_q8";
    if (weights < PSQ_Q8_I8 || weights > PSQ_Q8_E5M2) return set_error(PSQ_E_ARG, "%s: bad weights %d", name, weights);
    if (weights == PSQ_Q8_E5M2 && (activation != PSQ_ACT_NONE || y_f32))
        return set_error(PSQ_E_ARG, "%s: e5m2 weights take no activation and no fp32 output", name);
    if (y_f32 && activation != PSQ_ACT_NONE) return set_error(PSQ_E_ARG, "%s: an activation has no fp32 output", name);
    if (weights != PSQ_Q8_I8 && rot_group) return set_error(PSQ_E_ARG, "%s: the rotation is int8's", name);
    if (x_dtype != PSQ_BF16 && x_dtype != PSQ_F16) return set_error(PSQ_E_ARG, "%s: activations must be bf16/f16", name);
    if (bias && !valid_dtype(bias_dtype)) return set_error(PSQ_E_ARG, "%s: bad dtype", name);
    // refuse before the quantizer runs what the GEMM would refuse (its operand `a` is made here)
    if (int e = check_shapes(name, w, K, w, ldw, M, N, K)) return e;
    if (int e = check_act(name, activation, N, ldw, K, ldy)) return e;
    if (M == 0 || N == 0) return PSQ_OK;
    if (!w_scale || !y) return set_error(PSQ_E_ARG, "%s: null scale or output", name);
    uint8_t *q = (uint8_t *)scratch;
    float *sx = (float *)(q + ((M * K + 15) & ~15LL));
    const bool i8 = weights == PSQ_Q8_I8;
    const int kind = i8 ? Q8_I8 : weights == PSQ_Q8_E4M3 ? Q8_E4M3 : Q8_E5M2W;
    Q8Epi ep{sx, w_scale, i8 || w_scale_per_row ? 1 : 0, bias, bias_dtype, y, ldy, vec_ok(y, ldy, y_f32 ? 4 : 2)};
    const Q8Args args{q, K, (const uint8_t *)w, ldw, M, N, K, ep, (hipStream_t)stream, name};
    // one or two rows: quantized by the GEMM itself (what the quantizer would refuse goes to it)
    int rotk = 0;
    if (q8_vec_fits(M, K, activation) && x && ((uintptr_t)x & 15) == 0 && ldx >= K && ldx % 8 == 0 &&
        rot_log4(rot_group, K, rotk) == PSQ_OK) {
        if (int e = require_device()) return e;
        return q8_vec(kind, x, x_dtype, ldx, rotk, y_f32 ? 1 : 0, activation, args);
    }
    if (!scratch || ((uintptr_t)scratch & 15)) return set_error(PSQ_E_ARG, "%s: scratch must be 16-byte aligned", name);
    if (int e = i8 ? psq_quantize_rows_i8(x, x_dtype, M, K, ldx, rot_group, nullptr, (int8_t *)q, K, sx, stream)
                   : psq_quantize_rows_fp8(x, x_dtype, M, K, ldx, 0, nullptr, q, K, sx, stream))
        return e;
    const int out = !y_f32 ? x_dtype : x_dtype == PSQ_BF16 ? Q8_WIDE_BF16 : Q8_WIDE_F16;
    return run(kind, out, activation, args);
}

}  // extern "C"
