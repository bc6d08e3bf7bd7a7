// quantize.hpp -- the per-thread pieces of the activation quantizer (quantize_rows.hip, whose header has
// the conventions), shared with the GEMM that quantizes its own rows (gemm_q8_vec.hip).
#pragma once

#include "psq_common.hpp"

namespace psq {

template <int DT>
__device__ __forceinline__ void to_f32(const v4i (&raw)[2], float (&v)[16])
{
#pragma unroll
    for (int i = 0; i < 4; i++) {
        uint32_t a = (uint32_t)raw[0][i], b = (uint32_t)raw[1][i];
        v[2 * i] = half_to_f32<DT>(a);
        v[2 * i + 1] = half_to_f32<DT>(a >> 16);
        v[8 + 2 * i] = half_to_f32<DT>(b);
        v[8 + 2 * i + 1] = half_to_f32<DT>(b >> 16);
    }
}

// Largest |v| over the 16 values, NaN if any is NaN (IEEE maximum: gfx950's v_maximum3_f32 with
// |.| source modifiers, two values per instruction).  A row holding a NaN thereby gets a NaN scale,
// as torch's amax gives, and its dequantized output is NaN.
__device__ __forceinline__ float absmax16(const float (&v)[16])
{
    float m = __builtin_elementwise_maximum(__builtin_fabsf(v[0]), __builtin_fabsf(v[1]));
#pragma unroll
    for (int j = 2; j < 16; j += 2)
        m = __builtin_elementwise_maximum(m, __builtin_elementwise_maximum(__builtin_fabsf(v[j]), __builtin_fabsf(v[j + 1])));
    return m;
}

// Wave-wide max of non-negative values (a NaN wins): the bit patterns of non-negative floats order
// as unsigned integers like their values, and a positive NaN's pattern lies above +inf's.  DPP within
// rows of 16 lanes, then the gfx950 row swaps across rows (no LDS, no index arithmetic).
template <int CTRL>
__device__ __forceinline__ uint32_t dpp_u32(uint32_t v)
{
    return (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, CTRL, 0xF, 0xF, true);
}

__device__ __forceinline__ uint32_t wave_max_bits(uint32_t u)
{
    u = max(u, dpp_u32<DPP_QUAD_XOR1>(u));
    u = max(u, dpp_u32<DPP_QUAD_XOR2>(u));
    u = max(u, dpp_u32<DPP_ROW_HALF_MIRROR>(u));   // lane ^ 7: the other quad of the 8
    u = max(u, dpp_u32<DPP_ROW_MIRROR>(u));        // lane ^ 15: the other 8 of the row
    const auto a = __builtin_amdgcn_permlane16_swap(u, u, false, false);   // rows 0 <-> 1, 2 <-> 3
    u = max((uint32_t)a[0], (uint32_t)a[1]);
    const auto b = __builtin_amdgcn_permlane32_swap(u, u, false, false);   // halves
    return max((uint32_t)b[0], (uint32_t)b[1]);
}

// int8 code of u r: clamp to [-127, 127] (equal to clamping after rounding, the bounds being
// integers), then + 1.5 * 2^23, which rounds to the nearest integer (ties to even) and leaves the
// code's two's complement in the low byte of the sum.  A NaN clamps to -127, as fmax(NaN, -127)
// does in the rounding-first order.
constexpr float kRoundMagic = 12582912.0f;

__device__ __forceinline__ float i8_clamp(float u) { return __builtin_fminf(__builtin_fmaxf(u, -127.0f), 127.0f); }

// Four codes packed into one word by the adds that round them: the first add writes the whole word
// (its low byte is code 0), the other three are v_add_f32 with an SDWA destination, which writes
// the low byte of the sum into byte B of the word and keeps the other bytes.  No separate pack.
template <int B>
__device__ __forceinline__ void add_into_byte(uint32_t &w, float u, float magic)
{
    static_assert(B >= 1 && B <= 3, "byte 1-3");
    if constexpr (B == 1)
        asm("v_add_f32_sdwa %0, %1, %2 dst_sel:BYTE_1 dst_unused:UNUSED_PRESERVE src0_sel:DWORD src1_sel:DWORD"
            : "+v"(w) : "v"(u), "v"(magic));
    else if constexpr (B == 2)
        asm("v_add_f32_sdwa %0, %1, %2 dst_sel:BYTE_2 dst_unused:UNUSED_PRESERVE src0_sel:DWORD src1_sel:DWORD"
            : "+v"(w) : "v"(u), "v"(magic));
    else
        asm("v_add_f32_sdwa %0, %1, %2 dst_sel:BYTE_3 dst_unused:UNUSED_PRESERVE src0_sel:DWORD src1_sel:DWORD"
            : "+v"(w) : "v"(u), "v"(magic));
}

__device__ __forceinline__ uint32_t i8_codes4(float u0, float u1, float u2, float u3, float magic)
{
    uint32_t w = __float_as_uint(i8_clamp(u0) + magic);
    add_into_byte<1>(w, i8_clamp(u1), magic);
    add_into_byte<2>(w, i8_clamp(u2), magic);
    add_into_byte<3>(w, i8_clamp(u3), magic);
    return w;
}

// Four e4m3fn codes: gfx950's v_cvt_pk_fp8_f32 is the OCP encode with round to nearest even (subnormals
// included); the clamp keeps it off the overflow path and, as in the int8 codes, takes a NaN product
// to the lower bound.
__device__ __forceinline__ uint32_t e4m3_codes4(float u0, float u1, float u2, float u3)
{
    auto clamp = [](float u) { return __builtin_fminf(__builtin_fmaxf(u, -448.0f), 448.0f); };
    const int lo = __builtin_amdgcn_cvt_pk_fp8_f32(clamp(u0), clamp(u1), 0, false);
    return (uint32_t)__builtin_amdgcn_cvt_pk_fp8_f32(clamp(u2), clamp(u3), lo, true);
}

// rot_group 0 (rotk 0) or a power of 4 in [4, 1024] dividing K (rotk = its base-4 log)
inline int rot_log4(int rot_group, int64_t K, int &rotk)
{
    rotk = 0;
    if (!rot_group) return PSQ_OK;
    int g = rot_group;
    while (g > 1 && (g & 3) == 0) { g >>= 2; rotk++; }
    if (g != 1 || rotk < 1 || rotk > 5 || K % rot_group)
        return set_error(PSQ_E_SHAPE, "rotation group %d must be a power of 4 in [4,1024] dividing K=%lld", rot_group,
                         (long long)K);
    return PSQ_OK;
}

}  // namespace psq
