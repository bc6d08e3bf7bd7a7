// gemm_q8_vec.hip -- quantize one or two rows and multiply them by the int8 / fp8 weights in one kernel:
// the conditioning vectors and next-token calls, bound by the weight stream and by launches.
//
// Same values as quantize_rows.hip followed by gemm_q8_small.hip's 16 x 32 tiles.  A workgroup of 8
// waves computes 32 output columns: its first weight blocks are put in flight into the LDS ring, and
// while they travel every workgroup quantizes the rows for itself (20 KB of activations at K = 5120, L2
// hits, about 1 us of work) into LDS, where all its K blocks read their fragments.  That takes out a
// launch, the codes' round trip through memory and the gap between the kernels (us, against the two
// kernels, rotating weights): 1 x 15360 x 5120 18.7 -> 15.5, 1 x 5120 x 5120 11.2 -> 8.6, 1 x 25600 x 5120
// 29.3 -> 26.2, 2 x 5120 x 5120 11.2 -> 9.8, 1 x 1024 x 1024 8.8 -> 5.0.  Two rows at most: each
// workgroup repeats the quantization.
#include "quantize.hpp"
#include "gemm_q8.hpp"

namespace psq {
namespace {

constexpr int NW = 8, NCG = 2, KH = 4;           // waves: column groups of 16 x splits of K
constexpr int BN = 16 * NCG, BLK = 128;          // W rows of a tile, bytes of K per block
constexpr int ITB = KH * BN * BLK;               // ring bytes of an iteration of KH blocks (16 KB)
constexpr int SLOTS = 3, D = SLOTS - 1;          // iterations: in the ring, in flight
constexpr int LI = ITB / 1024 / NW;              // ring loads per wave and iteration
constexpr int MAXM = 2, MAXK = 8192;             // rows; one 16-element chunk of each per thread
constexpr int OPS_WORDS = 16 + 2 * BN + MAXM * NW;   // row scales, column scales, bias words, absmax words

// 16-byte chunk c of W row r sits at c ^ swz(r), as in gemm_q8_small.hip
__device__ __forceinline__ int swz(int r) { return ((r >> 1) & 1) | ((r >> 2) & 2) | (r & 4); }

// The two code rows lie K + 64 bytes apart, so that fragments of both rows fall on distinct banks.
__host__ __device__ constexpr int code_stride(int K) { return K + 64; }
// The raw activations wait in the ring's last slot (free until the first block is computed) when they
// fit it, else past the codes.
__host__ __device__ constexpr bool x_in_ring(int M, int K) { return M * K * 2 <= ITB; }
constexpr int smem_bytes(int M, int K)
{
    return SLOTS * ITB + 2 * code_stride(K) + (x_in_ring(M, K) ? 0 : M * K * 2) + OPS_WORDS * 4;
}

// At most `left` iterations' loads may stay in flight.
__device__ __forceinline__ void wait_left(int left)
{
    static_for<D + 1>([&](auto ic) {
        constexpr int i = D - decltype(ic)::value;
        if (left == i) wait_vmcnt<i * LI>();
    });
}

template <int KIND, int DT, int ROTK>
__global__ void __launch_bounds__(64 * NW, 4)
q8_vec_kernel(const uint16_t *__restrict__ x, int64_t ldx, const uint8_t *__restrict__ W, int64_t ldw, int M, int N,
              int K, Q8Epi ep, int wide, int act)
{
    using Acc = typename std::conditional<KIND == Q8_I8, v4i, v4f>::type;
    constexpr float LIM = KIND == Q8_I8 ? 127.0f : 448.0f;
    extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int cg = wave % NCG, kh = wave / NCG;
    const int n0 = xcd_rank(blockIdx.x, gridDim.x) * BN;
    const int nk = K / BLK, nit = (nk + KH - 1) / KH;
    const int cst = code_stride(K);
    uint8_t *const codes = smem + SLOTS * ITB;
    uint8_t *const xb = x_in_ring(M, K) ? smem + D * ITB : codes + 2 * cst;
    uint32_t *const ops = (uint32_t *)(codes + 2 * cst + (x_in_ring(M, K) ? 0 : M * K * 2));
    uint32_t *const amax_lds = ops + 16 + 2 * BN;

    // first the activations and the tile's epilogue operands, then the ring's first iterations
    const int xl = (2 * K + 1023) / 1024;          // 1 KB loads of a row
    for (int c = wave; c < M * xl; c += NW) {
        const int r = c / xl, o = (c - r * xl) * 1024;
        if (o + 16 * lane < 2 * K)
            __builtin_amdgcn_global_load_lds((glb_ptr)((const uint8_t *)(x + r * ldx) + o + 16 * lane),
                                             (lds_ptr)(xb + r * 2 * K + o), 16, 0, 0);
    }
    if (wave == 0) {
        const int n = min(n0 + (lane & (BN - 1)), N - 1);
        if (lane < BN) {
            __builtin_amdgcn_global_load_lds((glb_ptr)(ep.w_scale + (ep.w_per_row ? n : 0)), (lds_ptr)(ops + 16), 4, 0, 0);
            if (ep.bias && ep.bias_dtype == PSQ_F32)
                __builtin_amdgcn_global_load_lds((glb_ptr)((const uint32_t *)ep.bias + n), (lds_ptr)(ops + 16 + BN), 4, 0, 0);
            else if (ep.bias)
                __builtin_amdgcn_global_load_lds((glb_ptr)((const uint16_t *)ep.bias + n), (lds_ptr)(ops + 16 + BN), 2, 0, 0);
        }
    }
    // wave load i of an iteration: 8 W rows x 128 bytes of K block (i NW + wave) / 4
    const uint8_t *base[LI];
    uint32_t off[LI];
#pragma unroll
    for (int i = 0; i < LI; i++) {
        const int wr = 8 * ((i * NW + wave) % (BN / 8)), l = lane >> 3, r0 = min(n0 + wr, N - 1);
        base[i] = W + (int64_t)r0 * ldw;
        off[i] = (uint32_t)((min(n0 + wr + l, N - 1) - r0) * (int)ldw + (((lane & 7) ^ swz(wr + l)) << 4));
    }
    auto issue = [&](int it, int slot) {
#pragma unroll
        for (int i = 0; i < LI; i++) {
            const int idx = i * NW + wave, b = min(it * KH + idx / (BN / 8), nk - 1);
            __builtin_amdgcn_global_load_lds((glb_ptr)(base[i] + (int64_t)b * BLK + off[i]),
                                             (lds_ptr)(smem + slot * ITB + 1024 * idx), 16, 0, 0);
        }
    };
    const int ahead = min(D, nit);
    for (int it = 0; it < ahead; it++) issue(it, it);
    wait_left(ahead);                              // the activations, the older loads, have landed
    stage_barrier();

    // ---- quantize (quantize_rows.hip, one chunk of 16 elements per thread and row)
    const int lc = lane_chunk<ROTK>(tid), e0 = 16 * lc;
    const float post = ROTK ? __builtin_ldexpf(1.0f, -ROTK) : 1.0f;
    float v[MAXM][16];
#pragma unroll
    for (int r = 0; r < MAXM; r++) {
        if (r >= M) break;
        v4i raw[2] = {v4i{0, 0, 0, 0}, v4i{0, 0, 0, 0}};
        if (e0 < K) {
            raw[0] = *(const v4i *)(xb + r * 2 * K + 2 * e0);
            raw[1] = *(const v4i *)(xb + r * 2 * K + 2 * e0 + 16);
        }
        to_f32<DT>(raw, v[r]);
        rotate16<ROTK>(v[r]);
        const uint32_t bits = wave_max_bits(__float_as_uint(absmax16(v[r])));
        if (lane == 0) amax_lds[r * NW + wave] = bits;
    }
    stage_barrier();
#pragma unroll
    for (int r = 0; r < MAXM; r++) {
        if (r >= M) break;
        uint32_t bits = amax_lds[r * NW];
#pragma unroll
        for (int w = 1; w < NW; w++) bits = max(bits, amax_lds[r * NW + w]);
        const float amax = __uint_as_float(bits);
        const float mul = amax == 0.0f ? 1.0f : LIM / amax;
        if (tid == 0) ops[r] = __float_as_uint(amax == 0.0f ? 1.0f : (amax / LIM) * post);
        uint32_t p[4];
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const float *u = &v[r][4 * i];
            if constexpr (KIND == Q8_I8) p[i] = i8_codes4(u[0] * mul, u[1] * mul, u[2] * mul, u[3] * mul, kRoundMagic);
            else p[i] = e4m3_codes4(u[0] * mul, u[1] * mul, u[2] * mul, u[3] * mul);
        }
        if (e0 < K) *(v4i *)(codes + r * cst + 16 * (lc ^ rev_lanes<ROTK>())) = v4i{(int)p[0], (int)p[1], (int)p[2], (int)p[3]};
    }

    // ---- K loop.  Fragment rows past the second repeat rows 0 and 1: their output rows are dropped.
    const int fr = lane & 15, fs = lane >> 4;
    const uint32_t w0 = (uint32_t)((cg * 16 + fr) * BLK + ((fs ^ swz(fr)) << 4)), w1 = w0 ^ 64;
    const uint8_t *const ar = codes + (fr & 1) * cst + 16 * fs;
    Acc acc{};
    int slot = 0;
#pragma clang loop unroll(disable)
    for (int it = 0; it < nit; it++) {
        wait_left(min(D, nit - it) - 1);
        stage_barrier();      // landed for every wave (first: the codes too); the slot refilled next is free
        if (it + D < nit) issue(it + D, slot == 0 ? D : slot - 1);
        const int b = it * KH + kh;
        if (b < nk) {
            const uint8_t *sw = smem + slot * ITB + kh * BN * BLK;
            const v4i x0 = *(const v4i *)(ar + b * BLK), x1 = *(const v4i *)(ar + b * BLK + 64);
            const v4i y0 = *(const v4i *)(sw + w0), y1 = *(const v4i *)(sw + w1);
            if constexpr (KIND == Q8_I8) {
                acc = __builtin_amdgcn_mfma_i32_16x16x64_i8(y0, x0, acc, 0, 0, 0);
                acc = __builtin_amdgcn_mfma_i32_16x16x64_i8(y1, x1, acc, 0, 0, 0);
            } else {
                const v8i xf = v8i{x0[0], x0[1], x0[2], x0[3], x1[0], x1[1], x1[2], x1[3]};
                const v8i yf = v8i{y0[0], y0[1], y0[2], y0[3], y1[0], y1[1], y1[2], y1[3]};
                acc = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(yf, xf, acc, KIND == Q8_E5M2W ? 1 : 0, 0, 0, 127, 0, 127);
            }
        }
        slot = slot == D ? 0 : slot + 1;
    }

    // ---- the K splits' sums, added in split order; lane: row fr, columns 4 fs .. + 3 of the group
    stage_barrier();
    v4i *red = (v4i *)smem;
    if (kh) red[wave * 64 + lane] = __builtin_bit_cast(v4i, acc);
    stage_barrier();
    const int nl = cg * 16 + 4 * fs;
    if (kh || fr >= M || n0 + nl >= N) return;
#pragma unroll
    for (int h = 1; h < KH; h++) acc = acc + __builtin_bit_cast(Acc, red[(h * NCG + cg) * 64 + lane]);
    const float as = __uint_as_float(ops[fr]);
#pragma unroll
    for (int c = 0; c < 4; c++) {
        if (n0 + nl + c >= N) break;
        const float b = ep.bias ? bias_word(ops[16 + BN + nl + c], ep.bias_dtype) : 0.0f;
        uint32_t h = pack_half2<DT>(__builtin_fmaf((float)acc[c], as * __uint_as_float(ops[16 + nl + c]), b), 0.0f);
        if (act == ACT_GELU_TANH) h = pack_half2<DT>(gelu_tanh(half_to_f32<DT>(h)), 0.0f);
        const int64_t o = fr * ep.ldy + n0 + nl + c;
        if (wide) ((float *)ep.y)[o] = half_to_f32<DT>(h);
        else ((uint16_t *)ep.y)[o] = (uint16_t)h;
    }
}

template <int KIND, int DT, int ROTK>
int launch_vec(const uint16_t *x, int64_t ldx, int wide, int act, const Q8Args &a)
{
    auto kern = q8_vec_kernel<KIND, DT, ROTK>;
    constexpr int kMost = smem_bytes(MAXM, MAXK);
    static_assert(kMost <= 160 * 1024);
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess) return set_error(PSQ_E_DEVICE, "%s: no device", a.name);
    static bool attr_set[64] = {};   // per device; the attribute is idempotent
    if (dev >= 64 || !attr_set[dev]) {
        if (hipFuncSetAttribute((const void *)kern, hipFuncAttributeMaxDynamicSharedMemorySize, kMost) != hipSuccess)
            return set_error(PSQ_E_DEVICE, "%s: cannot reserve %d bytes of LDS", a.name, kMost);
        if (dev < 64) attr_set[dev] = true;
    }
    kern<<<dim3((unsigned)((a.N + BN - 1) / BN)), dim3(64 * NW), smem_bytes((int)a.M, (int)a.K), a.st>>>(
        x, ldx, a.w, a.ldw, (int)a.M, (int)a.N, (int)a.K, a.ep, wide, act);
    return check_launch(a.name);
}

template <int DT>
int launch_rot(int kind, const uint16_t *x, int64_t ldx, int rotk, int wide, int act, const Q8Args &a)
{
    if (kind == Q8_E4M3) return launch_vec<Q8_E4M3, DT, 0>(x, ldx, wide, act, a);
    if (kind == Q8_E5M2W) return launch_vec<Q8_E5M2W, DT, 0>(x, ldx, wide, act, a);
    switch (rotk) {
    case 0: return launch_vec<Q8_I8, DT, 0>(x, ldx, wide, act, a);
    case 1: return launch_vec<Q8_I8, DT, 1>(x, ldx, wide, act, a);
    case 2: return launch_vec<Q8_I8, DT, 2>(x, ldx, wide, act, a);
    case 3: return launch_vec<Q8_I8, DT, 3>(x, ldx, wide, act, a);
    case 4: return launch_vec<Q8_I8, DT, 4>(x, ldx, wide, act, a);
    default: return launch_vec<Q8_I8, DT, 5>(x, ldx, wide, act, a);
    }
}

}  // namespace

bool q8_vec_fits(int64_t M, int64_t K, int act) { return M >= 1 && M <= MAXM && K <= MAXK && act != ACT_SILU_GATE; }

int q8_vec(int kind, const void *x, int x_dtype, int64_t ldx, int rotk, int wide, int act, const Q8Args &a)
{
    const uint16_t *xp = (const uint16_t *)x;
    return x_dtype == PSQ_BF16 ? launch_rot<PSQ_BF16>(kind, xp, ldx, rotk, wide, act, a)
                               : launch_rot<PSQ_F16>(kind, xp, ldx, rotk, wide, act, a);
}

}  // namespace psq
