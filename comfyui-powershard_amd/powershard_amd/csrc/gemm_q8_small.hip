// gemm_q8_small.hip -- the W8A8 int8 and fp8 GEMMs for problems that leave CUs idle under the
// 256 x 256 tiles of gemm_q8.hip: one vector, a prompt's tokens, narrow layers.
//
// Same operands, arithmetic and epilogue as gemm_q8.hip (see there):
//   y[m][n] = round_out(act(round_out(fmaf((float)acc[m][n], a_scale[m] * w_scale[n], bias[n]))))
// int8 sums are exact, so the outputs are the same bits; fp8 sums are fp32, added in another order.
//
// One workgroup of 8 waves per tile.  K runs in blocks of 128 bytes (one cache line of every row)
// through an LDS ring filled by global->LDS loads, as deep as the LDS allows; the waves split the
// tile's rows, its columns and, where the tile is small, K: KH waves take KH consecutive blocks of an
// iteration, so one barrier serves KH blocks and a weight row is read KH lines at a time.  Their
// partial tiles meet in LDS at the end, in a fixed order.
//
// What bounds it, measured (us, back-to-back launches over rotating weights, against the 256 x 256
// tiles): the weight stream up to about 80 rows -- 1 x 15360 x 5120 67.5 -> 15.5 (5.1 TB/s), 77 x 15360
// x 5120 67.8 -> 22.4, 1 x 5120 x 5120 48.2 -> 6.4, 40 x 13824 x 5120 67.2 -> 17.9 -- then LDS traffic
// (fragment reads plus the ring's writes, about 110 bytes per cycle and CU): 160 x 5120 x 5120 48.1 ->
// 11.6, 512 x 5120 x 5120 49.4 -> 22.6, 1024 x 5120 x 5120 49.4 -> 32.0, 512 x 13824 x 5120 67.0 -> 46.5.
#include "psq_common.hpp"
#include "gemm_q8.hpp"

namespace psq {
namespace {

constexpr int BLK = 128;               // bytes (= elements) of K per block: one cache line of every row

// 16-byte chunk c of LDS row r sits at c ^ swz(r).  A fragment read takes 16 rows at chunk 4 h + s
// (s = lane >> 4); ds_read_b128 serves the lanes {0-3, 12-15, 20-23, 24-27} (and their complements)
// in one cycle each, and for these the swizzle gives 16 distinct (row parity, chunk) pairs.
__device__ __forceinline__ int swz(int r) { return ((r >> 1) & 1) | ((r >> 2) & 2) | (r & 4); }

template <int KIND> struct Kind;
template <> struct Kind<0> { typedef v4i Acc; };
template <> struct Kind<1> { typedef v4f Acc; };
template <> struct Kind<2> { typedef v4f Acc; };

template <int NW, int TM, int TN, int NRG, int NCG, int BUDGET>
struct Cfg {
    static constexpr int KH = NW / (NRG * NCG);          // waves that split K
    static constexpr int BM = 16 * TM * NRG, BN = 16 * TN * NCG;
    static constexpr int RBA = BM / 8, RBW = BN / 8;         // 8-row blocks loaded per K block
    static constexpr int TOT = KH * (RBA + RBW);             // 1 KB wave loads per iteration
    static constexpr int LI = (TOT + NW - 1) / NW;   // per wave
    static constexpr int BLKB = (BM + BN) * BLK;             // LDS bytes of a K block
    static constexpr int ITB = KH * BLKB;
    static constexpr int FIT = BUDGET / ITB, CAP = 60 / LI + 1;
    static constexpr int SLOTS = FIT < 2 ? 2 : (FIT > CAP ? CAP : (FIT > 12 ? 12 : FIT));
    static constexpr int D = SLOTS - 1;                      // iterations in flight
    static constexpr int REDB = KH > 1 ? NW * TM * TN * 1024 : 0;
    static constexpr int RING = SLOTS * ITB > REDB ? SLOTS * ITB : REDB;
    static constexpr int SMEM = RING + (BM + 2 * BN + 63) / 64 * 256;   // then the epilogue operands
    static_assert(SMEM <= 160 * 1024);
};

// Waves per SIMD that the registers allow: accumulators, one or two sets of fragments, addresses.
constexpr int min_waves(int tm, int tn, bool pipe)
{
    const int regs = 4 * tm * tn + (pipe ? 2 : 1) * 8 * (tm + tn) + 44;
    return regs <= 128 ? 4 : regs <= 256 ? 2 : 1;
}

template <int D, int LI>
__device__ __forceinline__ void wait_left(int left)   // at most `left` iterations may stay in flight
{
    if (left == D - 1) {
        wait_vmcnt<(D - 1) * LI>();
        return;
    }
    static_for<D - 1>([&](auto ic) {
        constexpr int i = decltype(ic)::value;
        if (left == i) wait_vmcnt<i * LI>();
    });
}

template <int KIND, int NW, int TM, int TN, int NRG, int NCG, int BUDGET, bool PIPE, bool GATE>
__global__ void __launch_bounds__(64 * NW, min_waves(TM, TN, PIPE))
q8_small_kernel(const uint8_t *__restrict__ A, int64_t lda, const uint8_t *__restrict__ W, int64_t ldw, int M, int N,
                int K, Q8Epi ep, int out, int act)
{
    using C = Cfg<NW, TM, TN, NRG, NCG, BUDGET>;
    using Acc = typename Kind<KIND>::Acc;
    constexpr int KH = C::KH, LI = C::LI, D = C::D;
    extern __shared__ __attribute__((aligned(16))) uint8_t smem[];

    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int cg = wave % NCG, rg = (wave / NCG) % NRG, kh = wave / (NCG * NRG);
    constexpr int ON = GATE ? C::BN / 2 : C::BN;             // output columns of a tile
    const int NO = GATE ? N >> 1 : N;
    const int nbm = (M + C::BM - 1) / C::BM;
    // tiles column after column, consecutive ones on one XCD: the row tiles of a column block read
    // its weights from that XCD's L2
    const int lid = xcd_rank(blockIdx.x, gridDim.x);
    const int m0 = (lid % nbm) * C::BM, n0 = (lid / nbm) * ON;
    const int nk = K / BLK, nit = (nk + KH - 1) / KH;

    // ring loads: wave load i of an iteration is 8 rows x 128 bytes of one K block
    const uint8_t *base[LI];
    uint32_t off[LI];
    int dst[LI], kb[LI];
#pragma unroll
    for (int i = 0; i < LI; i++) {
        const int idx = min(i * NW + wave, C::TOT - 1);
        kb[i] = idx / (C::RBA + C::RBW);
        const int rb = idx % (C::RBA + C::RBW);
        const int l = lane >> 3;
        if (rb < C::RBA) {
            const int r0 = min(m0 + 8 * rb, M - 1);
            base[i] = A + (int64_t)r0 * lda;
            off[i] = (uint32_t)((min(m0 + 8 * rb + l, M - 1) - r0) * (int)lda + (((lane & 7) ^ swz(8 * rb + l)) << 4));
            dst[i] = kb[i] * C::BLKB + 1024 * rb;
        } else {
            const int wr = 8 * (rb - C::RBA);                // row of the tile's W rows
            int n, lim;
            int64_t up = 0;
            if constexpr (GATE) {
                const int j = (wr >> 4) % TN, c = (wr >> 4) / TN;
                n = n0 + (c * (TN / 2) + j % (TN / 2)) * 16 + (wr & 15);
                lim = NO - 1;
                up = j >= TN / 2 ? NO : 0;
            } else {
                n = n0 + wr;
                lim = N - 1;
            }
            const int r0 = min(n, lim);
            base[i] = W + (r0 + up) * ldw;
            off[i] = (uint32_t)((min(n + l, lim) - r0) * (int)ldw + (((lane & 7) ^ swz(wr + l)) << 4));
            dst[i] = kb[i] * C::BLKB + C::BM * BLK + 1024 * (rb - C::RBA);
        }
    }
    // The tile's epilogue operands go to LDS past the ring: row scales, then the column scales and
    // raw bias words in the order of the tile's W rows.  Issued first, so they have landed when the
    // first block has.
    uint32_t *const ops = (uint32_t *)(smem + C::RING);
    for (int c = wave; c < (C::BM + 2 * C::BN + 63) / 64; c += NW) {
        const int e = 64 * c + lane;
        lds_ptr d = (lds_ptr)(ops + 64 * c);
        if (e < C::BM) {
            __builtin_amdgcn_global_load_lds((glb_ptr)(ep.a_scale + min(m0 + e, M - 1)), d, 4, 0, 0);
        } else if (e < C::BM + 2 * C::BN) {
            const int wr = (e - C::BM) % C::BN;
            int n;
            if constexpr (GATE) {
                const int j = (wr >> 4) % TN, g = (wr >> 4) / TN;
                n = min(n0 + (g * (TN / 2) + j % (TN / 2)) * 16 + (wr & 15), NO - 1) + (j >= TN / 2 ? NO : 0);
            } else {
                n = min(n0 + wr, N - 1);
            }
            if (e < C::BM + C::BN) {
                __builtin_amdgcn_global_load_lds((glb_ptr)(ep.w_scale + (ep.w_per_row ? n : 0)), d, 4, 0, 0);
            } else if (ep.bias) {
                if (ep.bias_dtype == PSQ_F32) __builtin_amdgcn_global_load_lds((glb_ptr)((const uint32_t *)ep.bias + n), d, 4, 0, 0);
                else __builtin_amdgcn_global_load_lds((glb_ptr)((const uint16_t *)ep.bias + n), d, 2, 0, 0);
            }
        }
    }
    auto issue = [&](int it, int slot) {
#pragma unroll
        for (int i = 0; i < LI; i++) {
            const int b = min(it * KH + kb[i], nk - 1);
            __builtin_amdgcn_global_load_lds((glb_ptr)(base[i] + (int64_t)b * BLK + off[i]),
                                             (lds_ptr)(smem + slot * C::ITB + dst[i]), 16, 0, 0);
        }
    };

    const int fr = lane & 15, fs = lane >> 4;
    const int mb = m0 + rg * TM * 16;
    constexpr int TO = GATE ? TN / 2 : TN, NG = GATE ? 2 : 1;
    const uint32_t c0 = (uint32_t)(fr * BLK + ((fs ^ swz(fr)) << 4)), c1 = c0 ^ 64;
    Acc acc[TM][TN];
#pragma unroll
    for (int i = 0; i < TM; i++)
#pragma unroll
        for (int j = 0; j < TN; j++) acc[i][j] = Acc{};

    // Fragments of one K block: chunks c0 and c1 of the wave's TN W tiles and TM A tiles.
    struct Frags {
        v4i w[2][TN], a[2][TM];
    };
    auto read = [&](int slot, Frags &f) {
        const uint8_t *sa = smem + slot * C::ITB + kh * C::BLKB + rg * TM * 16 * BLK;
        const uint8_t *sw = smem + slot * C::ITB + kh * C::BLKB + (C::BM + cg * TN * 16) * BLK;
#pragma unroll
        for (int h = 0; h < 2; h++) {
#pragma unroll
            for (int j = 0; j < TN; j++) f.w[h][j] = *(const v4i *)(sw + j * 16 * BLK + (h ? c1 : c0));
#pragma unroll
            for (int i = 0; i < TM; i++) f.a[h][i] = *(const v4i *)(sa + i * 16 * BLK + (h ? c1 : c0));
        }
    };
    auto compute = [&](const Frags &f) {
        if constexpr (KIND == 0) {
#pragma unroll
            for (int h = 0; h < 2; h++)
#pragma unroll
                for (int i = 0; i < TM; i++)
#pragma unroll
                    for (int j = 0; j < TN; j++)
                        acc[i][j] = __builtin_amdgcn_mfma_i32_16x16x64_i8(f.w[h][j], f.a[h][i], acc[i][j], 0, 0, 0);
        } else {
#pragma unroll
            for (int i = 0; i < TM; i++)
#pragma unroll
                for (int j = 0; j < TN; j++) {
                    const v4i x0 = f.a[0][i], x1 = f.a[1][i], y0 = f.w[0][j], y1 = f.w[1][j];
                    const v8i x = v8i{x0[0], x0[1], x0[2], x0[3], x1[0], x1[1], x1[2], x1[3]};
                    const v8i y = v8i{y0[0], y0[1], y0[2], y0[3], y1[0], y1[1], y1[2], y1[3]};
                    acc[i][j] = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(y, x, acc[i][j], KIND == 2 ? 1 : 0, 0, 0, 127, 0, 127);
                }
        }
    };
    // One iteration: block group `it` has landed; its fragments are read (into `nxt`) behind the
    // MFMAs of the previous one (`cur`), and the slot that held the previous one is refilled.
    for (int it = 0; it < D && it < nit; it++) issue(it, it);
    int slot = 0;
    auto advance = [&](int it) {
        wait_left<D, LI>(min(D, nit - it) - 1);
        stage_barrier();      // landed for every wave; every wave has read the slot refilled next
        if (it + D < nit) issue(it + D, slot == 0 ? D : slot - 1);
    };
    auto overlap = [&](Frags &cur, Frags &nxt) {
        constexpr int NR = 2 * (TM + TN), NM = (KIND == 0 ? 2 : 1) * TM * TN;
        __builtin_amdgcn_sched_barrier(0);
        read(slot, nxt);
        compute(cur);
        // one MFMA, then as many reads as spread them evenly
        static_for<NM>([&](auto pc) {
            constexpr int p = decltype(pc)::value, r = (p + 1) * NR / NM - p * NR / NM;
            if constexpr (r > 0) __builtin_amdgcn_sched_group_barrier(0x100, r, 0);
            __builtin_amdgcn_sched_group_barrier(0x8, 1, 0);
        });
        __builtin_amdgcn_sched_barrier(0);
    };
    if constexpr (PIPE) {
        Frags f0, f1;
        advance(0);
        read(0, f0);
        slot = slot == D ? 0 : slot + 1;
        int it = 1;
#pragma clang loop unroll(disable)
        for (; it + 1 < nit; it += 2) {
            advance(it);
            overlap(f0, f1);
            slot = slot == D ? 0 : slot + 1;
            advance(it + 1);
            overlap(f1, f0);
            slot = slot == D ? 0 : slot + 1;
        }
        // the last one or two block groups; with split K the last group may be short
        if (it < nit) {
            advance(it);
            overlap(f0, f1);
            if (KH == 1 || it * KH + kh < nk) compute(f1);
        } else if (KH == 1 || (nit - 1) * KH + kh < nk) {
            compute(f0);
        }
    } else {
#pragma clang loop unroll(disable)
        for (int it = 0; it < nit; it++) {
            Frags f;
            advance(it);
            if (KH == 1 || it * KH + kh < nk) {
                read(slot, f);
                __builtin_amdgcn_sched_barrier(0);
                compute(f);
            }
            slot = slot == D ? 0 : slot + 1;
        }
    }

    // the K splits' partial tiles meet in LDS; row tile i is summed and stored by split i % KH, the
    // partials added in split order
    if constexpr (KH > 1) {
        stage_barrier();
        v4i *red = (v4i *)smem;
        const int grp = rg * NCG + cg;
#pragma unroll
        for (int i = 0; i < TM; i++)
            if (i % KH != kh) {
#pragma unroll
                for (int j = 0; j < TN; j++)
                    red[(((grp * KH + kh) * TM + i) * TN + j) * 64 + lane] = __builtin_bit_cast(v4i, acc[i][j]);
            }
        stage_barrier();
#pragma unroll
        for (int i = 0; i < TM; i++)
            if (i % KH == kh) {
#pragma unroll
                for (int j = 0; j < TN; j++) {
                    const Acc own = acc[i][j];
                    Acc s{};
#pragma unroll
                    for (int h = 0; h < KH; h++) {
                        const Acc p = h == kh ? own
                                              : __builtin_bit_cast(Acc, red[(((grp * KH + h) * TM + i) * TN + j) * 64 + lane]);
                        s = h == 0 ? p : s + p;
                    }
                    acc[i][j] = s;
                }
            }
    }

    // lane: output row 16 i + (lane & 15) of the wave's rows, columns 4 (lane >> 4) + 0..3 of tile j
    auto finish = [&](auto outc, auto widec) {
        constexpr int OUT = decltype(outc)::value;
        constexpr bool WIDE = decltype(widec)::value;   // the 16-bit output's value stored as fp32
#pragma unroll
        for (int j = 0; j < TO; j++) {
            const int n = n0 + (cg * TO + j) * 16 + 4 * fs;
            if (n >= NO) continue;
            // the operands of the lane's 4 columns (gated: then of their up columns)
            float ws[NG][4], bs[NG][4];
#pragma unroll
            for (int g = 0; g < NG; g++) {
                const int wr = (cg * TN + j + g * TO) * 16 + 4 * fs;
                const v4i wv = *(const v4i *)(ops + C::BM + wr), bv = *(const v4i *)(ops + C::BM + C::BN + wr);
#pragma unroll
                for (int c = 0; c < 4; c++) {
                    ws[g][c] = __int_as_float(wv[c]);
                    bs[g][c] = ep.bias ? bias_word((uint32_t)bv[c], ep.bias_dtype) : 0.0f;
                }
            }
#pragma unroll
            for (int i = 0; i < TM; i++) {
                const int m = mb + 16 * i + fr;
                if ((KH > 1 && i % KH != kh) || m >= M) continue;
                const float as = __uint_as_float(ops[rg * TM * 16 + 16 * i + fr]);
                float v[4];
#pragma unroll
                for (int c = 0; c < 4; c++) {
                    v[c] = __builtin_fmaf((float)acc[i][j][c], as * ws[0][c], bs[0][c]);
                    if constexpr (OUT == PSQ_BF16 || OUT == PSQ_F16) {
                        if (WIDE || act != ACT_NONE) v[c] = half_to_f32<OUT>(f32_to_half<OUT>(v[c]));
                    }
                    if constexpr (GATE) {
                        float u = __builtin_fmaf((float)acc[i][j + TO][c], as * ws[NG - 1][c], bs[NG - 1][c]);
                        if constexpr (OUT == PSQ_BF16 || OUT == PSQ_F16) u = half_to_f32<OUT>(f32_to_half<OUT>(u));
                        v[c] = silu(v[c]) * u;
                    } else if (act == ACT_GELU_TANH) {
                        v[c] = gelu_tanh(v[c]);
                    }
                }
                const int64_t o = (int64_t)m * ep.ldy + n;
                if constexpr (OUT == PSQ_F32 || WIDE) {
                    float *p = (float *)ep.y + o;
                    if (ep.vec && n + 4 <= NO) *(v4f *)p = v4f{v[0], v[1], v[2], v[3]};
                    else
#pragma unroll
                        for (int c = 0; c < 4; c++)
                            if (n + c < NO) p[c] = v[c];
                } else {
                    uint16_t *p = (uint16_t *)ep.y + o;
                    const uint32_t lo = pack_half2<OUT>(v[0], v[1]), hi = pack_half2<OUT>(v[2], v[3]);
                    if (ep.vec && n + 4 <= NO) *(v2i *)p = v2i{(int)lo, (int)hi};
                    else {
                        p[0] = (uint16_t)lo;
                        if (n + 1 < NO) p[1] = (uint16_t)(lo >> 16);
                        if (n + 2 < NO) p[2] = (uint16_t)hi;
                        if (n + 3 < NO) p[3] = (uint16_t)(hi >> 16);
                    }
                }
            }
        }
    };
    using BF = std::integral_constant<int, PSQ_BF16>;
    using HF = std::integral_constant<int, PSQ_F16>;
    if (out == PSQ_BF16) finish(BF{}, std::false_type{});
    else if (out == PSQ_F16) finish(HF{}, std::false_type{});
    else if (out == PSQ_F32) finish(std::integral_constant<int, PSQ_F32>{}, std::false_type{});
    else if constexpr (!GATE && KIND != 2) {
        if (out == Q8_WIDE_BF16) finish(BF{}, std::true_type{});
        else finish(HF{}, std::true_type{});
    }
}

template <int KIND, int NW, int TM, int TN, int NRG, int NCG, int BUDGET, bool PIPE, bool GATE>
int launch_cfg(int out, int act, const Q8Args &x)
{
    using C = Cfg<NW, TM, TN, NRG, NCG, BUDGET>;
    auto kern = q8_small_kernel<KIND, NW, TM, TN, NRG, NCG, BUDGET, PIPE, GATE>;
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess) return set_error(PSQ_E_DEVICE, "%s: no device", x.name);
    static bool attr_set[64] = {};   // per device; the attribute is idempotent
    if (dev >= 64 || !attr_set[dev]) {
        if (hipFuncSetAttribute((const void *)kern, hipFuncAttributeMaxDynamicSharedMemorySize, C::SMEM) != hipSuccess)
            return set_error(PSQ_E_DEVICE, "%s: cannot reserve %d bytes of LDS", x.name, C::SMEM);
        if (dev < 64) attr_set[dev] = true;
    }
    const int64_t NO = GATE ? x.N / 2 : x.N, on = GATE ? C::BN / 2 : C::BN;
    const int64_t tiles = ((x.M + C::BM - 1) / C::BM) * ((NO + on - 1) / on);
    kern<<<dim3((unsigned)tiles), dim3(64 * NW), C::SMEM, x.st>>>(x.a, x.lda, x.w, x.ldw, (int)x.M, (int)x.N, (int)x.K, x.ep, out, act);
    return check_launch(x.name);
}

// The tile shapes: rows x W rows, the waves' split of them and of K, and whether a tile's fragments
// are double-buffered in registers (a wave computes enough per block to hide its LDS reads).  `wide`
// shapes leave room for two workgroups per CU.
struct Shape {
    int bm, bn;
    bool wide;
};
enum { T16x32, T32x64, T64x64, T80x64, T96x128, T128x128, T128x192, T256x128, NSHAPES };
constexpr Shape kShapes[NSHAPES] = {{16, 32, true},   {32, 64, true},    {64, 64, false},   {80, 64, false},
                                    {96, 128, false}, {128, 128, false}, {128, 192, false}, {256, 128, false}};
// the gate pairs W tiles inside a wave, so its narrow shapes hold two W tiles per wave
constexpr Shape kGateShapes[NSHAPES] = {{16, 64, true},   {32, 128, false},  {64, 128, false}, {0, 0, false},
                                        {96, 128, false}, {128, 128, false}, {0, 0, false},    {256, 128, false}};

// The cheapest shape whose tiles run in one round of workgroups, or -1 (the 256 x 256 tiles).
//
// One round costs (K / 128) c: c was measured at K = 5120 as (us per block) 0.09 / 0.14 for 16 x 32 on
// up to one / two workgroups per CU, 0.15 / 0.28 for 32 x 64, 0.20 for 64 x 64, 0.27 for 80 x 64, 0.47
// for 96 x 128, 0.50 for 128 x 128, 0.68 for 128 x 192 and 1.04 for 256 x 128, against 1.1 to 1.6 for a
// 256 x 256 tile: a smaller tile that still fits one round is always ahead.  With more than one round
// the big tile's reuse of LDS wins (2048 x 5120 x 5120: 53.4 us, in two rounds of 128 x 192 68.7 us).
// One or two row tiles of 16 rows are bound by the weight stream, whatever the number of rounds.
int pick_shape(bool gate, int64_t M, int64_t N, int cus)
{
    const Shape *sh = gate ? kGateShapes : kShapes;
    auto tiles = [&](int i) { return ((M + sh[i].bm - 1) / sh[i].bm) * ((N + sh[i].bn - 1) / sh[i].bn); };
    if (M <= 16) return T16x32;
    if (tiles(T16x32) <= 2 * cus) return T16x32;
    if (M <= 32 || tiles(T32x64) <= cus) return T32x64;
    if (tiles(T64x64) <= cus) return T64x64;
    if (sh[T80x64].bm && tiles(T80x64) <= cus) return T80x64;
    if (sh[T32x64].wide && tiles(T32x64) <= 2 * cus) return T32x64;
    for (int i = T96x128; i < NSHAPES; i++)
        if (sh[i].bm && tiles(i) <= cus) return i;
    return -1;
}

template <int KIND>
int launch_shape(int shape, bool gate, int out, int act, const Q8Args &x)
{
    constexpr int KB = 1024;
#define PSQ_GO(...) return launch_cfg<KIND, __VA_ARGS__>(out, act, x)
    if (gate) {
        if constexpr (KIND != 2) {
            switch (shape) {
            case T16x32: PSQ_GO(8, 1, 2, 1, 2, 80 * KB, false, true);
            case T32x64: PSQ_GO(8, 2, 2, 1, 4, 156 * KB, false, true);
            case T64x64: PSQ_GO(8, 4, 2, 1, 4, 156 * KB, true, true);
            case T96x128: PSQ_GO(8, 3, 2, 2, 4, 156 * KB, true, true);
            case T128x128: PSQ_GO(8, 4, 2, 2, 4, 156 * KB, true, true);
            default: PSQ_GO(8, 4, 4, 4, 2, 156 * KB, true, true);
            }
        }
        return set_error(PSQ_E_ARG, "%s: no gate for these weights", x.name);
    }
    switch (shape) {
    case T16x32: PSQ_GO(8, 1, 1, 1, 2, 76 * KB, false, false);
    case T32x64: PSQ_GO(8, 2, 1, 1, 4, 76 * KB, false, false);
    case T64x64: PSQ_GO(8, 4, 1, 1, 4, 156 * KB, true, false);
    case T80x64: PSQ_GO(8, 5, 1, 1, 4, 156 * KB, true, false);
    case T96x128: PSQ_GO(8, 3, 2, 2, 4, 156 * KB, true, false);
    case T128x128: PSQ_GO(8, 4, 2, 2, 4, 156 * KB, true, false);
    case T128x192: PSQ_GO(8, 4, 3, 2, 4, 156 * KB, true, false);
    default: PSQ_GO(8, 4, 4, 4, 2, 156 * KB, true, false);
    }
#undef PSQ_GO
}

}  // namespace

bool q8_small(int kind, int out, int act, const Q8Args &x, int &status)
{
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess) return false;   // the caller's launch reports it
    const bool gate = act == ACT_SILU_GATE;
    const int shape = pick_shape(gate, x.M, x.N, cu_count(dev));
    if (shape < 0) return false;
    switch (kind) {
    case Q8_I8: status = launch_shape<0>(shape, gate, out, act, x); break;
    case Q8_E4M3: status = launch_shape<1>(shape, gate, out, act, x); break;
    default: status = launch_shape<2>(shape, gate, out, act, x); break;
    }
    return true;
}

}  // namespace psq
