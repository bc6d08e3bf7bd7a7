// wonly_plan.hpp -- launch plan of the tiled weight-only kernel (gemm_wonly.hip) and the workspace it
// needs.  Host arithmetic only, without HIP, so that a CPU build can check it.
#pragma once

#include <stdint.h>

#include <algorithm>

#include "../../../include/psquant.h"

namespace psq {

enum { W_UINT4 = 0, W_INT8 = 1 };
constexpr int kPlanBN = 256, kPlanBK = 64;                  // columns of a tile, elements of K per stage

// Launch plan of the tiled kernel, in units of one 128-row tile's K stage on a lightly loaded GPU.
//  * Data-parallel (one tile per workgroup): ceil(tiles / CUs) rounds of nk stages.  Tiles are 128,
//    160, 192, 224 or 256 rows; a stage of theirs costs kRows[] of a 128-row one's (the
//    dequantization serves all the rows: us a stage on 100 CUs, uint4, 0.86, 0.97, 1.02, 1.15, 1.25).
//    The width in rows is the cheapest over the rounds it takes, so that a ragged M does not compute
//    a mostly empty row tile: 300 x 25600 x 5120 125.1 us with two 256-row tiles, 93.0 with two of 160;
//    384 x 25600 x 5120 127.5 -> 104.8 (192); 2048 x 25600 x 5120 529 -> 503 (224); f16 on int8 weights
//    2048 x 5120 x 5120 109.2 -> 100.3 (192).
//  * Stream-K, 128-row tiles only (the 256-row kernel has no registers to spare for it), over G
//    workgroups: ceil(tiles nk / G) stages each.  With G a multiple s of the tiles, each workgroup
//    takes one K range of one tile (one partial, written or added up); otherwise up to two
//    segments (a second ring prologue, two partials).  Each partial costs about kSkPartCost.
//  * The kernel is power-limited: with more than about 78% of the CUs busy the clock drops, a
//    stage taking about 1 + 0.6 (busy fraction - 0.78) times as long (M=128 x N=25600: 1.13 us a
//    stage on 200 CUs, 1.2-1.37 on 256).
// Stream-K is taken when it beats data-parallel by more than kSkMargin, and needs a workspace:
// the tiles' arrival counters (kSkCntBytes, room for kSkMaxTiles) and two fp32 partial tiles per
// workgroup.  f16 on int8 weights has so little dequantization that its stages are short beside the
// partials: there the same split is taken when it saves kSkF16I8 stages (one K range of one tile per
// workgroup) or kSkF16I8Runs (runs across tiles).  Measured (us, whole tiles against the split, over 150
// shapes the two meet at these savings): 8 stages saved, 679 x 4096 x 1024 15.4 / 20.6; 24, 202 x 1137 x
// 2048 31.7 / 28.0; runs, 19, 1024 x 5120 x 5120 55.8 / 58.1; 26, 383 x 14336 x 6656 85.1 / 78.2; 81, 827 x
// 5120 x 13824 141.7 / 122.6.
constexpr int kSkMinUnits = 8;                              // K stages per workgroup at least
constexpr double kSkPartCost = 3.0, kSkRestartCost = 2.0, kSkMargin = 0.9;
constexpr struct {
    int bm;
    double cost;
} kRows[] = {{128, 1.0}, {160, 1.10}, {192, 1.17}, {224, 1.32}, {256, 1.44}};
constexpr double kSkF16I8 = 17.0, kSkF16I8Runs = 28.0;
constexpr int64_t kSkMaxTiles = 16384;
constexpr int64_t kSkCntBytes = kSkMaxTiles * 4;
constexpr int64_t kSkSlotBytes = 128LL * kPlanBN * 4;       // one 128-row fp32 partial tile
constexpr int kSkMaxGroups = 256;
constexpr int64_t kMaxWsBytes = kSkCntBytes + 2 * kSkMaxGroups * kSkSlotBytes;   // 64 MB + 64 KB

inline double clock_factor(int64_t busy, int cus)
{
    const double f = (double)busy / cus - 0.78;
    return f > 0 ? 1.0 + 0.6 * f : 1.0;
}

struct TiledPlan {
    int bm = 128;
    int64_t tiles = 0;
    int sk = 0;                 // stream-K workgroups (0: data-parallel)
    int64_t ws_bytes = 0;
};

// The plan of a call: weight kind wk, activations of x_dtype (PSQ_BF16 or PSQ_F16).
inline TiledPlan plan_tiled(int wk, int x_dtype, int64_t M, int64_t N, int64_t K, int cus, bool allow_sk)
{
    TiledPlan p;
    const int64_t nbn = (N + kPlanBN - 1) / kPlanBN, nk = K / kPlanBK;
    double t_dp = 0.0;
    for (const auto &r : kRows) {
        const int64_t tiles = ((M + r.bm - 1) / r.bm) * nbn;
        const double t = (double)((tiles + cus - 1) / cus * nk) * r.cost * clock_factor(std::min<int64_t>(tiles, cus), cus);
        if (p.tiles && t >= t_dp) continue;
        t_dp = t;
        p.bm = r.bm;
        p.tiles = tiles;
    }
    if (!allow_sk) return p;
    const int64_t t128 = ((M + 127) / 128) * nbn, units = t128 * nk;
    if (t128 > kSkMaxTiles) return p;
    double best = 1e300, saved = 0.0;
    int64_t best_g = 0;
    bool runs = false;
    auto consider = [&](int64_t g, bool aligned) {
        if (g < 1 || g > cus || g > kSkMaxGroups || units / g < kSkMinUnits) return;
        const double stages = (double)((units + g - 1) / g) * clock_factor(g, cus);
        const double t = stages + (aligned ? kSkPartCost : 2 * kSkPartCost + kSkRestartCost);
        if (t < best) {
            best = t;
            saved = t_dp - stages;
            runs = !aligned;
            best_g = g;
        }
    };
    for (int64_t sp = 2; t128 * sp <= cus; sp++) consider(t128 * sp, true);   // one K range of one tile each
    consider(cus, false);
    const bool pays = wk == W_INT8 && x_dtype == PSQ_F16 ? saved > (runs ? kSkF16I8Runs : kSkF16I8) : true;
    if (best_g && best < kSkMargin * t_dp && pays) {
        p.bm = 128;
        p.tiles = t128;
        p.sk = (int)best_g;
        p.ws_bytes = kSkCntBytes + 2 * best_g * kSkSlotBytes;
    }
    return p;
}

// Workspace that covers a call of either activation type: the query knows the shape alone (f16 on int8
// weights runs whole tiles where bf16 splits 1024 x 5120 x 5120).
inline int64_t plan_workspace(int wk, int64_t M, int64_t N, int64_t K, int cus)
{
    return std::max(plan_tiled(wk, PSQ_BF16, M, N, K, cus, true).ws_bytes,
                    plan_tiled(wk, PSQ_F16, M, N, K, cus, true).ws_bytes);
}

}  // namespace psq
