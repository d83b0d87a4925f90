// sh_gemm_plan.hpp — which kernel a matrix product runs on, from its sizes alone (host code only).
#pragma once

#include <math.h>

#include <algorithm>

namespace sh {

// A product that the large tiles take whatever else: long inputs, and the classifier's very wide
// output from 256 rows on.
inline bool gemm_big(int M, int N) { return (M >= 1024 || (M >= 256 && N >= 16384)) && N % 128 == 0; }

// Whether a forward that may take its fp16 activations as one plane (EvalLogits) does so in this
// product. The shortest K keep the hi/lo pair, as they always have: it costs them next to nothing
// (the bytes of a second plane of 64 to 192 columns), and dropping it raises the product's error from
// about 1e-6 to 2e-4.
inline bool gemm_one_plane(int M, int N, int K) { return gemm_big(M, N) ? K % 128 == 0 : K >= 192; }

// Kernel, tile shape and K split of a 16-bit GEMM: the least of the candidates' estimated times.
// Fitted to sweeps over M = 33 .. 32736, N = 768 .. 32000, K = 768 .. 3072 (in us; two planes,
// then one plane):
//  - k_gemm_ring: its tiles run in rounds of 256 (two workgroups share a CU, but then each takes
//    twice as long), a K step of 32 costing 0.75 / 0.40 for 128 x 256 tiles, 0.48 / 0.26 for
//    128 x 128, 0.28 for 64 x 128 (two planes only) and 0.24 / 0.16 for 64 x 64 tiles.
//  - k_gemm_pipe on 32 x 32 tiles, K split in two or four until there are about 384 workgroups:
//    2.3 + 6.3e-4 / 4.1e-4 per tile and K step of 64. It keeps the short inputs' narrow products
//    (256 x 768 x 2048: 6.6 in two ranges against 17.4 for 64 x 64 ring tiles); from about 400
//    rows x 2304 columns on the ring wins (600 x 4096 x 1024: 18.0 against 29.5 for the 64 x 64
//    pipelined tiles that such products used to take; 173 x 6144 x 1024: 11.5 against 20.0).
//  - k_gemm_ring on 32 x 64 tiles with K split alike, where K is not a multiple of 64.
// (256 x 256 tiles equal 128 x 256 on the largest products and lose elsewhere.)
enum { GK_PIPE32 = 0, GK_RING128x256, GK_RING128x128, GK_RING64x128, GK_RING64x64, GK_RING32x64 };
struct GemmPlan {
    int kind, ranges, kc;
    int run;   // K steps of 32 that are added into one sum before it joins the total; 0: all of them
};
inline GemmPlan gemm_plan(int M, int N, int K, bool one_plane, bool bf16) {
    GemmPlan p{GK_RING64x64, 1, K, 0};
    float best = INFINITY;
    const auto tiles = [&](int bm, int bn) { return ((M + bm - 1) / bm) * (N / bn); };
    const auto ring = [&](int kind, int bm, int bn, float step, float base) {
        if (N % bn) return;
        const float t = base + step * (K / 32) * ((tiles(bm, bn) + 255) / 256);
        if (t < best) {
            best = t;
            p.kind = kind;
        }
    };
    // For want of tiles some products were split into K ranges by the kernels before these (large ones,
    // and those of K not a multiple of 64), each range with one sum of both planes' products.
    const int t = gemm_big(M, N) ? tiles(128, 128) : tiles(64, 64);
    int before = 1;
    if (!one_plane && !bf16 && t < 512 && (gemm_big(M, N) || K % 64))
        for (int r : {2, 3, 4})
            if (K % (32 * r) == 0 && K / r >= 256 && t * r <= 768) before = r;
    // These tiles' registers hold one sum per result, so a pair's lo products are added into the hi
    // products' sums: large products only, which never had two. Others keep sums of their own, at 64.7
    // us against 62.3 and an error of 2.9e-7 against 4.1e-7 for 700 x 6144 x 2048 (193 x 32000 x 768:
    // 37.0 against 34.4 us, 1.9e-7 against 2.6e-7).
    if (one_plane || (gemm_big(M, N) && before == 1))
        ring(GK_RING128x256, 128, 256, one_plane ? 0.40f : 0.75f, one_plane ? 6.3f : 7.0f);
    ring(GK_RING128x128, 128, 128, one_plane ? 0.26f : 0.48f, one_plane ? 4.0f : 4.5f);
    if (!one_plane) ring(GK_RING64x128, 64, 128, 0.28f, 3.0f);
    ring(GK_RING64x64, 64, 64, one_plane ? 0.16f : 0.24f, 2.4f);
    // splitting K leaves a partial per range for the next kernel to add: four at most
    const bool pipe = K % 64 == 0 && K / 64 >= 3;
    if (!pipe && one_plane) return p;
    const int unit = pipe ? 64 : 32, t32 = tiles(32, pipe ? 32 : 64), steps = K / unit;
    int ranges = 1;
    for (int r : {2, 4}) {
        if (t32 * ranges >= 384) break;
        if (pipe ? steps % r == 0 && steps / r >= 3 : steps / r >= 6) ranges = r;
    }
    const int per = (steps + ranges - 1) / ranges;   // K steps per range
    if (2.3f + per * std::max(t32 * ranges, 300) * (one_plane ? 4.1e-4f : 6.3e-4f) < best)
        p = GemmPlan{pipe ? GK_PIPE32 : GK_RING32x64, (steps + per - 1) / per, per * unit, 0};
    // As fp16 pairs such products keep sums no longer than those: where one plane's K steps are more, 512
    // of K at a time. 1100 x 1024 x 2048: relative error 1.6e-7, against 2.9e-7 in one sum and 2.2e-7 in
    // the four ranges before (29.8 -> 31.9 us); 1024 x 768 x 768 12.5 -> 13.1 us, 25.0 in ranges; 300 x
    // 2560 x 2016 1.6e-7 against 2.9e-7 and 2.4e-7, 24.2 -> 27.2 us, 27.5 in ranges. A bf16 pair's own
    // 1e-6 hides the sum's error.
    if (before > 1 && p.kc / 32 > 2 * (K / 32) / before) p.run = 16;
    return p;
}

constexpr int kLsRows = 32;   // rows of a k_linear_few workgroup
// Where k_linear_few's one launch beats the planes, GEMM and range-sum launches (us, measured on
// in x out = 256 x 256 to 2048 x 4096): always up to 16 rows (3.5 to 7.8 against 6.3 to 9.3), and
// in one round of workgroups while K leaves each wave few steps (128 x 768 x 768: 6.4 against
// 9.0; 32 x 4096 x 1024: 6.8 against 8.6; but 32 x 1088 x 2016: 10.2 against 9.8, and 48 x 4096 x
// 1024, two rounds: 9.3 against 9.4). Larger weights than were measured keep the tiled products.
inline bool linear_few(int M, int N, int K, bool cf) {
    if (cf || N > 4096 || K > 4096) return false;
    return M <= 16 || (K <= 1536 && (N / 16) * ((M + kLsRows - 1) / kLsRows) <= 256);
}

}  // namespace sh
