// fp8_forms.h - which kernel and tile the fp8 x fp8 GEMM (csrc/gemm_fp8.hip) runs
// a product on. Plain C++ so that the host tests can check the choice with the
// code the launcher runs.
#pragma once

#include <stdint.h>

namespace reng {

enum Fp8Form {
    FP8_WIDE_256x256,   // gemm_fp8_wide: 8 waves, 2 slots
    FP8_WIDE_256x128,   // 8 waves, 3 slots
    FP8_WIDE_128x160,   // 4 waves, 3 slots
    FP8_WIDE_128x128,   // 4 waves, 3 slots
    FP8_WIDE_64x64,     // 4 waves, 4 slots
    FP8_WIDE_MIXED,     // 256 x 256 over the leading n1 columns, then 256 x 192 (a second launch)
    FP8_ROWS_256x256,   // gemm_fp8_mfma (rows clamped at the edges)
    FP8_ROWS_256x128,
    FP8_ROWS_128x128,
    FP8_ROWS_64x64,
};

struct Fp8Pick {
    Fp8Form form;
    uint32_t n1;
};

inline uint64_t fp8_tiles(uint32_t M, uint32_t N, uint32_t bm, uint32_t bn) {
    return (uint64_t)((M + bm - 1) / bm) * ((N + bn - 1) / bn);
}

// Whether gemm_fp8_wide takes a product on bm x bn tiles: at least one tile each
// way, K in whole stages, byte offsets in 31 bits, 16-byte aligned output rows
// (of N, and of a wider output's stride, both multiples of 8).
inline bool fp8_wide_fits(uint32_t bm, uint32_t bn, uint32_t M, uint32_t N, uint32_t K, bool aligned) {
    return M >= bm && N >= bn && N % 8 == 0 && K % 128 == 0 && (uint64_t)M * K < (1ull << 31) &&
           (uint64_t)N * K < (1ull << 31) && aligned;
}

// A grid of 256 x 256 tiles that is not a whole number of rounds pays for its
// last, partial round in full. The mixed plan runs whole rounds of 256 x 256
// tiles over the leading n1 columns, then one round of 256 x 192 tiles over
// the rest (a second launch): on [1024, 27648, 5120] 252 + 240 tiles instead of
// 432 in two rounds. The narrower tile reads 0.875x the operand rows per output
// and its round measured 0.82-0.85x as long, so the plan gains 2-3% there
// (141-146 -> 138-141 us; K = 10240: 260-263 -> 253-254 us), not the 16% of a
// tile-count model: these tiles' rounds take time in proportion to the operand
// bytes they copy. (One launch holding both forms, the second's workgroups
// dispatched as the first's finish, measured the same as two launches.)
// n1 = 0: no plan. est takes the 256 x 256 form's (c0a, c1a) and the 256 x 192
// form's (c0b, c1b): 8.2, 1.353 fitted to timings at K = 2560, 5120 and 10240, and
// all four times 0.94 beside FP8_RAGGED, fitted with it.
struct Fp8MixedPlan {
    uint32_t n1;
    float est;
};

inline Fp8MixedPlan fp8_mixed_plan(uint32_t M, uint32_t N, uint32_t K, bool aligned, uint64_t cus, float c0a, float c1a,
                                   float c0b, float c1b) {
    Fp8MixedPlan best{0, 0.0f};
    if (M < 256 || N % 8 != 0 || K % 128 != 0) return best;
    const uint64_t tiles_m = (M + 255) / 256, stages = K / 128;
    const uint64_t rounds_a = tiles_m * (N / 256) / cus;   // whole rounds of the 256 x 256 tiles
    for (uint64_t r = 1; r <= rounds_a; ++r) {
        const uint64_t amax = r * cus / tiles_m;
        for (uint64_t a = amax; a + 3 > amax && a > 0; --a) {
            if (a * 256 >= N) continue;
            const uint32_t n1 = (uint32_t)(a * 256), rest = N - n1;
            if (rest < 192 || tiles_m * ((rest + 191) / 192) > cus) continue;
            if (!fp8_wide_fits(256, 256, M, n1, K, aligned) || !fp8_wide_fits(256, 192, M, rest, K, aligned)) continue;
            const float est = (float)((tiles_m * a + cus - 1) / cus) * (c0a + c1a * (float)stages) +
                              (c0b + c1b * (float)stages);
            if (best.n1 == 0 || est < best.est) best = Fp8MixedPlan{n1, est};
        }
    }
    return best;
}

// Where a wide tile fits, each form's time is modelled as rounds x (c0 + c1 x
// stages), rounds = ceil(tiles / (CUs x workgroups per CU)), stages = K / 128, and
// the cheapest form runs. There are two sets of (c0, c1), in microseconds.
//
// FP8_WHOLE chooses among the wide forms and stands where its choice divides the
// product. It is fitted to timings of every form on eleven products (M 256-2048, N
// 1024-27648, K 4096-27648): on those the choice is the fastest form measured.
//
// FP8_RAGGED chooses elsewhere, where tiles at the edge move back (against the
// clamped-row kernel [1000, 27648, 5120] 172 -> 134 us, [1000, 5120, 5120] 36.5 ->
// 29.5) and the clamped-row kernel can be ahead: 128 x 128 with two workgroups on
// a CU, where that makes one round of two ([271, 19624, 3328] 34.8 us against the
// wide forms' 40.2, [560, 11144, 4864] 42.6 against 51), 256 x 128 for short M
// over long K ([136, 25912, 10752] 84 against 113), and 64 x 64 where that tile
// does not divide the product ([100, 14336, 4096] 21.2 against 22.6, [130, 1000,
// 16384] 24.4 against 26.8). It is fitted to graph-replayed timings of every form
// on 436 such products (M 65-8192, N 512-28672, K 128-16384) and moved to where
// the choices cost least. On 188 others the choice is 1.0% over the fastest form
// in the mean. FP8_WHOLE, which prices short K 20-50% too high, is 4.5% over there
// and was up to 11% slower than the clamped-row kernel ([533, 13016, 896] 16.7 ->
// 18.6, now 16.5). Over 900 random products, two thirds of them ragged, timed in
// turn: 3.0% faster than with FP8_WHOLE alone, 12.4% than with the clamped-row
// kernel for every ragged one, two slower than with that, by 8 and 9% ([172, 27400,
// 9088] 79.9 -> 86.4). Below 128 either way only 64 x 64 tiles fit, and the choice
// by tile count stands.
struct Fp8Cost {
    Fp8Form form;
    uint32_t bm, bn, per_cu;
    float c0, c1;
};
constexpr Fp8Cost FP8_WHOLE[] = {
    {FP8_WIDE_256x256, 256, 256, 1, 16.2f, 1.318f}, {FP8_WIDE_256x128, 256, 128, 1, 12.2f, 0.739f},
    {FP8_WIDE_128x160, 128, 160, 1, 8.6f, 0.658f},  {FP8_WIDE_128x128, 128, 128, 1, 6.5f, 0.550f},
    {FP8_WIDE_64x64, 64, 64, 1, 1.1f, 0.246f},
};
constexpr Fp8Cost FP8_RAGGED[] = {
    {FP8_WIDE_256x256, 256, 256, 1, 11.0f, 1.291f}, {FP8_WIDE_256x128, 256, 128, 1, 7.5f, 0.716f},
    {FP8_WIDE_128x160, 128, 160, 1, 7.5f, 0.593f},  {FP8_WIDE_128x128, 128, 128, 1, 5.5f, 0.565f},
    {FP8_WIDE_64x64, 64, 64, 1, 1.9f, 0.286f},      {FP8_ROWS_256x128, 256, 128, 1, 14.9f, 0.839f},
    {FP8_ROWS_128x128, 128, 128, 2, 11.2f, 0.888f}, {FP8_ROWS_64x64, 64, 64, 1, 2.2f, 0.276f},
};

// The cheapest form that fits, null if none does. Of FP8_RAGGED's two 64 x 64 forms
// the wide one is for products it divides; two workgroups on a CU are priced for
// more tiles than CUs only.
template <size_t L>
inline const Fp8Cost *fp8_cheapest(const Fp8Cost (&costs)[L], uint32_t M, uint32_t N, uint32_t K, bool aligned,
                                   uint64_t cus, float *best) {
    const bool both64 = costs[L - 1].form == FP8_ROWS_64x64;
    const Fp8Cost *pick = nullptr;
    for (const Fp8Cost &c : costs) {
        const bool wide = c.form <= FP8_WIDE_64x64;
        const uint64_t tiles = fp8_tiles(M, N, c.bm, c.bn), at_once = cus * c.per_cu;
        if (wide && !fp8_wide_fits(c.bm, c.bn, M, N, K, aligned)) continue;
        if (both64 && c.bm == 64 && wide != (M % 64 == 0 && N % 64 == 0)) continue;
        if (tiles <= at_once - cus) continue;
        const float est = (float)((tiles + at_once - 1) / at_once) * (c.c0 + c.c1 * (float)(K / 128));
        if (!pick || est < *best) pick = &c, *best = est;
    }
    return pick;
}

inline Fp8Pick fp8_pick(uint32_t M, uint32_t N, uint32_t K, bool aligned, uint64_t cus) {
    float best = 0.0f;
    if (const Fp8Cost *pick = fp8_cheapest(FP8_WHOLE, M, N, K, aligned, cus, &best)) {
        Fp8MixedPlan mp = fp8_mixed_plan(M, N, K, aligned, cus, 16.2f, 1.318f, 8.2f, 1.353f);
        if (mp.n1 != 0 && mp.est < best) {
            if (M % 256 == 0 && N % 64 == 0) return {FP8_WIDE_MIXED, mp.n1};
        } else if (M % pick->bm == 0 && N % pick->bn == 0) {
            return {pick->form, 0};
        }
        if (fp8_wide_fits(128, 128, M, N, K, aligned)) {
            pick = fp8_cheapest(FP8_RAGGED, M, N, K, aligned, cus, &best);
            mp = fp8_mixed_plan(M, N, K, aligned, cus, 15.3f, 1.241f, 7.7f, 1.274f);
            if (mp.n1 != 0 && mp.est < best) return {FP8_WIDE_MIXED, mp.n1};
            return {pick->form, 0};
        }
    }
    const uint64_t t128 = fp8_tiles(M, N, 128, 128);
    // Everything else on the clamped-row kernel, by how many tiles each size gives
    // for the chip (measured on the M = 1024 prefill shapes): the largest tile that
    // still fills every CU; 256 x 128 for long K; 64 x 64 for small outputs.
    if (fp8_tiles(M, N, 256, 256) >= cus) return {FP8_ROWS_256x256, 0};
    if (t128 >= cus) return {K > 8192 ? FP8_ROWS_256x128 : FP8_ROWS_128x128, 0};
    if (K > 8192 && 2 * t128 >= cus) return {FP8_ROWS_256x128, 0};
    return {FP8_ROWS_64x64, 0};
}

}  // namespace reng
