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
// n1 = 0: no plan. est uses the 256 x 192 form's (c0, c1) fitted to its
// timings at K = 2560, 5120 and 10240.
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

// The wide forms, where at least a tile fits each way (ragged edges: the
// last tile moves back; same box against the clamped-row kernel [1000,
// 27648, 5120] 172 -> 134 us, [1000, 5120, 5120] 36.5 -> 29.5, [450, 20000,
// 1280] 28.2 -> 21.4, and against 64 x 64 tiles [1984, 4096, 4096] 71.5 ->
// 32.3). Each candidate's time is modelled as
// rounds x (c0 + c1 x stages), rounds = ceil(tiles / CUs), stages = K / 128,
// with (c0, c1) in microseconds fitted to timings of every form on eleven
// products (M 256-2048, N 1024-27648, K 4096-27648; shorter K is an
// extrapolation). Most timings lie within 10% of the fit, 64 x 64 and
// 256 x 128 up to 26% above it when their tiles take a single round. The
// cheapest form runs; on those products that is the fastest one measured.
//
// The clamped-row kernel has two forms that can be cheaper where the wide
// form's tiles do not divide the product: 128 x 128 with two workgroups on a CU,
// so that up to 512 tiles are one round ([271, 19624, 3328]: 34.8 us against the
// wide forms' 40.2; [560, 11144, 4864]: 42.6 against 51), and 256 x 128 where M is
// short and K long ([136, 25912, 10752]: 84 against 113). Their (c0, c1) are the
// upper side of a fit to 184 random products (M 65-2048), so that they are taken
// only where they are clearly ahead; below 8 stages the wide forms are faster than
// their model ([1773, 3784, 640] 256 x 128 13.4 us, modelled 15.9, against 15.3).
// On 220 other random products: 11.1% faster than the clamped-row kernel for every
// ragged one, none slower, against 10.5% and 13 of 184 up to 31% slower before.
inline Fp8Pick fp8_pick(uint32_t M, uint32_t N, uint32_t K, bool aligned, uint64_t cus) {
    struct Cand {
        Fp8Form form;
        uint32_t bm, bn;
        float c0, c1;
    };
    const Cand cands[] = {
        {FP8_WIDE_256x256, 256, 256, 16.2f, 1.318f}, {FP8_WIDE_256x128, 256, 128, 12.2f, 0.739f},
        {FP8_WIDE_128x160, 128, 160, 8.6f, 0.658f},  {FP8_WIDE_128x128, 128, 128, 6.5f, 0.550f},
        {FP8_WIDE_64x64, 64, 64, 1.1f, 0.246f},
    };
    const float stages = (float)(K / 128);
    const Cand *pick = nullptr;
    float best = 0.0f;
    for (const Cand &c : cands) {
        if (!fp8_wide_fits(c.bm, c.bn, M, N, K, aligned)) continue;
        const float est = (float)((fp8_tiles(M, N, c.bm, c.bn) + cus - 1) / cus) * (c.c0 + c.c1 * stages);
        if (!pick || est < best) pick = &c, best = est;
    }
    const uint64_t t256x128 = fp8_tiles(M, N, 256, 128), t128 = fp8_tiles(M, N, 128, 128);
    bool rows64 = false;
    Fp8Form form = pick ? pick->form : FP8_ROWS_64x64;
    if (pick && (M % pick->bm != 0 || N % pick->bn != 0)) {
        // Where 64 x 64 tiles are the cheapest, the clamped-row kernel is faster ([100,
        // 14336, 4096] 21.2 against 22.6 us, [130, 1000, 16384] 24.4 against 26.8).
        rows64 = pick->form == FP8_WIDE_64x64;
        const float e128 = (float)((t128 + 2 * cus - 1) / (2 * cus)) * (9.5f + 1.05f * stages);
        const float e256 = (float)((t256x128 + cus - 1) / cus) * (15.6f + 0.81f * stages);
        if (!rows64 && t128 > cus && stages >= 8.0f && e128 < best) form = FP8_ROWS_128x128, best = e128;
        if (!rows64 && e256 < best) form = FP8_ROWS_256x128, best = e256;
    }
    const Fp8MixedPlan mp = fp8_mixed_plan(M, N, K, aligned, cus, cands[0].c0, cands[0].c1, 8.2f, 1.353f);
    if (mp.n1 != 0 && (!pick || mp.est < best)) return {FP8_WIDE_MIXED, mp.n1};
    if (pick && !rows64) return {form, 0};
    // Everything else on the clamped-row kernel, by how many tiles each size gives
    // for the chip (measured on the M = 1024 prefill shapes): the largest tile that
    // still fills every CU; 256 x 128 for long K; 64 x 64 for small outputs.
    if (fp8_tiles(M, N, 256, 256) >= cus) return {FP8_ROWS_256x256, 0};
    if (t128 >= cus) return {K > 8192 ? FP8_ROWS_256x128 : FP8_ROWS_128x128, 0};
    if (K > 8192 && 2 * t128 >= cus) return {FP8_ROWS_256x128, 0};
    return {FP8_ROWS_64x64, 0};
}

}  // namespace reng
