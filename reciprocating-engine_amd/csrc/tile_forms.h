// tile_forms.h - which output tile the w8a16 product for more than 64 activation
// rows (csrc/gemm_tiles.hip) runs on, and which products it takes. Plain C++ so
// that the host tests can check the choice with the code the launcher runs.
#pragma once

#include <stdint.h>

namespace reng {

namespace tiles {

inline uint64_t tile_count(uint32_t M, uint32_t N, uint32_t bm, uint32_t bn) {
    return (uint64_t)((M + bm - 1) / bm) * ((N + bn - 1) / bn);
}

// Long K (at least 64 stages of 128 codes) over fewer 128 x 128 tiles than
// half the CUs: one tile per block would leave most of the chip idle.
inline bool streamk_suits(uint32_t M, uint32_t N, uint32_t K, uint64_t cus) {
    return K % 128 == 0 && K >= 8192 && 2 * tile_count(M, N, 128, 128) < cus;
}

// Tile choice. Long K (K >= 8192) over fewer 128 x 128 tiles than half the
// CUs runs stream-K on 128 x 128 tiles of 128-code stages (M = 256
// [4096, 14336]: 92.8 -> 66.5 us). Otherwise each form's time is modelled as
// rounds x (c0 + c1 x K / 64), rounds = ceil(tiles / CUs), and the cheapest form
// runs. (c0, c1), in microseconds, are fitted to graph-replayed timings of every
// form on 655 random products (M 65-1024, N 400-27648, K 64-20000) and moved to
// where the picks cost least: one set for K % 128 = 0 and one for the 64-code stages
// and short last stages of any other K. On a quarter of the products kept out of the
// fit the picks are 0.2% over the fastest form in the mean and 21% at worst. The
// constants before, one set from eleven products of K >= 4096, priced short K too low
// where a form takes many rounds (M = 780 [26741, 640] on 128 x 160 85 us, modelled
// 58, against 65 on 128 x 256): 5% over the fastest form for K % 128 = 0 and 3% for
// other K in the mean, 71% at worst. Stream-K takes
// (G + tiles - 1) BM BN floats of partials (6.3 Mi floats at most on 256
// CUs) and a counter per tile (fewer than 128).
enum TileForm { TILES_256x256, TILES_128x256, TILES_128x160, TILES_128x128, TILES_64x128, TILES_64x64 };

struct TilePick {
    TileForm form;
    float est;   // modelled microseconds
};

inline TilePick tile_pick(uint32_t M, uint32_t N, uint32_t K, uint64_t cus) {
    struct Cand {
        uint32_t bm, bn;
        float c0, c1;   // K % 128 == 0
        float d0, d1;   // any other K
    };
    const Cand cands[] = {
        {256, 256, 29.3f, 0.953f, 25.6f, 1.185f},   // 8 waves of 128 x 64, 64-code stages, 3 slots
        {128, 256, 12.3f, 0.761f, 12.3f, 0.764f},   // 8 waves of 64 x 64
        {128, 160, 13.9f, 0.629f, 13.2f, 0.629f},   // 4 waves of 32 x 160, 128-code stages, 2 slots: not K = 64 mod 128
        {128, 128, 8.0f, 0.456f, 8.4f, 0.422f},     // 8 waves of 64 x 32, 64-code stages, 6 slots
        {64, 128, 6.2f, 0.314f, 5.4f, 0.351f},      // 8 waves of 32 x 32
        {64, 64, 2.8f, 0.195f, 3.4f, 0.185f},       // 4 waves of 32 x 32
    };
    const bool whole = K % 128 == 0;
    TilePick best{TILES_256x256, 0.0f};
    for (int i = 0; i < 6; ++i) {
        if (i == TILES_128x160 && K % 128 == 64) continue;
        const uint64_t rounds = (tile_count(M, N, cands[i].bm, cands[i].bn) + cus - 1) / cus;
        const float c0 = whole ? cands[i].c0 : cands[i].d0, c1 = whole ? cands[i].c1 : cands[i].d1;
        const float est = (float)rounds * (c0 + c1 * (float)((K + 63) / 64));
        if (i == 0 || est < best.est) best = TilePick{(TileForm)i, est};
    }
    return best;
}

// K % 64 == 0: below half the CUs in 64 x 128 tiles the 64-row kernels, which
// split K, are faster (M = 100 [3000, 4096]: 22.2 against 28.1 us) - unless
// the product suits stream-K. K no multiple of 128: the 64-row launches, each
// about 6 us + N K / 2.9 TB/s there (M = 128 [14336, 4112] 25 us a launch,
// M = 300 [3000, 3600] 10, M = 700 [1500, 1296] 7.4), against the tiles' own
// model, 40% and more with K added for few tiles (M = 70 [4000, 6160]: tiles 30.8
// us, two launches 27.7; M = 86 [5636, 16944]: 83 and 68). M = 256 [4096, 4112] 54.1 ->
// 22.7 us, M = 300 [3000, 3600] 50.2 -> 20.7, M = 1000 [10000, 1552] 174 -> 51,
// M = 1024 [2048, 16400] 340 -> 105.
inline bool tiles_take(uint32_t M, uint32_t N, uint32_t K, uint64_t cus) {
    if (M <= 64) return false;
    if (K % 64 == 0 && (streamk_suits(M, N, K, cus) || 2 * tile_count(M, N, 64, 128) >= cus)) return true;
    if (K % 128 == 0) return false;
    const float loop = (float)((M + 63) / 64) * (6.0f + (float)N * (float)K / 2.9e6f);
    return (1.4f + (float)K / 128000.0f) * tile_pick(M, N, K, cus).est < loop;
}

}  // namespace tiles

}  // namespace reng
