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
// rounds x (c0 + c1 x K / 64), rounds = ceil(tiles / CUs), with (c0, c1) in
// microseconds fitted to graph-replayed timings of every form on eleven
// products (M 128-1024 over the Llama-3.1-8B and Qwen2.5-32B shapes; most
// within 16% of the fit), scaled per form to this pipeline's times (0.91-0.93;
// 256 x 256 and 64 x 64 1.06-1.08), and the cheapest form runs. On 22 products
// (M 80-1024, N 1200-28672, K 1024-10240) the picks were all faster than
// those of the earlier fit and pipeline, by 4-33% (M = 700 [3000, 2048] 25.5
// -> 17.3 us, M = 150 [25000, 1536] 31.0 -> 23.4). The constants of 128 x 256,
// 64 x 128 and 64 x 64 are those of 128-code stages; K = 64 mod 128 and the padded K
// run 64-code ones on them, and their picks are within 2 and 3% of the fastest form
// (70 random products each, the worst 22 and 26%; none slower than before the refit,
// the first kind 36% faster in the mean). Stream-K takes
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
        float c0, c1;
        bool fits;
    };
    const Cand cands[] = {
        {256, 256, 28.6f, 1.200f, true},                            // 8 waves of 128 x 64, 64-code stages, 3 slots
        {128, 256, 16.6f, 0.650f, true},                            // 8 waves of 64 x 64
        {128, 160, 5.2f, 0.650f, K % 64 != 0 || K % 128 == 0},      // 4 waves of 32 x 160, 128-code stages, 2 slots
        {128, 128, 9.3f, 0.425f, true},                             // 8 waves of 64 x 32, 64-code stages, 6 slots
        {64, 128, 4.6f, 0.318f, true},                              // 8 waves of 32 x 32
        {64, 64, 0.0f, 0.270f, true},                               // 4 waves of 32 x 32
    };
    TilePick best{TILES_256x256, 0.0f};
    for (int i = 0; i < 6; ++i) {
        if (!cands[i].fits) continue;
        const uint64_t rounds = (tile_count(M, N, cands[i].bm, cands[i].bn) + cus - 1) / cus;
        const float est = (float)rounds * (cands[i].c0 + cands[i].c1 * (float)((K + 63) / 64));
        if (i == 0 || est < best.est) best = TilePick{(TileForm)i, est};
    }
    return best;
}

// K % 64 == 0: below half the CUs in 64 x 128 tiles the 64-row kernels, which
// split K, are faster (M = 100 [3000, 4096]: 22.2 against 28.1 us) - unless
// the product suits stream-K. K no multiple of 128: the 64-row launches, each
// about 6 us + N K / 2.9 TB/s there (M = 128 [14336, 4112] 25 us a launch,
// M = 300 [3000, 3600] 10, M = 700 [1500, 1296] 7.4), against the tiles' own
// model, a quarter added for the short stage's checks and few tiles (M = 70
// [4000, 6160]: tiles 30.8 us, two launches 27.7). M = 256 [4096, 4112] 54.1 ->
// 22.7 us, M = 300 [3000, 3600] 50.2 -> 20.7, M = 1000 [10000, 1552] 174 -> 51,
// M = 1024 [2048, 16400] 340 -> 105.
inline bool tiles_take(uint32_t M, uint32_t N, uint32_t K, uint64_t cus) {
    if (M <= 64) return false;
    if (K % 64 == 0 && (streamk_suits(M, N, K, cus) || 2 * tile_count(M, N, 64, 128) >= cus)) return true;
    if (K % 128 == 0) return false;
    const float loop = (float)((M + 63) / 64) * (6.0f + (float)N * (float)K / 2.9e6f);
    return 1.25f * tile_pick(M, N, K, cus).est < loop;
}

}  // namespace tiles

}  // namespace reng
