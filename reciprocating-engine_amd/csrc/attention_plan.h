// attention_plan.h - how the decode attention (csrc/layer.hip) cuts a cache into
// splits and its heads into workgroups. Plain C++ so that the host tests can
// check the plans with the code the launcher runs.
#pragma once

#include <stddef.h>
#include <stdint.h>

namespace reng {

constexpr int ATT_SPLIT_MAX = 64, ATT_SPLIT_ROWS = 256, ATT_ONE_PASS_MAX = 512;

struct AttnPlan {
    uint32_t splits, chunk;
};

// One pass (S = 1) for caches of up to 512 rows or without a workspace; else
// S = min(64, ceil(len / 256)) splits of equal length (the last one shorter),
// none empty.
inline AttnPlan attn_plan(size_t len, bool split) {
    if (!split || len <= (size_t)ATT_ONE_PASS_MAX) return {1u, (uint32_t)len};
    size_t s = (len + ATT_SPLIT_ROWS - 1) / ATT_SPLIT_ROWS;
    if (s > (size_t)ATT_SPLIT_MAX) s = ATT_SPLIT_MAX;
    const size_t chunk = (len + s - 1) / s;
    return {(uint32_t)((len + chunk - 1) / chunk), (uint32_t)chunk};
}

constexpr int ATS_TILE = 64, ATS_WAVES = 8, ATS_ONE_PASS_MAX = 1024, ATS_XCDS = 8;

// The streaming kernel's splits: the first `more` take tiles + 1 tiles of
// ATS_TILE rows, the others `tiles`.
struct StreamSplit {
    uint32_t splits, tiles, more;
};

// attn_plan's splits (the workspace is theirs), each of whole tiles and none
// more than one tile longer than another: rounding every split up to whole tiles
// instead left 61-63 of 64, which the rules of stream_launch took for too few
// workgroups and which put head groups on different XCDs (8 heads on 2 of 128
// dimensions: 20000 rows 22.1 -> 13.4 us, 70000 rows 47.3 -> 23.7, where
// attention_split16 took 18.0 and 35.3; 16 on 1, 70000 rows: 49.3 -> 23.5 and
// 39.4; 28 on 4, 20000 rows: 28.4 -> 20.9 and 71). One pass up to 1024 rows, where the merge's launch costs more than the split saves (one pass /
// split, 32 heads on 8 of 128 dimensions: 7.1 / 9.1 us at 768 rows, 9.0 / 9.7 at
// 1024, 25 / 12 at 4096; 8 heads on 2 of 64: 6.5 / 8.2 at 1024).
inline StreamSplit stream_split(uint32_t splits, size_t len) {
    if (len <= (size_t)ATS_ONE_PASS_MAX) splits = 1;
    const uint32_t tiles = (uint32_t)((len + ATS_TILE - 1) / ATS_TILE);
    return {splits, tiles / splits, tiles % splits};
}

// The launch: gb query heads a wave, hgw groups of gb heads side by side in a
// workgroup of `waves` waves, gx workgroups along the splits and gy along the
// key/value heads and their remaining groups.
struct StreamLaunch {
    uint32_t gb, hgw, waves, gx, gy;
};

inline StreamLaunch stream_launch(const StreamSplit &sp, size_t nh, size_t nkv, size_t cus) {
    // Four heads a wave once that still gives every CU a workgroup: fewer heads
    // a wave read the rows again from L2, but short caches need the workgroups.
    // The head groups of one key/value head share a workgroup where the splits
    // alone fill the chip. Workgroups of four waves where two fit on every CU
    // (their 64 KB of keys each), else of eight.
    const size_t per_kv = nh / nkv, tiles = sp.tiles + (sp.more > 0);
    uint32_t gb = 4;
    while (gb > 1 && (gb / 2 >= per_kv || sp.splits * nkv * ((per_kv + gb - 1) / gb) < cus)) gb /= 2;
    const size_t hgroups = (per_kv + gb - 1) / gb;
    size_t hgw = 1, waves = ATS_WAVES;
    if (sp.splits * nkv >= cus && hgroups > 1) hgw = hgroups > 2 ? 4 : 2;
    else if (sp.splits * nkv * hgroups >= 2 * cus) waves = ATS_WAVES / 2;
    if (waves > tiles * hgw) waves = tiles * hgw;
    // Workgroups go to the XCDs in turn, x first, so the groups of one key/value
    // head run on one XCD, and its L2 gives them the rows after the first, if gx
    // times nkv is a multiple of the XCDs: up to seven empty workgroups a row of
    // the grid (8 heads on 2 of 128 dimensions, 12000 rows: 15.8 -> 12.8 us).
    size_t gx = sp.splits;
    while (sp.splits > 1 && hgroups > hgw && gx * nkv % ATS_XCDS != 0) ++gx;
    return {gb, (uint32_t)hgw, (uint32_t)waves, (uint32_t)gx, (uint32_t)(nkv * ((hgroups + hgw - 1) / hgw))};
}

}  // namespace reng
