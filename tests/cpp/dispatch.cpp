// The launchers' choices (plain C++ headers of reciprocating-engine_amd/csrc)
// for tests/test_dispatch.py and for the GPU tests that name a kernel form.
#include "../../reciprocating-engine_amd/csrc/attention_plan.h"
#include "../../reciprocating-engine_amd/csrc/fp8_forms.h"
#include "../../reciprocating-engine_amd/csrc/tile_forms.h"

using namespace reng;

// out: splits, tiles, more; gb, hgw, waves, gx, gy.
extern "C" void attention_stream_plan(size_t nh, size_t nkv, size_t len, int split, size_t cus, uint32_t *out) {
    const StreamSplit sp = stream_split(attn_plan(len, split != 0).splits, len);
    const StreamLaunch l = stream_launch(sp, nh, nkv, cus);
    const uint32_t v[] = {sp.splits, sp.tiles, sp.more, l.gb, l.hgw, l.waves, l.gx, l.gy};
    for (int i = 0; i < 8; ++i) out[i] = v[i];
}

extern "C" uint32_t attention_splits(size_t len) { return attn_plan(len, true).splits; }

extern "C" int fp8_form(uint32_t M, uint32_t N, uint32_t K, int aligned, uint64_t cus) {
    return fp8_pick(M, N, K, aligned != 0, cus).form;
}

// -2: the 64-row kernels; -1: stream-K on 128 x 128 tiles.
extern "C" int w8a16_form(uint32_t M, uint32_t N, uint32_t K, uint64_t cus) {
    if (!tiles::tiles_take(M, N, K, cus)) return -2;
    return tiles::streamk_suits(M, N, K, cus) ? -1 : (int)tiles::tile_pick(M, N, K, cus).form;
}
