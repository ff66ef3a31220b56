"""The launchers' choices on an MI355X's 256 CUs, on the host."""
import pytest

import dispatch as D
import test_gpu_gemm as G

LENGTHS = [1, 63, 64, 65, 512, 513, 1024, 1025, 1500, 3000, 6000, 12000, 16000, 16384, 16385, 20000, 32768, 70000,
           131071, 131072]


@pytest.mark.parametrize("nh,nkv", [(1, 1), (8, 1), (16, 1), (8, 2), (14, 2), (28, 4), (32, 8), (40, 8), (128, 8),
                                    (32, 32), (20, 1)])
def test_attention_stream_plan(nh, nkv):
    """Every tile in one split and the splits even, as many as the workspace is
    sized for past 1024 rows; every query head in one wave's group; whole groups
    of waves; and, over several splits, the head groups of a key/value head on one XCD
    (workgroup number mod 8)."""
    per = nh // nkv
    for split in (False, True):
        for length in LENGTHS:
            p = D.attention_stream_plan(nh, nkv, length, split)
            tiles = -(-length // 64)
            assert p["splits"] * p["tiles"] + p["more"] == tiles and p["more"] < p["splits"] and p["tiles"] >= 1
            want = D.lib().attention_splits(length) if split and length > 1024 else 1
            assert p["splits"] == want, (length, p)
            if split and length > 63 * 256:
                assert p["splits"] == 64, (length, p)
            assert p["splits"] <= p["gx"] < p["splits"] + 8
            assert p["waves"] % p["hgw"] == 0 and 0 < p["waves"] <= 8
            groups = -(-per // p["gb"])
            assert p["gy"] == nkv * -(-groups // p["hgw"]), (length, p)
            heads = [y // nkv * p["hgw"] * p["gb"] + w * p["gb"] for y in range(0, p["gy"], nkv)
                     for w in range(p["hgw"])]
            assert sorted(h for h in heads if h < per) == list(range(0, per, p["gb"])), (length, p)
            if p["splits"] > 1:
                for s in range(p["splits"]):
                    for g in range(nkv):
                        assert len({(s + p["gx"] * y) % 8 for y in range(g, p["gy"], nkv)}) == 1, (length, p)


@pytest.mark.parametrize("M,N,K,form", [
    # The clamped-row kernel where it is ahead of the wide forms: two 128 x 128
    # workgroups on a CU, and 256 x 128 for short M over long K.
    (271, 19624, 3328, "rows 128x128"), (560, 11144, 4864, "rows 128x128"), (324, 20696, 3968, "rows 128x128"),
    (136, 25912, 10752, "rows 256x128"),
    # Beside them, and on whole tiles, the wide forms.
    (1000, 5120, 5120, "wide 128x160"), (1000, 27648, 5120, "wide mixed"), (322, 16384, 1536, "wide 256x128"),
    (1024, 1024, 5120, "wide 64x64"), (1024, 5120, 5120, "wide 128x160"), (1024, 27648, 5120, "wide mixed"),
    (256, 19456, 3328, "wide 128x160"), (1773, 3784, 640, "wide 256x128"), (512, 11264, 4864, "wide 256x128"),
])
def test_fp8_forms(M, N, K, form):
    assert D.fp8_form(M, N, K) == form
    assert D.fp8_form(M, N, K, aligned=False).startswith("rows")


@pytest.mark.parametrize("M,N,K,form", G.FP8_WIDE + G.FP8_RAGGED)
def test_fp8_test_shapes_run_the_forms_they_name(M, N, K, form):
    assert D.fp8_form(M, N, K) == form
    assert M % 64 == 0 and N % 64 == 0 if (M, N, K, form) in G.FP8_WIDE else M % 64 != 0 or N % 64 != 0


def test_fp8_test_shapes_run_every_wide_form():
    wide = {f for f in D.FP8_FORMS if f.startswith("wide")}
    assert {c[3] for c in G.FP8_WIDE} == wide
    assert {c[3] for c in G.FP8_RAGGED} & wide == wide - {"wide 64x64"}


@pytest.mark.parametrize("M,N,K,fmt,form", G.W8A16_TILES + G.W8A16_STAGES_128 + G.W8A16_TAIL)
def test_w8a16_test_shapes_run_the_forms_they_name(M, N, K, fmt, form):
    assert D.w8a16_form(M, N, K) == form


def test_w8a16_test_shapes_run_every_form():
    """All six tiles whole and with a short last stage, and, of the three that
    have two stage widths, both."""
    six = set(D.W8A16_FORMS[:6])
    assert {c[4] for c in G.W8A16_TILES} == six and {c[4] for c in G.W8A16_TAIL} == six
    assert all(c[2] % 64 == 0 for c in G.W8A16_TILES) and all(c[2] % 64 for c in G.W8A16_TAIL)
    two = {"128x256", "64x128", "64x64"}
    assert {c[4] for c in G.W8A16_STAGES_128} == two and all(c[2] % 128 == 0 for c in G.W8A16_STAGES_128)
    assert two <= {c[4] for c in G.W8A16_TILES if c[2] % 128}
    assert D.w8a16_form(256, 2048, 8192) == D.w8a16_form(200, 1000, 8320) == "stream-K"
    assert D.w8a16_form(100, 3000, 4096) == "64 rows"


@pytest.mark.parametrize("M,N,K,form", [
    # Short K over many rounds, which a model fitted on long K priced too low.
    (780, 26741, 640, "128x256"), (895, 13283, 1024, "256x256"), (166, 19625, 4080, "128x160"),
    # The sizes in use, and few tiles over a K that no whole stage divides.
    (256, 4096, 4096, "64x64"), (256, 14336, 4096, "128x128"), (512, 5120, 5120, "128x128"),
    (1024, 5120, 5120, "128x160"), (1024, 27648, 5120, "256x256"), (1024, 5120, 27648, "128x160"),
    (256, 4096, 14336, "stream-K"), (86, 5636, 16944, "64 rows"), (70, 4000, 6160, "64 rows"),
])
def test_w8a16_forms(M, N, K, form):
    assert D.w8a16_form(M, N, K) == form
