"""Dequantize and the row-error statistics at the edges of their vector forms,
against the CPU oracle: widths around a unit (4 and 8 values), a wave and a
workgroup of units, widths that leave units crossing row ends, views that start
off a vector's alignment, every code (the reserved ones too), zero and tiny
weights, and scales past the fast division's range.

Dequantized values and the maxima are exact; the mean is an f64 sum in another
order, rounded once to f32 (2^-24 relative, held to 1e-6).
"""
import numpy as np
import pytest

import oracle as O
from helpers import E4M3, E5M2, bf16_bits

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

SHAPES = [(1, 1), (5, 3), (3, 7), (9, 8), (7, 9), (33, 64), (5, 511), (6, 1024), (5, 1031), (3, 8192), (4, 8195),
          (2, 20011), (300, 17), (2100, 40)]
# Past 2^19 values the expansion runs in units of 8 (bf16) or 4 codes, one a thread, and
# past 2^23 (2^21 for f32) four: widths of one unit, one value more, no multiple of a
# unit and wider than a workgroup's chunk.
UNIT_SHAPES = [(70000, 8), (60000, 9), (1100, 511), (513, 1031), (27, 20011), (1, 600000), (1030000, 9), (65000, 131),
               (300, 28001)]
# The statistics' forms: a weight or a unit of eight per lane, a wave or a workgroup
# per row, by the width (64, 128, 256, 1024) and by whether the rows pass 256.
ERR_SHAPES = [(256, 65), (257, 127), (300, 128), (257, 1023), (40, 200), (256, 256), (256, 257), (300, 1031)]


@pytest.fixture(scope="module")
def R():
    import reng_hip

    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    reng_hip.lib()
    return reng_hip


def dev(a, shift):
    """numpy -> device tensor that starts `shift` elements into its buffer."""
    a = np.ascontiguousarray(a)
    a = a.view(np.int16) if a.dtype == np.uint16 else a
    t = torch.empty(a.size + shift, dtype=torch.from_numpy(a[:1]).dtype, device="cuda")
    t[shift:] = torch.from_numpy(a)
    return t[shift:]


@pytest.mark.parametrize("fmt", [E4M3, E5M2])
@pytest.mark.parametrize("shift", [0, 1])
def test_dequantize_at_unit_edges(R, fmt, shift):
    rng = np.random.default_rng(5)
    for rows, cols in SHAPES + UNIT_SHAPES:
        codes = rng.integers(0, 256, rows * cols).astype(np.uint8)
        scales = np.exp2(rng.integers(-20, 20, rows)).astype(np.float32) * np.float32(1.37)
        want = O.Quantized(fmt, "pcs", rows, cols, codes, scales, 0).dequantize()
        q = R.Quantized(fmt, "pcs", rows, cols, dev(codes, shift), dev(scales, shift), 0)
        got = q.dequantize().cpu().numpy()
        nan = np.isnan(want)
        assert np.array_equal(np.isnan(got), nan), (rows, cols)
        assert np.array_equal(got[~nan].view(np.uint32), want[~nan].view(np.uint32)), (rows, cols)
        got = q.dequantize_bf16().cpu().numpy().view(np.uint16)
        assert np.array_equal(got, O.bf16_bits(want)), (rows, cols)


def weights(rng, rows, cols, kind):
    x = (rng.standard_normal((rows, cols)) * 0.02).astype(np.float32)
    if kind == "zeros":
        x[rng.random((rows, cols)) < 0.4] = 0.0
    if kind == "wide":   # magnitudes from the bf16 subnormals to past 2^60, each met by whatever code comes
        x = (x * np.exp2(rng.integers(-126, 100, (rows, cols))).astype(np.float32)).astype(np.float32)
    return bf16_bits(x).ravel()


@pytest.mark.parametrize("fmt", [E4M3, E5M2])
@pytest.mark.parametrize("kind", ["plain", "zeros", "wide", "reserved", "scales"])
@pytest.mark.parametrize("shift", [0, 1])
def test_row_errors_at_unit_edges(R, fmt, kind, shift):
    rng = np.random.default_rng(9)
    for rows, cols in SHAPES + ERR_SHAPES:
        w = weights(rng, rows, cols, kind)
        ref = O.quantize(w, rows, cols, fmt, "pcs" if kind != "wide" else "unit")
        if kind == "reserved":
            at = rng.integers(0, rows * cols, max(1, rows * cols // 50))
            ref.codes[at] = rng.integers(0, 256, at.size)
        if kind == "scales":
            ref.scales[:] = rng.choice(np.float32([0.0, -1.0, 1e-40, 2.0**43, 2.0**44, 3e38, np.inf, np.nan]), rows)
        q = R.Quantized(fmt, "pcs", rows, cols, dev(ref.codes, shift), dev(ref.scales, shift), 0)
        for n in (0, 3):
            got = R.row_errors(dev(w, shift), q) if n == 0 else R.sample_row_errors(dev(w, shift), q, n)
            with np.errstate(all="ignore"):
                want = O.row_errors(w, ref) if n == 0 else O.sample_row_errors(w, ref, n)
            mean, mx = (t.cpu().numpy() for t in got)
            assert np.array_equal(mx, want[1], equal_nan=True), (rows, cols)
            assert np.allclose(mean, want[0], rtol=1e-6, atol=0, equal_nan=True), (rows, cols)
