"""The quantizer's any-width, any-alignment rows and the hardware-bias scheme's
tensor maximum, bit for bit against the CPU oracle: widths around a vector (4 f32,
8 bf16), a wave and the register-resident limit, buffers that start off a
vector's alignment, odd row pitches, a maximum (or NaN, inf) in the last element
of the last row, and maxima that select each hardware bias.
"""
import numpy as np
import pytest

import oracle as O
from helpers import E4M3, E5M2, bf16_bits

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


@pytest.fixture(scope="module")
def R():
    import reng_hip

    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    reng_hip.lib()
    return reng_hip


def check(R, x, rows, cols, ld, dtype, fmt, scaling, shift):
    """Quantize the first cols of each ld-wide row of x, all buffers starting `shift` elements in."""
    w = bf16_bits(x) if dtype == "bf16" else x
    flat = w.ravel()[: (rows - 1) * ld + cols]
    buf = torch.empty(flat.size + shift, dtype=torch.int16 if dtype == "bf16" else torch.float32, device="cuda")
    buf[shift:] = torch.from_numpy(flat.view(np.int16) if dtype == "bf16" else flat)
    codes = torch.full((rows * cols + shift + 1,), 0xA5, dtype=torch.uint8, device="cuda")
    scales = torch.empty(rows, dtype=torch.float32, device="cuda")
    bias = torch.empty(1, dtype=torch.int32, device="cuda")
    R.quantize_into(buf[shift:], rows, cols, fmt, scaling, 1.0, codes[shift:], scales, bias, ld=ld)
    ref = O.quantize_with(np.ascontiguousarray(w[:, :cols]).ravel(), rows, cols, fmt, scaling, 1.0)
    label = (rows, cols, ld, dtype, fmt, scaling, shift)
    got = codes.cpu().numpy()
    assert np.array_equal(got[shift:-1], ref.codes), label
    assert got[-1] == 0xA5 and (shift == 0 or got[0] == 0xA5), label   # nothing past either end
    assert np.array_equal(scales.cpu().numpy().view(np.uint32), ref.scales.view(np.uint32)), label
    assert int(bias.item()) == ref.exp_bias, label


@pytest.mark.parametrize("dtype", ["bf16", "f32"])
@pytest.mark.parametrize("scaling", ["pcs", "hw", "unit"])
@pytest.mark.parametrize("shift", [0, 1])
def test_any_width_and_alignment(R, dtype, scaling, shift):
    rng = np.random.default_rng(3)
    for rows, cols, pad in [(1, 1, 0), (3, 7, 0), (5, 8, 1), (9, 9, 0), (4, 511, 0), (4, 513, 2), (700, 33, 0),
                            (6, 1025, 0), (5, 2049, 7), (5, 4097, 0), (3, 8191, 0), (3, 16390, 0), (2, 32771, 1),
                            (2, 65529, 0), (2, 65537, 0)]:
        ld = cols + pad
        x = (rng.standard_normal((rows, ld)) * 0.02).astype(np.float32)
        for fmt in (E4M3, E5M2):
            check(R, x, rows, cols, ld, dtype, fmt, scaling, shift)
        for last in (np.nan, -np.inf, 0.9375, -14.0, 200.0, 1e4):
            x[rows - 1, cols - 1] = last
            check(R, x, rows, cols, ld, dtype, E4M3, scaling, shift)


def test_hardware_bias_over_a_batch_of_mixed_widths(R):
    """One launch of maxima per kernel form; each matrix keeps its own bias."""
    rng = np.random.default_rng(17)
    mats, refs = [], []
    for i, (rows, cols) in enumerate([(300, 1000), (7, 999), (64, 4096), (129, 1001), (1, 5), (2000, 1000), (3, 20000)]):
        w = bf16_bits((rng.standard_normal((rows, cols)) * 0.02 * 8.0**i).astype(np.float32))
        refs.append(O.quantize_with(w.ravel(), rows, cols, E4M3, "hw", 1.0))
        mats.append((torch.from_numpy(w.view(np.int16)).cuda(), rows, cols,
                     torch.empty(rows * cols, dtype=torch.uint8, device="cuda"),
                     torch.empty(rows, dtype=torch.float32, device="cuda"),
                     torch.zeros(1, dtype=torch.int32, device="cuda")))
    R.quantize_batch(mats, E4M3, "hw")
    for m, ref in zip(mats, refs):
        assert np.array_equal(m[3].cpu().numpy(), ref.codes), m[1:3]
        assert np.array_equal(m[4].cpu().numpy(), ref.scales) and int(m[5].item()) == ref.exp_bias, m[1:3]
    assert len({ref.exp_bias for ref in refs}) > 2
