"""The transform of any length (tiled DFTs of primes above 5, ping-pong LDS)
against the FP64 oracle, at the edges of its tiles."""
import numpy as np
import pytest

from oracle import field as OF
from oracle import spectrum as OS

pytestmark = pytest.mark.gpu

# primes that end one or three past a tile of four outputs, the smallest and
# large ones; products of two primes (twiddled second DFT); with radices 8, 4,
# 2, 3, 5; the lengths where a block takes 16, 8, 4, 2 and 1 pencils
LENGTHS = [7, 29, 31, 37, 67, 257, 1021, 77, 13 * 31, 7 * 7 * 7, 8 * 7 * 3, 2 * 11, 4 * 5 * 13, 309, 310, 602, 1202,
           2403, 4093, 4096]


@pytest.mark.parametrize("n", LENGTHS)
@pytest.mark.parametrize("axis", [0, 1, 2])
def test_field_from_noise_length_on_each_axis(lib, n, axis):
    from turbulence_tracing_amd import turboGen
    shape = [3, 5, 7]
    shape[axis] = n
    rs = np.random.RandomState(n + axis)
    Wr, Wi = rs.randn(*shape), rs.randn(*shape)
    S = OF.sqrt_powerlaw(tuple(shape), -11 / 3)
    want = OF.gaussian_field(Wr, Wi, S)
    got = turboGen.gaussian_field_from_noise(Wr, Wi, S).double().cpu().numpy()
    # every field's bar against FP64
    assert np.sqrt(np.mean((got - want) ** 2) / np.mean(want ** 2)) <= 1e-5


@pytest.mark.parametrize("shape", [(67, 5, 14), (6, 31, 33), (9, 4, 257), (18, 37, 3)])
def test_power_of_prime_lengths(lib, shape):
    from turbulence_tracing_amd.calculate_spectrum_3d import power_bins
    f = np.random.RandomState(sum(shape)).randn(*shape).astype(np.float32).astype(np.float64)
    sums, counts = power_bins(f, 0.5, 40, 0, OS.bin_width(shape, 0.5, 40))
    so, co = OS.binned(f, 0.5, 40)
    np.testing.assert_array_equal(counts.cpu().numpy(), co)
    # the bars of the binned-power tests of other lengths
    np.testing.assert_allclose(sums.cpu().numpy(), so, rtol=2e-5, atol=1e-6 * so.max())
