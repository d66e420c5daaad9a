"""The power spectrum's binning: every fixed length along z and some others,
spectra whose columns are no whole number of tiles, more tiles than blocks, bins
too many for the histogram's copies in LDS, both estimators; the counts exactly,
the sums against an FFT in float64."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

SHAPES = [(2, 3, 128), (9, 40, 192), (130, 33, 256), (6, 5, 384), (30, 47, 512), (7, 8, 1024), (128, 128, 128),
          (65, 64, 33), (5, 2, 2), (12, 10, 67), (16, 300, 64)]  # x', y', z'


@pytest.fixture(scope="module")
def lib():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from turbulence_tracing_amd import _lib
    return _lib.load()


def power(lib, f, mode, nbins, dx, bin_w):
    from turbulence_tracing_amd import _lib
    nz, ny, nx = f.shape
    plan, nbytes = _lib.C.c_void_p(), _lib.C.c_size_t()
    lib.tt_fft_plan_create(nx, ny, nz, _lib.C.byref(plan))
    lib.tt_fft_workspace_bytes(plan, _lib.C.byref(nbytes))
    ws = torch.empty(nbytes.value, dtype=torch.uint8, device="cuda")
    out = torch.zeros((2, nbins), dtype=torch.float64, device="cuda")
    d = torch.as_tensor(f, device="cuda")
    lib.tt_power_spectrum(plan, _lib.ptr(d), mode, nbins, dx, bin_w, _lib.ptr(ws), _lib.ptr(out[0]), _lib.ptr(out[1]),
                          _lib.stream_ptr())
    torch.cuda.synchronize()
    lib.tt_fft_plan_destroy(plan)
    return out.cpu().numpy()


def visited(n):
    """The value the reference's loop gives to each index (NaN: none)."""
    v = np.full(n, np.nan)
    for i in range(-n // 2, n // 2 - 1):
        v[i % n] = i
    return v


@pytest.mark.parametrize("many", [False, True])
@pytest.mark.parametrize("shape", SHAPES)
def test_counts_and_sums(lib, shape, many):
    f = np.random.default_rng(sum(shape)).normal(size=shape[::-1]).astype(np.float32)
    p = np.abs(np.fft.fftn(f.astype(np.float64))) ** 2
    nt, dx = f.size, 0.5
    k = [np.fft.fftfreq(n, dx) for n in f.shape]
    K = np.sqrt((k[0][:, None, None] ** 2 + k[1][None, :, None] ** 2) + k[2][None, None, :] ** 2)
    nbins = 2048 if many else 37
    bin_w = K.max() / (nbins - 2)
    b = np.searchsorted(bin_w * np.arange(nbins), K, "right") - 1
    on = b <= nbins - 2
    v = [visited(n) for n in f.shape]
    with np.errstate(invalid="ignore"):
        r = np.rint(np.sqrt(v[0][:, None, None] ** 2 + v[1][None, :, None] ** 2 + v[2][None, None, :] ** 2))
    on1 = r < nbins
    r = np.where(on1, r, 0).astype(int)
    # an element's error is that of the float32 transform, some log2(n) roundings
    # of 2^-24 of the mean amplitude: of a bin's sum, twice that over its mean
    tol = 2 * 4 * np.log2(nt) * 2.0 ** -24
    for mode, idx, sel, scale in ((0, b, on, 1.0), (1, r, on1, 1.0 / nt ** 2)):
        got = power(lib, f, mode, nbins, dx, bin_w)
        want_n = np.bincount(idx[sel], minlength=nbins)[:nbins]
        want_s = np.bincount(idx[sel], weights=p[sel] * scale, minlength=nbins)[:nbins]
        np.testing.assert_array_equal(got[1], want_n)
        mean = np.maximum(want_s, want_n * p.mean() * scale)
        assert (np.abs(got[0] - want_s) <= tol * mean).all(), mode
