"""Many rays on few bins (whole histograms in LDS, detectors in launches of up to
16384 bins), against the same rays in calls too small for that: the same counts, and
weights that are sums of the same terms."""
import pytest

import test_gpu_detect_groups as groups

torch = groups.torch
pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def lib():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from turbulence_tracing_amd import _lib
    return _lib.load()


# s shadowgram, i interferogram of the same optics, k schlieren, K its
# interferogram, b the shadowgram in one bin more; the largest launch's bins
@pytest.mark.parametrize("which,pix,bins", [("s", 1, 1), ("sik", 1, 3), ("i", 7, 49), ("skiK", 16, 1024),
                                            ("sbi", 63, 12034), ("sik", 90, 16200), ("kiKs", 128, 16384),
                                            ("bs", 127, 16384), ("s", 128, 16384)])
@pytest.mark.parametrize("extra", [-1, 0, 333])
def test_whole_histograms_equal_windows(lib, which, pix, bins, extra):
    from turbulence_tracing_amd import _lib
    n = 200 * bins + extra  # -1: one ray short of whole histograms
    g = torch.Generator(device="cuda").manual_seed(n)
    rf = 2e-3 * torch.randn((4, n), generator=g, dtype=torch.float64, device="cuda")
    rf[0, ::5] = 3e-4  # many in one column of bins
    rf[2, ::7] = float("nan")
    phase = 1e4 * torch.rand(n, generator=g, dtype=torch.float64, device="cuda")
    arr, outs = groups.detectors(which, pix)
    groups.run(lib, arr, rf, phase)
    small, refs = groups.detectors(which, pix)
    part = max(1, 190 * min(pix * pix, bins // 2 + 1))
    for i in range(0, n, part):
        m = min(part, n - i)
        lib.tt_detect(small, len(small), _lib.ptr(rf[:, i:]), n, _lib.ptr(phase[i:]), m, _lib.stream_ptr())
    cnt = {c: groups.detectors(c, pix) for c in "sk"}
    for one, _ in cnt.values():
        groups.run(lib, one, rf, phase)
    assert int(cnt["s"][1][0].sum()) > n // 3
    for c, got, ref in zip(which, outs, refs):
        if c in "iK":  # m weights of at most 2 in any order: m - 1 roundings of a sum of at most 2 m
            m = cnt["k" if c == "K" else "s"][1][0].double()
            assert bool(((got.double() - ref.double()).abs() <= 2 * m * 2 * m * 2.0 ** -24).all())
            assert abs(float(got.double().sum() - ref.double().sum())) <= 1e-5 * float(ref.double().sum())
        else:
            assert torch.equal(got, ref)
