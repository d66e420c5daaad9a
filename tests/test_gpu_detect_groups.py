"""Detectors in one call against one call each: groups that share a train and
bins (in any order), rays that are no whole number of blocks, blocks with no ray
on the detector, windows larger than LDS; and bins at the exact edges of
np.histogram2d."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def lib():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from turbulence_tracing_amd import _lib
    return _lib.load()


def detectors(which, pix):
    from turbulence_tracing_amd import _lib
    from turbulence_tracing_amd.ray_transfer_matrix import (hist_desc, make_train, op_knife, schlieren_ops,
                                                            shadowgraphy_ops)
    arr, outs = (_lib.Detector * len(which))(), []
    for k, c in enumerate(which):
        sh = shadowgraphy_ops(400, 25, 0.0)
        arr[k].train = make_train(schlieren_ops(400, 25, 0.0, [op_knife(0.0, "x", 1)]) if c in "kK" else sh, to_mm=True)
        n = pix + 1 if c == "b" else pix
        arr[k].hist = hist_desc(13.5, 13.5, n, n)
        arr[k].mode = int(c in "iK")
        arr[k].tilt_k = 2.0
        outs.append(torch.zeros((n, n), dtype=torch.float32 if c in "iK" else torch.int32, device="cuda"))
        if c in "iK":
            arr[k].wsum = outs[-1].data_ptr()
        else:
            arr[k].counts = outs[-1].data_ptr()
    return arr, outs


def run(lib, arr, rf, phase):
    from turbulence_tracing_amd import _lib
    n = rf.shape[1]
    lib.tt_detect(arr, len(arr), _lib.ptr(rf), n, _lib.ptr(phase), n, _lib.stream_ptr())
    torch.cuda.synchronize()


# s shadowgram, i interferogram of the same optics, k schlieren, K its
# interferogram, b the shadowgram in other bins
@pytest.mark.parametrize("which", ["sik", "ski", "iks", "kiKs", "sbsi", "s", "kK"])
@pytest.mark.parametrize("n,pix", [(1, 16), (511, 64), (513, 300), (4097, 2048)])
def test_groups_equal_single_calls(lib, which, n, pix):
    rng = np.random.default_rng(n)
    rf = np.stack([rng.normal(0, 2e-3, n), rng.normal(0, 2e-3, n), rng.normal(0, 2e-3, n), rng.normal(0, 2e-3, n)])
    rf[0, 512:1024] = 1.0  # a block whose rays all miss
    rf[2, ::7] = np.nan
    rf = torch.as_tensor(rf, device="cuda")
    phase = torch.as_tensor(rng.uniform(0, 1e4, n), device="cuda")
    arr, outs = detectors(which, pix)
    run(lib, arr, rf, phase)
    for c, got in zip(which, outs):
        one, ref = detectors(c, pix)
        run(lib, one, rf, phase)
        if c in "iK":  # m weights of at most 2 in any order: m - 1 roundings of a sum of at most 2 m
            cnt = detectors("k" if c == "K" else "s", pix)
            run(lib, cnt[0], rf, phase)
            m = cnt[1][0].double()
            assert bool(((got.double() - ref[0].double()).abs() <= 2 * m * 2 * m * 2.0 ** -24).all())
        else:
            assert torch.equal(got, ref[0])


@pytest.mark.parametrize("nb", [1, 3, 7, 1000, 1361])
def test_edges_as_histogram2d(lib, nb):
    from turbulence_tracing_amd import _lib
    from turbulence_tracing_amd.ray_transfer_matrix import hist_desc, make_train
    lo, hi = -6.75, 6.75
    e = np.linspace(lo, hi, nb + 1)
    v = np.concatenate([e, np.nextafter(e, -np.inf), np.nextafter(e, np.inf), [lo - 1, hi + 1]])
    rf = np.zeros((4, v.size))
    rf[0], rf[2] = v, v[::-1]
    H = torch.zeros((nb, nb), dtype=torch.int32, device="cuda")
    arr = (_lib.Detector * 1)()
    arr[0].train = make_train([], to_mm=False)
    arr[0].hist = hist_desc(hi - lo, hi - lo, nb, nb)
    arr[0].mode = 0
    arr[0].counts = H.data_ptr()
    run(lib, arr, torch.as_tensor(rf, device="cuda"), None)
    want = np.histogram2d(rf[0], rf[2], bins=[nb, nb], range=[[lo, hi], [lo, hi]])[0].T
    np.testing.assert_array_equal(H.cpu().numpy(), want)
