"""The path estimate writes every feature of every ray: a buffer of NaN and one
of zeros end up the same, for rays that start before, in and behind the grid, in
blocks that are shorter and longer than a feature segment and do not divide the
grid; segments no ray step lies in are zero."""
import ctypes as C

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


@pytest.mark.parametrize("nz,k", [(65, 16), (65, 1), (40, 7), (20, 8), (9, 16), (2, 1), (130, 64)])
def test_every_feature_written(lib, nz, k):
    from turbulence_tracing_amd import _lib
    n, c = 2000, 299792458.0
    rng = np.random.default_rng(nz + k)
    g = _lib.Grid(12, 10, nz, 0.0, 0.0, 0.0, 1e-4, 1e-4, 1e-4)
    f4 = torch.as_tensor(rng.normal(0, 1e-4, (nz, 10, 12, 4)).astype(np.float32), device="cuda")
    s0 = np.zeros((6, n))
    s0[:2] = rng.uniform(1e-4, 8e-4, (2, n))
    s0[2] = rng.choice([0.0, -1e-4, 0.3, 0.5, 1.0, 1.2], n) * (nz - 1) * 1e-4
    s0[3:5] = rng.normal(0, 1e-3 * c, (2, n))
    s0[5] = np.where(rng.random(n) < 0.02, -c, c * 0.9999)  # some the estimate cannot follow
    s0 = torch.as_tensor(s0, device="cuda")
    nb = (nz - 1 + k - 1) // k
    GM = None
    if k > 1:
        GM = torch.zeros((10, 12, nb, 2, 4), device="cuda")
        lib.tt_field_blocks(_lib.ptr(f4), C.byref(g), k, _lib.ptr(GM), _lib.stream_ptr())
    outs = []
    for fill in (float("nan"), 0.0):
        feat = torch.full((48, n), fill, device="cuda")
        base = torch.full((5, n), fill, dtype=torch.float64, device="cuda")
        lib.tt_path_features(_lib.ptr(f4), _lib.ptr(GM), k, C.byref(g), _lib.ptr(s0), n, n, None, _lib.ptr(feat), n,
                             _lib.ptr(base), n, _lib.stream_ptr())
        outs.append(feat)
    assert not bool(torch.isnan(outs[0]).any())
    assert torch.equal(outs[0], outs[1])
    assert bool((outs[0][:32, s0[2] > 1.1 * (nz - 1) * 1e-4] == 0).all())  # start behind: no step
