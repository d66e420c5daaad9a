"""tt_detect beyond 2^32 rays, as many as one axis of a launch does not hold."""
import ctypes as C

import pytest
import torch

pytestmark = pytest.mark.gpu


def test_more_rays_than_threads_along_an_axis(lib):
    from turbulence_tracing_amd import _lib
    n = 2 ** 32 + 5 * 512 + 3
    if torch.cuda.mem_get_info()[0] < 4 * 8 * n + (4 << 30):
        pytest.skip("the rays do not fit this GPU's free memory")
    rf = torch.full((4, n), float("nan"), dtype=torch.float64, device="cuda")  # lost rays
    at = [0, 511, 512, 3 * 512 + 7, 2 ** 31 - 1, 2 ** 31, 2 ** 32 - 1, 2 ** 32, 2 ** 32 + 513, n - 1]
    rf[:, torch.tensor(at, device="cuda")] = 0.5
    H = torch.zeros((2, 2), dtype=torch.int32, device="cuda")
    d = (_lib.Detector * 1)()
    d[0].hist = _lib.Hist(2, 2, -1.0, 1.0, -1.0, 1.0)
    d[0].counts = H.data_ptr()
    lib.tt_detect(d, 1, _lib.ptr(rf), n, None, n, _lib.stream_ptr())
    assert H.tolist() == [[0, 0], [0, len(at)]]
    del rf
    torch.cuda.empty_cache()
