"""The h = 1/2 march's two forms (rays of a wave at one step, rays at different
steps) and its cell addressing, bit for bit against each other."""
import numpy as np
import pytest
import torch

from turbulence_tracing_amd import _lib

pytestmark = pytest.mark.gpu
C0 = 299792458.0
D = 1e-4


def grid_of(n):
    return _lib.Grid(*n, *(-D * (m - 1) / 2 for m in n), D, D, D)


def rays(n, count, planes, slope, g):
    """Rays over (and a little beyond) the grid, ray i launched from plane
    planes[i % len(planes)], some of them on the grid's edges."""
    u = torch.rand((2, count), generator=g, dtype=torch.float64) - 0.5
    th = torch.randn((2, count), generator=g, dtype=torch.float64) * slope
    s0 = torch.stack([u[0] * 1.02 * D * (n[0] - 1), u[1] * 1.02 * D * (n[1] - 1),
                      -D * (n[2] - 1) / 2 + D * torch.tensor(planes, dtype=torch.float64)[torch.arange(count) % len(planes)],
                      C0 * th[0], C0 * th[1], C0 * torch.sqrt(1 - th[0] ** 2 - th[1] ** 2)])
    s0[0, : count // 16] = -D * (n[0] - 1) / 2
    s0[1, : count // 32] = D * (n[1] - 1) / 2
    return s0.cuda()


def trace(lib, f4, n, s0, order=None, sf=False, forms=None):
    N = s0.shape[1]
    new = lambda *s: torch.full(s, -1.0, dtype=torch.float64, device="cuda")
    rf, ph, out, st = new(4, N), new(N), new(6, N) if sf else None, torch.full((N,), -1, dtype=torch.int32, device="cuda")
    opts = _lib.TraceOpts(0.5, 10 * D * n[2], 0, None if forms is None else forms.data_ptr())
    g = grid_of(n)
    lib.tt_trace_rk4(_lib.ptr(f4), _lib.C.byref(g), _lib.C.byref(opts), _lib.ptr(s0), N, N, _lib.ptr(order), _lib.ptr(rf), N,
                     _lib.ptr(ph), _lib.ptr(out), N, _lib.ptr(st), _lib.stream_ptr())
    torch.cuda.synchronize()
    return [t.cpu().numpy() for t in (rf, ph, st) + ((out,) if sf else ())]


@pytest.mark.parametrize("n,count,amp,slope", [((2, 2, 2), 1, 1e-4, 1e-3), ((33, 18, 25), 63, 1e-4, 1e-3),
                                               ((33, 18, 25), 4099, 1e-3, 2e-2), ((64, 64, 9), 20000, 2e-2, 5e-2)])
@pytest.mark.parametrize("form", ["plain", "sf", "forms"])
def test_waves_at_one_step_equal_mixed_waves(lib, n, count, amp, slope, form):
    g = torch.Generator().manual_seed(count)
    f4 = (torch.randn((n[2], n[1], n[0], 4), generator=g) * amp).cuda()
    planes = [0.0] if n[2] == 2 else [0.0, 3.0, 3.5, 6.25, 7.5]
    s0 = rays(n, count, planes, slope, g)
    forms = None
    if form == "forms":
        forms = torch.empty((n[2], n[1], n[0], 16), device="cuda")
        gr = grid_of(n)
        lib.tt_plane_forms(_lib.ptr(f4), _lib.C.byref(gr), _lib.ptr(forms), _lib.stream_ptr())
    mixed = trace(lib, f4, n, s0, None, form == "sf", forms)  # every wave holds all launch planes
    # one wave per launch plane at most: the rays of a plane are consecutive
    # and each plane is traced in a launch of its own
    for p in range(len(planes)):
        at = torch.arange(p, count, len(planes), device="cuda")
        if at.numel() == 0:
            continue
        one = trace(lib, f4, n, s0[:, at].contiguous(), None, form == "sf", forms)
        for a, b in zip(mixed, one):
            np.testing.assert_array_equal(a[..., at.cpu().numpy()], b)


@pytest.mark.parametrize("nx,ny", [(4096, 4096), (4097, 4096)])
def test_cell_addressing_at_the_largest_planes(lib, nx, ny):
    """Planes of 2^24 nodes (32-bit cell offsets) and just above (64-bit): rays
    near the far corner see the same field as in a crop around them."""
    g = torch.Generator().manual_seed(nx)
    m, n = 24, (nx, ny, 3)
    crop = (torch.randn((3, m, m, 4), generator=g) * 1e-3).cuda()
    f4 = torch.zeros((3, ny, nx, 4), device="cuda")
    f4[:, ny - m:, nx - m:] = crop
    s0 = rays((m, m, 3), 2000, [0.0], 5e-3, g)
    s0[:2] *= 0.5  # clear of the crop's edges, which the full plane does not have
    big = s0.clone()
    big[0] += D * (nx - m) / 2
    big[1] += D * (ny - m) / 2
    a, b = trace(lib, f4, n, big), trace(lib, crop, (m, m, 3), s0)
    np.testing.assert_array_equal(a[2], b[2])
    shift = np.array([D * (nx - m) / 2, 0, D * (ny - m) / 2, 0])[:, None]
    # an in-cell coordinate is rounded to fp32 at a cell number of up to 4096
    # (2^-12 cells); over two cells that moves the field by 2^-12 of its change
    # per cell (about 5 amplitudes), so an angle by 2 * 5e-3 * 2^-12 and a
    # position by 2^-12 cells, twice
    assert np.abs(a[0] - shift - b[0])[[0, 2]].max() <= 2 * D * 2.0 ** -12
    assert np.abs(a[0] - b[0])[[1, 3]].max() <= 2 * 5e-3 * 2.0 ** -12
