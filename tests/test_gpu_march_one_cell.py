"""The h = 1/2 march on the smallest grid, one cell: against the same steps by
per-stage gathers (variant 1)."""
import pytest

import test_gpu_march as march

_lib, torch = march._lib, march.torch
pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("count", [1, 64, 1000])
def test_one_cell_as_by_gathers(lib, count):
    n, amp, slope = (2, 2, 2), 1e-4, 1e-3
    g = torch.Generator().manual_seed(count)
    f4 = (torch.randn((2, 2, 2, 4), generator=g) * amp).cuda()
    s0 = march.rays(n, count, [0.0], slope, g)
    s0[:2] *= 0.9  # rays that stay inside
    got = march.trace(lib, f4, n, s0)
    rf = torch.full((4, count), -1.0, dtype=torch.float64, device="cuda")
    ph, st = torch.full((count,), -1.0, dtype=torch.float64, device="cuda"), torch.zeros(count, dtype=torch.int32, device="cuda")
    opts, gr = _lib.TraceOpts(0.5, 1.0, 1, None), march.grid_of(n)
    lib.tt_trace_rk4(_lib.ptr(f4), _lib.C.byref(gr), _lib.C.byref(opts), _lib.ptr(s0), count, count, None, _lib.ptr(rf),
                     count, _lib.ptr(ph), None, count, _lib.ptr(st), _lib.stream_ptr())
    rf, ph = rf.cpu().numpy(), ph.cpu().numpy()
    assert (got[2] == 0).all() and not bool(st.any())
    # two steps of four stages, each with a few roundings of 2^-24: of in-cell
    # coordinates below 1, of velocities of up to 5 slopes and of a field of up to 5
    # amplitudes (the phase as well, which is summed by another rule of fourth order:
    # its integrand is a cubic along the ray, so both are exact but for |v| / W, off by
    # the square of a slope times a deflection)
    u = 32 * 2.0 ** -24
    assert abs(got[0] - rf)[[0, 2]].max() <= u * march.D
    assert abs(got[0] - rf)[[1, 3]].max() <= u * (5 * slope + 5 * amp)
    assert abs(got[1] - ph).max() <= 5 * amp * (u + (5 * slope) ** 2)
    # and the field was seen at all: it turns the rays
    free = march.trace(lib, torch.zeros_like(f4), n, s0)
    assert abs(got[0] - free[0])[[1, 3]].max() > 1e3 * u * 5 * amp / 32
