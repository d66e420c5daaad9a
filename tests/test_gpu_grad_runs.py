"""The gradient stencil where a block marches through many planes (runs of 4, 8,
16 and 32 that do not divide the grid) and on grids of a few planes (columns
instead of tiles), over the memory orders of its input, against the second-order
differences of np.gradient formed in float64."""
import itertools

import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

# Runs by order (x-, y- / z-contiguous) in fp32 and fp64: 8 / 4 and 16 / 4; 16 / 16
# and 32 / 16; 32 / 32 and 32 / 32
DEEP = [(201, 201, 203), (260, 250, 270), (400, 330, 420)]
# up to 4, 6 or 8 planes along y or z (by order), and one more
THIN = [(150, 40, 4), (40, 150, 5), (40, 150, 6), (40, 150, 7), (33, 8, 70), (300, 5, 33), (130, 7, 2), (65, 9, 17),
        (2, 2, 700), (700, 2, 2), (3, 700, 3), (64, 4, 64)]


@pytest.fixture(scope="module")
def lib():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from turbulence_tracing_amd import _lib
    return _lib.load()


def difference(s, axis, d):
    """np.gradient of s along an axis."""
    s = s.movedim(axis, 0)
    g = torch.empty_like(s)
    g[1:-1] = (s[2:] - s[:-2]) / (2 * d)
    g[0] = (s[1] - s[0]) / d
    g[-1] = (s[-1] - s[-2]) / d
    return g.movedim(0, axis)


def stencil(lib, f, alpha, beta, ne_max, k0, d):
    from turbulence_tracing_amd import _lib
    n = f.shape
    g = _lib.Grid(*n, 0.0, 0.0, 0.0, *d)
    out = torch.full((n[2], n[1], n[0], 4), 7.0, device="cuda")
    lib.tt_grad_stencil(_lib.ptr(f), int(f.dtype == torch.float64), *f.stride(), _lib.C.byref(g), alpha, beta, ne_max,
                        k0, None, 0, _lib.ptr(out), _lib.stream_ptr())
    return out


@pytest.mark.parametrize("dtype", [torch.float32, torch.float64])
@pytest.mark.parametrize("n", DEEP + THIN)
def test_every_memory_order(lib, n, dtype):
    alpha, beta, ne_max, k0, d = 0.1, 0.7, 0.8, 300.0, (0.5, 0.25, 2.0)
    g = torch.Generator(device="cuda").manual_seed(sum(n))
    f = (0.3 + 0.4 * torch.randn(n, generator=g, dtype=torch.float64, device="cuda")).to(dtype)
    s = (beta * f.double()).clamp(max=ne_max - alpha)
    # the tolerances of the stencil's test over memory orders: an error of u |s| for
    # s, its two factors and the bound each, times the weights, and one rounding
    u = 2.0 ** -24 if dtype == torch.float32 else 2.0 ** -53
    err = 2 * u * float(s.abs().max())
    first = None
    for order in itertools.permutations(range(3)):
        v = f.permute(*order).contiguous().permute(*[order.index(i) for i in range(3)])
        got = stencil(lib, v, alpha, beta, ne_max, k0, d)
        if first is None:
            first = got
            for i in range(4):
                w = -0.5 * d[2] * difference(s, i, d[i]) if i < 3 else k0 * d[2] * ((1 - alpha - s).sqrt() - 1)
                tol = 2 * err * d[2] * 0.5 / d[i] if i < 3 else k0 * d[2] * (1.12 * err + 4 * 2.0 ** -53)
                e = (got[..., i].permute(2, 1, 0) - w).abs()
                assert bool((e <= tol + 4 * 2.0 ** -24 * w.abs()).all()), (i, float(e.max()))
        assert torch.equal(got, first), order
