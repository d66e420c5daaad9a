"""Rays traced in time by four lanes each against one lane each where the field
holds NaN or infinite nodes, or a ray starts at infinity, at rest or without a
velocity along z: the same bits and the same NaNs."""
from types import SimpleNamespace

import pytest

import test_gpu_time_quads as quads

torch = quads.torch
pytestmark = pytest.mark.gpu
lib, scene = quads.lib, quads.scene


@pytest.mark.parametrize("what", [float("nan"), float("inf"), -float("inf")])
@pytest.mark.parametrize("channel", [0, 2, 3])
def test_field_with_a_bad_node(lib, scene, what, channel):
    cube, s0 = scene
    f4 = cube.field4.clone()
    f4[12, ::4, ::5, channel] = what
    bad = SimpleNamespace(field4=f4, grid=cube.grid), s0
    one = quads.trace(lib, bad, quads.QUADS + 1)
    few = quads.trace(lib, bad, 4000)
    assert bool(torch.isnan(one[0]).any()) or bool(torch.isnan(one[2]).any())
    for a, b in zip(few[:3], one[:3]):
        assert quads.same(a, b[..., :4000])


def test_rays_from_nowhere(lib, scene):
    cube, s0 = scene
    s0 = s0.clone()
    s0[0, 0::9] = float("inf")
    s0[2, 1::9] = -float("inf")
    s0[3, 2::9] = float("inf")
    s0[3:, 3::9] = 0.0
    s0[5, 4::9] = 0.0
    s0[5, 5::9] = -s0[5, 5::9]
    odd = cube, s0
    one = quads.trace(lib, odd, quads.QUADS + 1)
    few = quads.trace(lib, odd, 4000)
    for a, b in zip(few[:3], one[:3]):
        assert quads.same(a, b[..., :4000])
