"""Short lengths in large fields, where a block of the general transform takes 32
to 256 pencils: against the FP64 oracle, on each axis."""
import numpy as np
import pytest

from oracle import field as OF

pytestmark = pytest.mark.gpu

# length, and the other two axes' so that 2^10 blocks of 2^8, 2^7, 2^6 and 2^5
# pencils (2048 elements at most) are there, or just not
SHAPES = [(2, 1024, 512), (3, 1022, 512), (7, 1024, 512), (8, 1024, 514), (12, 512, 512), (16, 510, 512), (16, 512, 510),
          (31, 510, 257), (33, 254, 256), (60, 256, 257)]


@pytest.mark.parametrize("n,u,v", SHAPES)
@pytest.mark.parametrize("axis", [0, 1, 2])
def test_field_from_noise(lib, n, u, v, axis):
    from turbulence_tracing_amd import turboGen
    shape = [u, v]
    shape.insert(axis, n)
    rs = np.random.RandomState(n + axis)
    Wr, Wi = rs.randn(*shape), rs.randn(*shape)
    S = OF.sqrt_powerlaw(tuple(shape), -11 / 3)
    want = OF.gaussian_field(Wr, Wi, S)
    got = turboGen.gaussian_field_from_noise(Wr, Wi, S).double().cpu().numpy()
    # every field's bar against FP64
    assert np.sqrt(np.mean((got - want) ** 2) / np.mean(want ** 2)) <= 1e-5
