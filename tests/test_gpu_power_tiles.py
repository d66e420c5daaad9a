"""The power spectrum where a block of its last pass takes several tiles: every
fixed length with more tiles than blocks, a part of them in the last turn, the last
one ragged; and short lengths with many pencils a block."""
import pytest

import test_gpu_power_bins as bins

pytestmark = pytest.mark.gpu

LDS_ELEMENTS, BLOCKS = 8192, 512  # of a tile; of the launch
SHAPES = [(360, 182, 128), (300, 143, 192), (206, 104, 384), (128, 127, 512), (128, 65, 1024)]  # x', y', z'


@pytest.fixture(scope="module")
def lib():
    if not bins.torch.cuda.is_available():
        pytest.skip("no GPU")
    from turbulence_tracing_amd import _lib
    return _lib.load()


@pytest.mark.parametrize("shape", SHAPES)
def test_more_tiles_than_blocks(lib, shape):
    pencils, columns = LDS_ELEMENTS // shape[2], (shape[0] // 2 + 1) * shape[1]
    tiles = -(-columns // pencils)
    assert tiles > BLOCKS and tiles % BLOCKS and columns % pencils
    bins.test_counts_and_sums(lib, shape, False)


@pytest.mark.parametrize("shape,many", [((256, 256, 256), False), ((128, 127, 512), True), ((300, 143, 192), True),
                                        ((700, 700, 4), False), ((254, 257, 33), True)])
def test_other_bins_and_short_lengths(lib, shape, many):
    bins.test_counts_and_sums(lib, shape, many)
