"""The batched trace's map from blocks to chunks: chunk counts around the
number of XCDs, chunks that are no whole number of blocks, ragged last chunks,
each steps-per-cell form: the bits of one tt_trace_rk4 call per member."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def lib():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from turbulence_tracing_amd import _lib
    return _lib.load()


@pytest.mark.parametrize("h", [1.0, 0.5, 0.25])
@pytest.mark.parametrize("rays,chunk,block,bpc", [([1], 64, 256, 0), ([64 * 7, 1], 64, 64, 0), ([900, 129], 129, 128, 0),
                                                  ([700, 255, 257, 33], 300, 256, 3), ([2000, 1], 257, 64, 64)])
def test_every_ray_once(lib, rays, chunk, block, bpc, h):
    from turbulence_tracing_amd.ensemble import Ensemble, Member
    ens = Ensemble([Member(n=20 + 7 * i, beta=-3.4, aniso=1.0, rms=0.1, ne0=1e24, n_rays=r, seed=i)
                    for i, r in enumerate(rays)], pix=32, h=h)
    ens.generate()
    ens.order()
    ref = []
    for p in ens.pipes:
        p.trace()
        ref.append((p.rf.clone(), p.phase.clone()))
        p.rf.fill_(7.0)
        p.phase.fill_(7.0)
    ens.tuning = {"block": block, "blocks_per_cu": bpc, "variant": 0, "chunk": chunk, "brick_shift": 0}
    ens.trace()
    for (rf, ph), p in zip(ref, ens.pipes):
        np.testing.assert_array_equal(p.rf.cpu().numpy(), rf.cpu().numpy())
        np.testing.assert_array_equal(p.phase.cpu().numpy(), ph.cpu().numpy())
