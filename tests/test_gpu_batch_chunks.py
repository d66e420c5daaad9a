"""Chunks of the batched trace far above its members' rays: the launch is sized by
the rays there are, and one that would hold 2^32 threads or more is split."""
import ctypes as C

import pytest
import torch

pytestmark = pytest.mark.gpu


def ensemble(rays, chunk, block):
    from turbulence_tracing_amd.ensemble import Ensemble, Member
    ens = Ensemble([Member(n=n, beta=-3.4, aniso=1.0, rms=0.1, ne0=1e24, n_rays=r, seed=i)
                    for i, (n, r) in enumerate(rays)], pix=16)
    ens.generate()
    ens.order()
    ens.tuning = {"block": block, "blocks_per_cu": 0, "variant": 0, "chunk": chunk, "brick_shift": 0}
    return ens


def check(ens):
    ref = []
    for p in ens.pipes:
        p.trace()
        ref.append((p.rf.clone(), p.phase.clone()))
        p.rf.fill_(7.0)
        p.phase.fill_(7.0)
    ens.trace()
    for (rf, ph), p in zip(ref, ens.pipes):
        assert torch.equal(p.rf.view(torch.int64), rf.view(torch.int64))
        assert torch.equal(p.phase.view(torch.int64), ph.view(torch.int64))


@pytest.mark.parametrize("block", [64, 256])
def test_small_members_in_the_largest_chunk(lib, block):
    # one chunk each: 257 * 2^24 threads if every chunk got the blocks of a full one
    ens = ensemble([(8, 70)] * 257, 1 << 24, block)
    check(ens)
    assert ens.info.chunk == 256 and ens.info.nchunks == 257


def test_launch_above_the_thread_limit(lib):
    # the large member's chunk sizes the others': 264 * 2^24 threads
    ens = ensemble([(4, 1 << 24)] + [(4, 1)] * 256, 1 << 24, 256)
    check(ens)
    assert ens.info.chunk == 1 << 24 and ens.info.nchunks == 257


@pytest.mark.parametrize("chunk,want", [(64, 256), (256, 256), (257, 512), (300, 512), (4096, 1024)])
def test_chunks_are_whole_blocks(lib, chunk, want):
    ens = ensemble([(12, 1000), (9, 3)], chunk, 128)
    check(ens)
    assert ens.info.chunk == want
    nbytes = C.c_size_t()
    lib.tt_batch_workspace_bytes(ens._items(), 2, chunk, C.byref(nbytes))
    small = torch.empty(nbytes.value, dtype=torch.uint8, device="cuda")
    lib.tt_batch_prepare(ens._items(), 2, 0.5, chunk, small.data_ptr(), small.numel(), C.byref(ens.info))
    assert ens.info.nchunks == -(-1000 // want) + 1
