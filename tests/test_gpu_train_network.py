"""Surrogate.train where the caller's `log` changes the network between two
epochs: what the next epoch's steps read and write, against the same training
called layer by layer.  At up to 512 rows a step both have the same bits: one
partial sum a weight, and two a bias, which add up alike in either order."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu
NAMES = ("W", "b", "dW", "db", "mW", "vW", "mb", "vb")


def surrogate(seed):
    from turbulence_tracing_amd.surrogate import Norm, Surrogate
    return Surrogate(Norm(np.zeros(48, np.float32), np.ones(48, np.float32), 1.0, 1.0, 1.0), seed=seed)


def load(sur):
    from turbulence_tracing_amd.surrogate import MLP
    sur.mlp.load_state(MLP(seed=9).state())


def replace_tensors(sur):
    m = sur.mlp
    for name in NAMES + ("Wb",):
        setattr(m, name, [t.clone() for t in getattr(m, name)])


def replace_network(sur):
    from turbulence_tracing_amd.surrogate import MLP
    sur.mlp = MLP(seed=9)


def replace_loss(sur):
    sur.tau = 0.7
    sur.w_reg = torch.tensor([0.5, 1.0, 2.0, 1.0, 0.25], dtype=torch.float32, device="cuda")


@pytest.mark.parametrize("change", [load, replace_tensors, replace_network, replace_loss])
def test_next_epoch_uses_the_network_as_it_is(lib, change):
    n, batch, g = 512, 256, torch.Generator().manual_seed(3)
    feat = torch.randn((n, 48), generator=g).cuda()
    target = torch.randn((n, 5), generator=g).cuda()

    def train(layered):
        sur, calls = surrogate(5), []
        if layered:
            sur._fused_step = lambda *a: None

        def log(line):
            calls.append(line)
            if len(calls) == 2:
                change(sur)

        return sur, sur.train(feat, target, epochs=4, batch=batch, wd=1e-3, log=log)

    (a, la), (b, lb) = train(False), train(True)
    # the loss sums are fp64 sums of the same fp32 terms
    np.testing.assert_allclose(np.array(la), np.array(lb), rtol=1e-12)
    assert a.mlp.step == b.mlp.step
    for name in NAMES:
        for l, (x, y) in enumerate(zip(getattr(a.mlp, name), getattr(b.mlp, name))):
            assert torch.equal(x, y), (name, l)
    for w, wb in zip(a.mlp.W, a.mlp.Wb):
        assert torch.equal(wb, w.to(torch.bfloat16))


def test_more_rows_a_step_than_there_are(lib):
    """No step is run, whatever the batch, and nothing of its size is asked for."""
    sur, g = surrogate(5), torch.Generator().manual_seed(1)
    feat, target = torch.randn((100, 48), generator=g).cuda(), torch.randn((100, 5), generator=g).cuda()
    before = [w.clone() for w in sur.mlp.W]
    for batch in (101, 2 ** 24 + 1):
        hist = sur.train(feat, target, epochs=2, batch=batch)
        assert len(hist) == 2 and sur.mlp.step == 0
    assert all(torch.equal(x, y) for x, y in zip(before, sur.mlp.W))
    # the network's outputs (32 bytes a row) and their gradients (16)
    torch.cuda.reset_peak_memory_stats()
    base = torch.cuda.memory_allocated()
    sur.train(feat, target, epochs=1, batch=1 << 22)
    assert torch.cuda.max_memory_allocated() - base <= (1 << 22) * (16 + 32) + (1 << 20)


def test_steps_the_one_call_form_does_not_take(lib):
    """Above 2^24 rows a step and for tensors off 16 bytes the layers are called one by one."""
    sur = surrogate(5)
    X, target = torch.zeros((8, 48), dtype=torch.bfloat16, device="cuda"), torch.zeros((8, 5), device="cuda")
    assert sur._fused_step(X, target, 2 ** 24 + 1, 0.0) is None
    assert sur._fused_step(X, target, 0, 0.0) is None
    assert sur._fused_step(X, target, 8, 0.0) is not None


@pytest.mark.parametrize("name,l", [("Wb", 1), ("b", 0)])
def test_tensors_off_the_alignment(lib, name, l):
    g = torch.Generator().manual_seed(2)
    feat, target = torch.randn((256, 48), generator=g).cuda(), torch.randn((256, 5), generator=g).cuda()
    plain, moved = surrogate(5), surrogate(5)
    t = getattr(moved.mlp, name)[l]
    flat = torch.empty(t.numel() + 8, dtype=t.dtype, device="cuda")
    view = flat[1:1 + t.numel()].view(t.shape).copy_(t)
    assert view.data_ptr() % 16
    getattr(moved.mlp, name)[l] = view
    for sur in (plain, moved):
        sur.train(feat, target, epochs=3, batch=256)
    for x, y in zip(plain.mlp.W + plain.mlp.b, moved.mlp.W + moved.mlp.b):
        assert torch.equal(x, y)
