"""tt_mlp_train_step against the same step called layer by layer."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


def surrogate(seed):
    from turbulence_tracing_amd.surrogate import Norm, Surrogate
    return Surrogate(Norm(np.zeros(48, np.float32), np.ones(48, np.float32), 1.0, 1.0, 1.0), seed=seed)


class Layered:
    """Stands in for Surrogate._fused_step: the layer-by-layer path."""

    def __init__(self, sur):
        self.sur = sur

    def __enter__(self):
        self.sur._fused_step = lambda *a: None
        return self.sur

    def __exit__(self, *a):
        del self.sur._fused_step


# edges of a chunk of 32 rows, of a block's 16, of a bias group's 256, of the
# gradients' splits (2048: below it one product per weight, so the same bits) and
# of the two row-block sizes (8192)
@pytest.mark.parametrize("batch", [1, 16, 31, 33, 257, 2047, 2048, 8191, 8192, 8209])
def test_fused_step_matches_layers(lib, batch):
    g = torch.Generator().manual_seed(batch)
    feat = torch.randn((batch, 48), generator=g).cuda()
    target = torch.randn((batch, 5), generator=g).cuda()
    a, b = surrogate(5), surrogate(5)
    assert a._fused_step(a.standardize(feat), target, batch, 0.0) is not None
    la = a.train(feat, target, epochs=1, batch=batch, wd=1e-3)
    with Layered(b):
        lb = b.train(feat, target, epochs=1, batch=batch, wd=1e-3)
    assert a.mlp.step == b.mlp.step == 1
    # the loss sums are fp64 sums of the same fp32 terms
    np.testing.assert_allclose(la[0], lb[0], rtol=1e-12)
    for name in ("dW", "db"):
        for l, (x, y) in enumerate(zip(getattr(a.mlp, name), getattr(b.mlp, name))):
            x, y = x.double(), y.double()
            if batch < 2048 and name == "dW":
                assert torch.equal(x, y), (name, l)
            else:
                # the same fp32 partial sums, added in another order: rounding
                # grows like sqrt(n) steps of 2^-24 of the running sum at most
                assert float((x - y).norm()) <= 4 * batch ** 0.5 * 2.0 ** -24 * float(y.norm()), (name, l)
    # Adam's update follows from the step's own gradient
    for l in range(4):
        gw = b.mlp.dW[l]
        same = a.mlp.dW[l] == gw
        assert torch.equal(a.mlp.W[l][same], b.mlp.W[l][same])
        assert torch.equal(a.mlp.Wb[l], a.mlp.W[l].to(torch.bfloat16))


@pytest.mark.parametrize("batch", [96, 8192])
def test_fused_steps_track_the_layers(lib, batch):
    """Several steps: the transposed copies the backward reads are refreshed
    with the weights, and strided targets and a final partial batch are served."""
    n, g = 5 * batch + 7, torch.Generator().manual_seed(1)
    feat = torch.randn((n, 48), generator=g).cuda()
    wide = torch.randn((n, 9), generator=g).cuda()
    wide[:, 2:7] = torch.tanh(feat[:, :5]) + 0.1 * wide[:, 2:7]
    target = wide[:, 2:7]
    a, b = surrogate(2), surrogate(2)
    la = a.train(feat, target, epochs=2, batch=batch)
    with Layered(b):
        lb = b.train(feat, target, epochs=2, batch=batch)
    # ten Adam steps of at most 2e-3 each; a stale transpose would change the
    # loss by far more than the order of the gradient sums does
    np.testing.assert_allclose(np.array(la), np.array(lb), rtol=1e-3)
    for x, y in zip(a.mlp.W, b.mlp.W):
        assert float((x - y).norm()) <= 1e-2 * float(y.norm())
