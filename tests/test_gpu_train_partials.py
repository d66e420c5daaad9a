"""The gradients of a training step of 2048 rows and more, where a weight's is
the sum of one partial sum for every 1024 rows and a bias' one for every 256:
tt_mlp_train_step gives the partial sums of tt_gemm_bf16 and tt_bias_grad, added
in order of the rows, bit for bit.  (Called layer by layer they are added by
atomics, in any order.)"""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


def in_order(parts):
    s = torch.zeros_like(parts[0])
    for p in parts:
        s = s + p
    return s


@pytest.mark.parametrize("batch", [2048, 8192, 8209, 16384])
def test_gradients_are_the_partial_sums_in_order(lib, batch):
    from turbulence_tracing_amd import _lib
    from turbulence_tracing_amd.surrogate import Norm, Surrogate
    sur = Surrogate(Norm(np.zeros(48, np.float32), np.ones(48, np.float32), 1.0, 1.0, 1.0), seed=5)
    m = sur.mlp
    g = torch.Generator().manual_seed(batch)
    X = sur.standardize(torch.randn((batch, 48), generator=g).cuda())
    T = torch.randn((batch, 5), generator=g).cuda()
    # forward, loss and activation gradients layer by layer
    Y = torch.empty((batch, 8), device="cuda")
    dZ = torch.empty((batch, 8), dtype=torch.bfloat16, device="cuda")
    loss = torch.zeros((2, 2), dtype=torch.float64, device="cuda")
    m.forward(X, out=Y, keep=True)
    lib.tt_surrogate_loss(Y.data_ptr(), 8, T.data_ptr(), 5, dZ.data_ptr(), 8, batch, 5, sur.w_reg.data_ptr(), 2,
                          sur.err_lo.data_ptr(), sur.err_hi.data_ptr(), float(sur.tau), 8, loss[0].data_ptr(),
                          _lib.stream_ptr())
    want = [None] * 4
    for l in range(3, -1, -1):
        fin, fout = m.dims[l], m.dims[l + 1]
        H, _ = m.cache[l]
        dW = [torch.zeros((fout, fin), device="cuda") for _ in range(0, batch, 1024)]
        for i, p in enumerate(dW):
            k = min(1024, batch - 1024 * i)
            m._gemm(dZ[1024 * i:], 1, fout, H[1024 * i:], fin, 1, fout, fin, k, Cf=p, ldc=fin, ksplit=1024)
        db = [torch.zeros(fout, device="cuda") for _ in range(0, batch, 256)]
        for i, p in enumerate(db):
            lib.tt_bias_grad(dZ[256 * i:].data_ptr(), min(256, batch - 256 * i), fout, fout, p.data_ptr(),
                             _lib.stream_ptr())
        want[l] = in_order(dW), in_order(db)
        if l > 0:
            dH = torch.empty((batch, fin), device="cuda")
            m._gemm(dZ, fout, 1, m.Wb[l], fin, 1, batch, fin, fout, Cf=dH, ldc=fin)
            dZ = torch.empty((batch, fin), dtype=torch.bfloat16, device="cuda")
            lib.tt_gelu_backward(dH.data_ptr(), None, m.cache[l - 1][1].data_ptr(), dZ.data_ptr(), batch * fin,
                                 _lib.stream_ptr())
    sur._fused_step(X, T, batch, 0.0)(torch.arange(batch, device="cuda"), 1e-3, loss[1])
    for l in range(4):
        assert torch.equal(m.dW[l], want[l][0]), l
        assert torch.equal(m.db[l], want[l][1]), l
    # fp64 sums of the same fp32 terms
    np.testing.assert_allclose(loss[1].cpu().numpy(), loss[0].cpu().numpy(), rtol=1e-12)
