"""The training step at the batch sizes where its tiling can go wrong (tiles of 32 rows, two
waves of 16, 512 blocks that loop over tiles): loss and gradients against the FP64
restatement (oracle/mlp.py).  The bound is 1e-5 of the largest gradient: FP32 sums of up to
20000 rows in blocks of 32 round by a few 2^-24 of the sum of magnitudes."""
import numpy as np
import pytest

from oracle import mlp as om

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("offset", [0, 1])
@pytest.mark.parametrize("batch", [1, 15, 16, 17, 31, 32, 33, 64, 95, 16384, 16385, 20001])
def test_loss_and_gradient(batch, offset):
    torch = pytest.importorskip("torch")
    from idefix_amd import learned
    rng = np.random.default_rng(batch)
    X = np.zeros((batch, 72), dtype=np.float32)
    x = rng.uniform(-1, 1, (batch, 8, 6))
    x[:, :, 3] = -x[:, :, 2]
    X[:, :48] = x.reshape(batch, 48)
    X[:, 48:64] = rng.uniform(0.2, 0.8, (batch, 16))
    X[:, 64:72] = rng.uniform(0.5, 1.5, (batch, 8))
    tau = rng.uniform(-0.5, 0.5, (batch, 8)).astype(np.float32)
    P = learned.unpack(learned.init_params(3))
    P["W3"] = 0.2 * rng.standard_normal(P["W3"].shape)
    p = learned.pack(P)
    tr = learned.Trainer(batch, p)
    # offset 1: rows that start 4 bytes past a multiple of 16
    buf = torch.zeros(offset + X.size, device="cuda")
    xb = buf[offset:].view(batch, 72)
    xb.copy_(torch.from_numpy(X))
    loss, grad = tr.loss_grad(xb, torch.from_numpy(tau).cuda())
    X = X.astype(np.float64)
    want_loss, want = om.loss_and_grad(learned.unpack(p), X[:, :48], tau.astype(np.float64),
                                       X[:, 48:64], X[:, 64:72])
    want = learned.pack(want).astype(np.float64)
    assert loss == pytest.approx(want_loss, rel=1e-5)
    assert np.abs(grad - want).max() <= 1e-5 * np.abs(want).max()
