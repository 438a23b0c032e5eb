"""Closure kernels on grids whose sides are no multiples of their tiles: forward
pass, loss and gradients against the closure oracle with bf16 storage.

Tolerances: a bf16 value is 2^-9 off at most, and a pre-activation that rounds
the other way changes an output by about that share of one of many terms, so
5e-3 forward and 2e-2 for gradients (relative L2), as for the cubic grid."""
import numpy as np
import pytest

from oracle import closure as OC

pytestmark = pytest.mark.gpu


def _split(p):
    W, b, o = [], [], 0
    for cin, cout in ((3, 32), (32, 32), (32, 6)):
        W.append(p[o:o + 27 * cout * cin].reshape(27, cout, cin))
        o += 27 * cout * cin
        b.append(p[o:o + cout])
        o += cout
    return W, b


def _rel(a, b):
    return np.linalg.norm(np.asarray(a, np.float64) - b) / np.linalg.norm(b)


@pytest.mark.parametrize("N", [(16, 8, 32), (5, 16, 256), (12, 4, 256), (4, 6, 512), (16, 8, 96), (4, 32, 32)])
def test_shapes(N):
    import torch
    from spectraldns_amd.closure import Closure, init_params
    rng = np.random.default_rng(3)
    p = init_params(2) + 0.02 * rng.standard_normal(init_params(2).size).astype(np.float32)
    c = Closure(N, params=p)
    c.in_scale, c.out_scale = 1.5, 0.5
    u = rng.standard_normal((3,) + N).astype(np.float32)
    t = 0.3 * rng.standard_normal((6,) + N).astype(np.float32)
    ud, td = torch.from_numpy(u).cuda(), torch.from_numpy(t).cuda()
    tau = c.forward(ud).cpu().numpy()
    loss = float(c.train_step(ud, td).item())
    W, b = _split(p)
    x = np.moveaxis(u * np.float32(1.5), 0, -1)
    tt = np.moveaxis(t * np.float32(2.0), 0, -1)
    y, saved = OC.forward(x, W, b, bf16_storage=True)
    dW, db = OC.backward(y, tt, saved, bf16_storage=True)
    assert _rel(tau, 0.5 * np.moveaxis(y, -1, 0)) < 5e-3
    assert abs(loss - OC.loss(y, tt)) <= 1e-3 * OC.loss(y, tt)
    gW, gb = _split(c.grad.cpu().numpy())
    for layer in range(3):
        assert _rel(gW[layer], dW[layer]) < 2e-2 and _rel(gb[layer], db[layer]) < 2e-2
