"""The plain transforms at sizes on both sides of the rules for their stores (row
length, output size) and for the order of their tiles (x lines, short rows),
against NumPy in FP64; 1e-13 (FP64) or 2e-6 (FP32, three passes of relative error
about 2e-7 each), relative L2."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision", ["double", "single"])
@pytest.mark.parametrize("N", [(64, 64, 64), (96, 96, 96), (16, 16, 1536), (32, 32, 512), (128, 128, 16), (16, 16, 32),
                               (1024, 16, 128), (16, 1024, 64), (72, 48, 144), (128, 96, 192), (256, 64, 32)])
def test_transforms(N, precision):
    import torch
    from spectraldns_amd._abi import Plan
    p = Plan(N, (2 * np.pi,) * 3, precision, "2/3-rule", tuned=False)
    x = np.random.default_rng(3).standard_normal((3,) + N)
    tol = 1e-13 if precision == "double" else 2e-6
    xd = torch.from_numpy(x).to(p.real_dtype).cuda()
    xh = torch.full((3,) + p.spectral_shape, float("nan"), dtype=p.complex_dtype, device="cuda")
    p.forward(xd, xh)
    ref = np.fft.rfftn(x, axes=(1, 2, 3)) / np.prod(N)
    assert np.linalg.norm(xh.cpu().numpy() - ref) <= tol * np.linalg.norm(ref)
    y = torch.full_like(xd, float("nan"))
    p.backward(xh, y)
    assert np.linalg.norm(y.cpu().numpy() - x) <= tol * np.linalg.norm(x)
    one = torch.full_like(xh[:1], float("nan"))   # one component: a third of the output
    p.forward(xd[1:2].contiguous(), one)
    assert np.linalg.norm(one[0].cpu().numpy() - ref[1]) <= tol * np.linalg.norm(ref[1])
