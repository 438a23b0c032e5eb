"""Column tiles of the x and y passes: boxes whose tile counts are below one run
of tiles per XCD, whole runs, and runs with a remainder; rows shorter than a tile
(kept and dropped modes in one tile) and tiles without kept modes.  One RK4 step
and a transform against the FP64 oracle; tolerances are the solver's own, 1e-12
in FP64 and 1e-5 in FP32, relative L2."""
import numpy as np
import pytest

from oracle.ns import Grid

pytestmark = pytest.mark.gpu
L = (2 * np.pi,) * 3


@pytest.mark.parametrize("dealias", ["2/3-rule", "3/2-rule"])
@pytest.mark.parametrize("precision", ["double", "single"])
@pytest.mark.parametrize("N", [(96, 64, 8), (32, 64, 48), (48, 96, 128), (64, 128, 256), (128, 192, 96)])
def test_tile_runs(N, precision, dealias):
    import torch
    from spectraldns_amd._abi import Plan
    from spectraldns_amd.isotropic import random_solenoidal_field
    u0 = random_solenoidal_field(N, L, seed=7, k0=3.0, energy=0.5)
    if precision == "single":
        u0 = u0.astype(np.complex64).astype(np.complex128)
    tol = 1e-12 if precision == "double" else 1e-5
    plan = Plan(N, L, precision, dealias)
    u = torch.from_numpy(u0).to(plan.complex_dtype).cuda()
    x = np.random.default_rng(7).standard_normal((3,) + N)
    x = torch.from_numpy(x).to(plan.real_dtype).cuda()
    xh = torch.empty_like(u)
    plan.forward(x, xh)
    xref = np.fft.rfftn(x.cpu().numpy().astype(np.float64), axes=(1, 2, 3)) / np.prod(N)
    assert np.linalg.norm(xh.cpu().numpy() - xref) <= tol * np.linalg.norm(xref)
    y = torch.empty_like(x)
    plan.backward(xh, y)
    assert torch.linalg.norm(y - x) <= tol * torch.linalg.norm(x)
    ref = Grid(N, L, "double", dealias).rk4_step(u0.copy(), 0.01, 0.01)
    plan.rk4_steps(u, [0.01], 0.01)
    assert np.linalg.norm(u.cpu().numpy() - ref) <= tol * np.linalg.norm(ref)
