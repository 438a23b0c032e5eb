"""Stage storage of the RK4 step: every combination of rule, precision and
compensation that keeps its stages differently, against the FP64 oracle, and a
box whose state is beyond a buffer descriptor's reach.

Tolerances are the solver's own: 1e-12 in FP64 and 1e-5 in FP32, relative L2."""
import numpy as np
import pytest

from oracle.ns import Grid

pytestmark = pytest.mark.gpu
L = (2 * np.pi,) * 3


def _run(N, precision, dealias, u0, steps, nu, dt, comp=False):
    import torch
    from spectraldns_amd._abi import Plan
    plan = Plan(N, L, precision, dealias)
    u = torch.from_numpy(u0).to(plan.complex_dtype).cuda()
    lo = torch.zeros_like(u) if comp else None
    diag = torch.zeros(2 * steps, dtype=torch.float64, device="cuda")
    plan.rk4_steps(u, [dt] * steps, nu, diag=diag, u_lo=lo)
    return u.cpu().numpy().astype(np.complex128) + (lo.cpu().numpy() if comp else 0), diag.cpu().numpy()


@pytest.mark.parametrize("dealias", ["2/3-rule", "3/2-rule", "None"])
@pytest.mark.parametrize("precision,comp", [("double", False), ("single", False), ("single", True)])
@pytest.mark.parametrize("N", [(16, 32, 64), (96, 16, 32)])
def test_stage_storage(N, precision, comp, dealias):
    from spectraldns_amd.isotropic import random_solenoidal_field
    nu, dt, steps = 0.01, 0.01, 3
    u0 = random_solenoidal_field(N, L, seed=5, k0=3.0, energy=0.5)
    if precision == "single":
        u0 = u0.astype(np.complex64).astype(np.complex128)
    g = Grid(N, L, "double", None if dealias == "None" else dealias)
    ref = u0.copy()
    for _ in range(steps):
        ref = g.rk4_step(ref, dt, nu)
    u, diag = _run(N, precision, dealias, u0, steps, nu, dt, comp)
    tol = 1e-12 if precision == "double" else 1e-5
    assert np.linalg.norm(u - ref) <= tol * np.linalg.norm(ref)
    assert abs(diag[-2] - g.kinetic_energy(ref)) <= tol


def test_state_beyond_a_descriptor():
    """512 x 512 x 384 in FP64: three components span 2.4 GB.  The Taylor-Green
    modes that a step reaches are those of a 32^3 box."""
    from spectraldns_amd.ensemble import taylor_green_hat
    small, big = (32, 32, 32), (512, 512, 384)
    ref = Grid(small, L, "double", "2/3-rule").rk4_step(taylor_green_hat(small), 0.01, 0.000625)
    u0 = np.zeros((3, 512, 512, 193), dtype=np.complex128)
    s = taylor_green_hat(small)
    k = np.r_[0:8, -8:0]
    pick = lambda a: a[:, k][:, :, k][:, :, :, :8]  # noqa: E731
    for a in k:
        for b in k:
            u0[:, a, b, :8] = s[:, a, b, :8]
    u, diag = _run(big, "double", "2/3-rule", u0, 1, 0.000625, 0.01)
    assert np.linalg.norm(pick(u) - pick(ref)) <= 1e-12 * np.linalg.norm(ref)
    assert abs(np.linalg.norm(u) - np.linalg.norm(ref)) <= 1e-12 * np.linalg.norm(ref)
