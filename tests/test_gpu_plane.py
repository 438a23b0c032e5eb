"""The one-launch x-plane of small boxes (y-inverse, z pass and y-forward in LDS)
against the oracle: every compiled pair of lengths, the rules and the given
vorticity, and batched boxes; 1e-13 (one FP64 right-hand side) and 1e-5 (FP32),
relative L2, the solver's own bars."""
import numpy as np
import pytest

from oracle.ns import Grid

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")
L = (6.0, 2 * np.pi, 4.0)


def _field(N, seed):
    from spectraldns_amd.isotropic import random_solenoidal_field
    return random_solenoidal_field(N, L, seed=seed, k0=3.0, energy=0.5)


def _rel(a, b):
    return np.linalg.norm(a - b) / np.linalg.norm(b)


CASES = [((n0, n1, n2), "2/3-rule", 0) for n0, n1, n2 in
         [(8, 16, 16), (12, 16, 64), (16, 32, 48), (8, 48, 16), (24, 48, 48), (16, 48, 64), (32, 64, 16), (8, 64, 32),
          (16, 64, 48), (128, 64, 64), (192, 64, 64), (16, 32, 32), (8, 16, 48), (8, 32, 64), (8, 48, 32), (16, 32, 16),
          (8, 16, 32)]]
CASES += [((16, 16, 16), "3/2-rule", 0), ((8, 32, 32), "3/2-rule", 0), ((16, 32, 32), "None", 0),
          ((16, 48, 32), "2/3-rule", 1), ((8, 64, 16), "None", 0)]


@pytest.mark.parametrize("N,rule,mode", CASES)
@pytest.mark.parametrize("precision", ["double", "single"])
def test_plane_rhs(N, rule, mode, precision):
    from spectraldns_amd._abi import Plan
    print("\n[case]", N, rule, mode, precision, flush=True)
    g = Grid(N, L, "double", None if rule == "None" else rule, dealias_mode=mode)
    plan = Plan(N, L, precision, rule, True, mode)
    u0 = _field(N, 4)
    u = torch.from_numpy(u0).to(plan.complex_dtype).cuda()
    rhs = plan.compute_rhs(u, torch.empty_like(u), 0.01)
    ref = g.compute_rhs(u.cpu().numpy().astype(np.complex128), 0.01)
    assert _rel(rhs.cpu().numpy(), ref) <= (1e-13 if precision == "double" else 1e-5)
    # the given vorticity equals the curl formed in the passes
    w = torch.empty_like(u)
    plan.cross2(w, u)
    given = plan.convection_uw(u, w, torch.empty_like(u))
    own = plan.convection(u, torch.empty_like(u))
    assert _rel(given.cpu().numpy(), own.cpu().numpy()) <= (1e-13 if precision == "double" else 1e-5)


@pytest.mark.parametrize("rule,sizes", [("2/3-rule", [16, 32, 48, 64, 32]), ("3/2-rule", [16, 32, 16]),
                                        ("2/3-rule", [64, 96])])
@pytest.mark.parametrize("precision", ["double", "single"])
def test_batched_planes(rule, sizes, precision):
    from spectraldns_amd.ensemble import Ensemble
    ens = Ensemble(sizes, precision=precision, dealias=rule, dt=0.01, init="random", k0=3.0)
    ens.steps(2)
    for n, nu, u0, u in zip(sizes, ens.nu, ens.u0, ens.u_hat):
        g = Grid((n,) * 3, (2 * np.pi,) * 3, "double", rule)
        ref = u0
        for _ in range(2):
            ref = g.rk4_step(ref, 0.01, nu)
        assert _rel(u.cpu().numpy(), ref) <= (1e-12 if precision == "double" else 1e-5)
