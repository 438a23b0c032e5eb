"""The VV and MHD solvers' fused right-hand side and RK4 step against the same
module running step by step (a replaced hook sends it there), on random fields
with every rule: one RHS within 1e-13 (FP64) or 2e-6 (FP32, two transforms of
relative error about 3e-7 each way), a step within 1e-14 / 1e-6 of the state."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")


def _context(name, N, precision, dealias, mask):
    from spectraldns_amd import config, get_solver
    conv = "Divergence" if name == "MHD" else "Vortex"
    config.update({"nu": 0.02, "dt": 0.01, "T": 1e9, "eta": 0.03, "L": [6.0, 2 * np.pi, 4.0], "convection": conv,
                   "dealias": dealias, "precision": precision, "integrator": "RK4", "mask_nyquist": mask})
    try:
        solver = get_solver(parse_args=[name])
        config.params["N"] = list(N)
        c = solver.get_context()
        solver.conv = solver.getConvection(conv)
        return solver, c, config
    finally:
        config.params.pop("N", None)
        config.update({"convection": "Vortex", "dealias": "2/3-rule", "precision": "double", "mask_nyquist": True,
                       "L": [2 * np.pi] * 3})


def _rel(a, b):
    return float((a - b).abs().pow(2).sum().sqrt() / b.abs().pow(2).sum().sqrt())


@pytest.mark.parametrize("name", ["VV", "MHD"])
@pytest.mark.parametrize("precision", ["double", "single"])
@pytest.mark.parametrize("N,dealias,mask", [((16, 32, 64), "2/3-rule", True), ((96, 16, 32), "3/2-rule", True),
                                            ((24, 72, 16), "2/3-rule", False), ((32, 64, 128), "None", True),
                                            ((64, 32, 48), "3/2-rule", False), ((8, 16, 32), "3/2-rule", True)])
def test_fused_equals_steps(name, N, precision, dealias, mask, monkeypatch):
    print("\n[case]", name, N, precision, dealias, mask, flush=True)
    solver, c, config = _context(name, N, precision, dealias, mask)
    assert (c["T"] if name == "MHD" else c["VT"]).plan.fused_stages
    g = torch.Generator(device="cuda").manual_seed(3)
    phys = torch.randn((c.u.shape[0],) + N, generator=g, device="cuda", dtype=torch.float64)
    start = torch.fft.rfftn(phys, dim=(1, 2, 3), norm="forward").to(c.u.dtype)  # with mean, gradients and Nyquist modes
    start[:, 0, 0, 0] = 0.1
    c.u.copy_(start)
    if name == "VV":
        c.Source.copy_(0.1 * start)
    fused = solver.ComputeRHS(torch.empty_like(c.dU), c.u, solver, **c).clone()
    p_fused = c.P_hat.clone() if name == "MHD" else None
    step = solver.getintegrator(c.dU, c.u, solver, c)
    step()
    after, p_after = c.u.clone(), (c.P_hat.clone() if name == "MHD" else None)
    # step by step
    hook = "add_linear" if name == "VV" else "add_pressure_diffusion"
    own = getattr(solver, hook)
    monkeypatch.setattr(solver, hook, lambda *a, **k: own(*a, **k))
    c.u.copy_(start)
    ref = solver.ComputeRHS(torch.empty_like(c.dU), c.u, solver, **c).clone()
    tol = 1e-13 if precision == "double" else 2e-6
    assert _rel(fused, ref) <= tol
    if name == "MHD":
        assert _rel(p_fused, c.P_hat) <= tol
    step()
    assert _rel(after, c.u) <= (1e-14 if precision == "double" else 1e-6)
    if name == "MHD":
        assert _rel(p_after, c.P_hat) <= 10 * tol
