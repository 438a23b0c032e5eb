"""What a fused VV or MHD step leaves behind, and the sizes whose grids fill the
chip: against the same module running step by step (a replaced hook sends it
there), whose arithmetic the solver tests hold to the oracle.

Tolerances: a step 1e-14 (FP64) or 1e-6 (FP32) of the state; a right-hand side,
which two transforms of relative error about 3e-7 each way separate, 1e-13 or
2e-6, and ten times that where the stage states differ by their own rounding."""
import numpy as np
import pytest

from test_gpu_fused_solvers import _context, _rel

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")


def _start(c, N, seed=3, steep=2.0):
    g = torch.Generator(device="cuda").manual_seed(seed)
    phys = torch.randn((c.u.shape[0],) + tuple(N), generator=g, device="cuda", dtype=torch.float64)
    u = torch.fft.rfftn(phys, dim=(1, 2, 3), norm="forward")
    k = [torch.fft.fftfreq(n, 1.0 / n, device="cuda") for n in N[:2]] + \
        [torch.fft.rfftfreq(N[2], 1.0 / N[2], device="cuda")]
    k2 = k[0][:, None, None] ** 2 + k[1][None, :, None] ** 2 + k[2] ** 2
    return u * (1 + k2) ** (-0.5 * steep)


def _by_steps(solver, name, monkeypatch):
    hook = "add_linear" if name == "VV" else "add_pressure_diffusion"
    own = getattr(solver, hook)
    monkeypatch.setattr(solver, hook, lambda *a, **k: own(*a, **k))


@pytest.mark.parametrize("name", ["VV", "MHD"])
@pytest.mark.parametrize("precision", ["double", "single"])
def test_step_leaves_the_last_right_hand_side(name, precision, monkeypatch):
    """context.dU after an RK4 step holds the last stage's right-hand side."""
    for N, dealias in (((16, 32, 64), "2/3-rule"), ((32, 16, 16), "3/2-rule"), ((256, 16, 32), "2/3-rule")):
        print("\n[case]", name, precision, N, dealias, flush=True)
        solver, c, config = _context(name, N, precision, dealias, True)
        start = _start(c, N).to(c.u.dtype)
        c.u.copy_(start)
        step = solver.getintegrator(c.dU, c.u, solver, c)
        step()
        got, after = c.dU.clone(), c.u.clone()
        with monkeypatch.context() as m:
            _by_steps(solver, name, m)
            c.u.copy_(start)
            c.dU.zero_()
            solver.getintegrator(c.dU, c.u, solver, c)()
            assert float(c.dU.abs().max()) > 0
            assert _rel(got, c.dU) <= (1e-12 if precision == "double" else 2e-5)
            assert _rel(after, c.u) <= (1e-14 if precision == "double" else 1e-6)


@pytest.mark.parametrize("precision", ["double", "single"])
def test_vv_source_is_the_state(precision, monkeypatch):
    """A Source that is the vorticity itself acts as its value at the step's start."""
    N = (16, 32, 64)
    print("\n[case] VV", precision, N, flush=True)
    solver, c, config = _context("VV", N, precision, "2/3-rule", True)
    start = _start(c, N).to(c.u.dtype)
    c.u.copy_(start)
    c.Source = c.u
    solver.getintegrator(c.dU, c.u, solver, c)()
    after = c.u.clone()
    with monkeypatch.context() as m:
        _by_steps(solver, "VV", m)
        c.u.copy_(start)
        solver.getintegrator(c.dU, c.u, solver, c)()
    assert _rel(after, c.u) <= (1e-14 if precision == "double" else 1e-6)
    c.u.copy_(start)
    c.Source = start.clone()
    solver.getintegrator(c.dU, c.u, solver, c)()
    assert torch.equal(after, c.u)


@pytest.mark.parametrize("name", ["VV", "MHD"])
@pytest.mark.parametrize("precision", ["double", "single"])
@pytest.mark.parametrize("N,dealias", [((256, 32, 64), "2/3-rule"), ((64, 128, 256), "2/3-rule"),
                                       ((128, 64, 128), "None"), ((128, 32, 64), "3/2-rule")])
def test_whole_tiles(name, precision, N, dealias, monkeypatch):
    """x lines of 128 points and more, and grids of 512 blocks and more, whose
    column tiles are not divided."""
    print("\n[case]", name, N, precision, dealias, flush=True)
    solver, c, config = _context(name, N, precision, dealias, True)
    start = _start(c, N).to(c.u.dtype)
    c.u.copy_(start)
    fused = solver.ComputeRHS(torch.empty_like(c.dU), c.u, solver, **c).clone()
    solver.getintegrator(c.dU, c.u, solver, c)()
    after = c.u.clone()
    with monkeypatch.context() as m:
        _by_steps(solver, name, m)
        c.u.copy_(start)
        ref = solver.ComputeRHS(torch.empty_like(c.dU), c.u, solver, **c).clone()
        assert _rel(fused, ref) <= (1e-13 if precision == "double" else 2e-6)
        solver.getintegrator(c.dU, c.u, solver, c)()
        assert _rel(after, c.u) <= (1e-14 if precision == "double" else 1e-6)


@pytest.mark.parametrize("name", ["VV", "MHD"])
def test_many_single_precision_steps(name, monkeypatch):
    """50 FP32 steps of a smooth field: no further from FP64 than the stage by
    stage step with its accumulator, whose error is the yardstick (1.5 times it:
    the two round differently)."""
    N = (32, 32, 32)
    print("\n[case]", name, N, "50 steps", flush=True)

    def run(precision, by_steps):
        solver, c, config = _context(name, N, precision, "2/3-rule", True)
        u = _start(c, N, 5, 4.0).to(torch.complex64)
        c.u.copy_(u * (0.5 / float(u.abs().pow(2).sum().sqrt())))
        with monkeypatch.context() as m:
            if by_steps:
                _by_steps(solver, name, m)
            step = solver.getintegrator(c.dU, c.u, solver, c)
            for _ in range(50):
                step()
        return c.u.to(torch.complex128).clone()
    ref = run("double", True)
    fused, steps = _rel(run("single", False), ref), _rel(run("single", True), ref)
    print("fused %.2e, stage by stage %.2e" % (fused, steps), flush=True)
    assert fused <= 1.5 * steps and fused <= 1e-5
