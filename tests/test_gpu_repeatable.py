"""The same call on the same data gives the same bits: right-hand sides and steps
of the three solvers in FP64, whose 16-byte stores were once overwritten now and
then, and the x-forward pass of every length class.  No tolerance."""
import numpy as np
import pytest

from test_gpu_fused_solvers import _context

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")


def _random(shape, dtype):
    g = torch.Generator(device="cuda").manual_seed(3)
    phys = torch.randn(shape, generator=g, device="cuda", dtype=torch.float64)
    return torch.fft.rfftn(phys, dim=(1, 2, 3), norm="forward").to(dtype)


@pytest.mark.parametrize("name", ["NS", "VV", "MHD"])
@pytest.mark.parametrize("precision", ["double", "single"])
@pytest.mark.parametrize("N,dealias", [((128, 64, 128), "None"), ((256, 32, 64), "2/3-rule"), ((64, 128, 256), "2/3-rule"),
                                       ((64, 32, 32), "3/2-rule"), ((32, 32, 32), "2/3-rule")])
def test_same_bits(name, precision, N, dealias):
    print("\n[case]", name, N, precision, dealias, flush=True)
    solver, c, config = _context(name, N, precision, dealias, True)
    start = _random((c.u.shape[0],) + N, c.u.dtype)
    step = solver.getintegrator(c.dU, c.u, solver, c)
    first = None
    for _ in range(6):
        c.u.copy_(start)
        rhs = solver.ComputeRHS(torch.empty_like(c.u), c.u, solver, **c).clone()
        step()
        if first is None:
            first = rhs, c.u.clone()
            assert bool(torch.isfinite(torch.view_as_real(rhs)).all())
        assert torch.equal(torch.view_as_real(rhs), torch.view_as_real(first[0]))
        assert torch.equal(torch.view_as_real(c.u), torch.view_as_real(first[1]))
