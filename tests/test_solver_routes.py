"""Which route the solvers' right-hand side and RK4 step take, with a plan that
only records its calls: the fused route is for the module's own steps alone, and
whatever it cannot serve goes step by step."""
from functools import wraps
from types import SimpleNamespace

import numpy as np
import pytest

torch = pytest.importorskip("torch")

FUSED = ("compute_rhs", "rk4_steps", "vv_rhs", "vv_rk4_steps", "mhd_rhs", "mhd_rk4_steps")


class _Plan:
    """Stands for a Plan: notes the name of each method called on it."""
    nyquist_masked, fused_stages, mhd_fused = True, True, True
    dealiased_shape, real_dtype, device = (2, 2, 2), torch.float64, "cpu"

    def __init__(self):
        self.calls = []

    def __getattr__(self, name):
        if name.startswith("__"):
            raise AttributeError(name)

        def method(*args, **kw):
            self.calls.append(name)
            return args[0] if args else None
        return method


def _setup(name):
    import importlib
    from spectraldns_amd import config
    module = importlib.import_module("spectraldns_amd.solvers." + name)
    plan = _Plan()
    ncomp = 6 if name == "MHD" else 3
    u, dU = (torch.zeros((ncomp, 2, 2, 2), dtype=torch.complex128) for _ in range(2))
    space = SimpleNamespace(plan=plan, backward=lambda a, b: b)
    c = config.AttributeDict(T=space, VT=space, Tp=space, VTp=space, VMp=space, mask=1, Source=torch.zeros_like(dU[:3]),
                             P_hat=torch.zeros_like(u[0]), K=space, K2=space, K_over_K2=space, u=u, dU=dU, W_hat=u,
                             work=_Work(), ub_dealias=None, u_dealias=u, ZZ_hat=torch.zeros((3, 3, 2, 2, 2)),
                             float=np.float64)
    solver = SimpleNamespace(**{k: v for k, v in vars(module).items() if not k.startswith("__")})
    solver.conv = module.getConvection("Divergence" if name == "MHD" else "Vortex")
    return module, solver, c, plan


class _Work(dict):
    def __missing__(self, key):
        return torch.zeros_like(key[0])


def _routes(plan):
    fused = [n for n in plan.calls if n in FUSED]
    plan.calls.clear()
    return fused


@pytest.fixture
def rk4():
    from spectraldns_amd import config
    old = dict(config.params)
    config.params.update(integrator="RK4", nu=0.1, eta=0.1, dt=0.1, compensated=False, precision="double")
    yield config.params
    config.params.clear()
    config.params.update(old)


@pytest.mark.parametrize("name,rhs,step", [("NS", "compute_rhs", "rk4_steps"), ("VV", "vv_rhs", "vv_rk4_steps"),
                                           ("MHD", "mhd_rhs", "mhd_rk4_steps")])
def test_own_steps_are_fused(name, rhs, step, rk4):
    from spectraldns_amd.maths.integrators import getintegrator
    module, solver, c, plan = _setup(name)
    solver.ComputeRHS(torch.empty_like(c.dU), c.u, solver, **c)
    assert _routes(plan) == [rhs]
    getintegrator(c.dU, c.u, solver, c)()
    assert _routes(plan) == [step]


@pytest.mark.parametrize("name,hook", [("VV", "add_linear"), ("MHD", "add_pressure_diffusion")])
@pytest.mark.parametrize("as_module", [True, False])
def test_replaced_hook_is_called(name, hook, as_module, rk4, monkeypatch):
    """Also where the solver is the module itself, whose name the hook then is."""
    from spectraldns_amd.maths.integrators import getintegrator
    module, solver, c, plan = _setup(name)
    if as_module:
        monkeypatch.setattr(module, "conv", solver.conv, raising=False)
        solver = module
    seen = []
    monkeypatch.setattr(solver, hook, lambda rhs, *a, **k: seen.append(1) or rhs)
    solver.ComputeRHS(torch.empty_like(c.dU), c.u, solver, **c)
    assert seen == [1] and _routes(plan) == []
    getintegrator(c.dU, c.u, solver, c)()
    assert len(seen) == 5 and _routes(plan) == []


def test_replaced_cross_product_is_called(rk4, monkeypatch):
    """The VV convection calls the cross2 of its module."""
    module, solver, c, plan = _setup("VV")
    seen = []
    monkeypatch.setattr(module, "cross2", lambda out, *a: seen.append(1) or out)
    solver.ComputeRHS(torch.empty_like(c.dU), c.u, solver, **c)
    assert seen == [1] and _routes(plan) == []


@pytest.mark.parametrize("name", ["NS", "VV", "MHD"])
def test_wrapped_convection_is_called(name, rk4):
    """functools.wraps copies the attributes of the function it wraps."""
    from spectraldns_amd.maths.integrators import getintegrator
    module, solver, c, plan = _setup(name)
    own, seen = solver.conv, []

    @wraps(own)
    def conv(rhs, *args, **kw):
        seen.append(1)
        return rhs
    solver.conv = conv
    solver.ComputeRHS(torch.empty_like(c.dU), c.u, solver, **c)
    assert seen == [1] and _routes(plan) == []
    getintegrator(c.dU, c.u, solver, c)()
    assert len(seen) == 5 and _routes(plan) == []


def test_mhd_solver_without_the_module_helpers(rk4):
    """ComputeRHS needs conv and add_pressure_diffusion of its solver argument, no more."""
    from spectraldns_amd.solvers import MHD
    _, full, c, plan = _setup("MHD")
    solver = SimpleNamespace(conv=full.conv, add_pressure_diffusion=MHD.add_pressure_diffusion)
    MHD.ComputeRHS(torch.empty_like(c.dU), c.u, solver, **c)
    assert _routes(plan) == ["mhd_rhs"]


def test_mhd_replaced_helper_of_the_module(rk4, monkeypatch):
    """The convection calls the helpers of its own module."""
    module, solver, c, plan = _setup("MHD")
    seen = []
    monkeypatch.setattr(module, "set_Elsasser", lambda c, zz, K: seen.append(1) or c)
    solver.ComputeRHS(torch.empty_like(c.dU), c.u, solver, **c)
    assert seen == [1] and _routes(plan) == []


def test_vv_source_that_overlaps_the_state(rk4):
    """A Source shifted into the state is read after the state's update by no
    stage-by-stage step; the fused last stage writes the state while it reads the
    Source, so only an identical or a separate Source may take it."""
    from spectraldns_amd.maths.integrators import getintegrator
    module, solver, c, plan = _setup("VV")
    both = torch.zeros((4,) + tuple(c.u.shape[1:]), dtype=c.u.dtype)
    for source, fused in ((both[:3], True), (both[1:], False), (torch.zeros_like(c.u), True)):
        c.u = c.W_hat = both[:3]
        c.Source = source
        getintegrator(c.dU, c.u, solver, c)()
        assert (_routes(plan) == ["vv_rk4_steps"]) == fused


@pytest.mark.parametrize("name,hook", [("VV", "add_linear"), ("MHD", "add_pressure_diffusion")])
def test_stage_arrays_exist_before_the_first_step(name, hook, rk4):
    """A step that runs stage by stage allocates nothing (it may be captured)."""
    from spectraldns_amd.maths.integrators import getintegrator
    module, solver, c, plan = _setup(name)
    setattr(solver, hook, lambda rhs, *a, **k: rhs)
    step = getintegrator(c.dU, c.u, solver, c)
    clones = []

    class State(torch.Tensor):
        def clone(self, *a, **k):
            clones.append(1)
            return super().clone(*a, **k)
    c2_u = c.u.as_subclass(State)
    step2 = getintegrator(c.dU, c2_u, solver, c)
    assert len(clones) == 2
    step()
    step2()
    assert len(clones) == 2


def test_stage_arrays_of_the_other_convections(rk4):
    from spectraldns_amd.maths.integrators import getintegrator
    module, solver, c, plan = _setup("NS")
    solver.conv = module.getConvection("Standard")
    clones = []

    class State(torch.Tensor):
        def clone(self, *a, **k):
            clones.append(1)
            return super().clone(*a, **k)
    getintegrator(c.dU, c.u.as_subclass(State), solver, c)
    assert len(clones) == 2


def test_mhd_without_memory_for_the_workspace(monkeypatch):
    """No memory left for the fused workspace: the step-by-step arrays, which the
    context holds, still serve."""
    from spectraldns_amd._abi import Plan

    def plan():
        p = object.__new__(Plan)
        p._h = None
        p._lib = SimpleNamespace(sdns_mhd_workspace_bytes=lambda h: 1024, sdns_fused_stages=lambda h: 1)
        p.device = torch.device("cpu")
        return p
    asked = []

    def no_memory(*a, **k):
        asked.append(1)
        raise torch.OutOfMemoryError("out of memory")
    with monkeypatch.context() as m:
        m.setattr(torch, "empty", no_memory)
        p = plan()
        assert not p.mhd_fused and not p.mhd_fused and asked == [1]
    p = plan()
    assert p.mhd_fused
    ptr, nbytes = p._mhd_workspace()
    assert ptr.value % 256 == 0 and nbytes >= 1024


def test_mhd_plan_without_the_workspace_goes_step_by_step(rk4, monkeypatch):
    from spectraldns_amd.maths.integrators import getintegrator
    module, solver, c, plan = _setup("MHD")
    plan.mhd_fused = False
    solver.ComputeRHS(torch.empty_like(c.dU), c.u, solver, **c)
    assert _routes(plan) == []
    getintegrator(c.dU, c.u, solver, c)()
    assert _routes(plan) == []
