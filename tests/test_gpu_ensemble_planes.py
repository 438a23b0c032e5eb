"""Which ensembles run their y, z and y passes as plane launches: one launch per side
and stage, which pays off for few sides or many planes.  Ensembles on both sides of
the line against the single-box path: 3 steps, 1e-12 (FP64) or 1e-5 (FP32), relative L2."""
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("sizes,precision,rule,plane", [
    ([32], "single", "2/3-rule", True), ([64], "double", "2/3-rule", False), ([64, 64], "double", "2/3-rule", True),
    ([16, 32], "single", "2/3-rule", True), ([16, 32], "single", "3/2-rule", False),
    ([32, 48] * 2, "double", "2/3-rule", False), ([32, 48] * 4, "double", "2/3-rule", True),
    ([16, 24, 32, 48], "single", "2/3-rule", False), ([16, 24, 32, 48] * 8, "single", "2/3-rule", True),
    ([16, 24, 32, 48] * 8, "double", "2/3-rule", False), ([32, 48, 64] * 4, "single", "2/3-rule", False),
    ([32, 96], "single", "2/3-rule", False)])
def test_plane_rule_of_ensembles(sizes, precision, rule, plane):
    import torch
    from spectraldns_amd._abi import Plan
    from spectraldns_amd.ensemble import Ensemble
    print("\n[case]", sizes[:4], len(sizes), precision, rule, flush=True)
    ens = Ensemble(sizes, precision=precision, dealias=rule, init="random", tuned=False)
    assert [ens.batch.launches(k) for k in range(5)] == [True] + [not plane] * 3 + [True]
    start = [u.clone() for u in ens.u_hat]
    ens.steps(3)
    seen = set()
    for i, (n, u) in enumerate(zip(sizes, start)):
        if n in seen:
            continue
        seen.add(n)
        p = Plan((n,) * 3, (6.283185307179586,) * 3, precision, rule, tuned=False)
        p.rk4_steps(u, [ens.dt[i]] * 3, ens.nu[i])
        rel = float(torch.linalg.vector_norm(u - ens.u_hat[i]) / torch.linalg.vector_norm(u))
        assert rel <= (1e-12 if precision == "double" else 1e-5), (n, rel)
