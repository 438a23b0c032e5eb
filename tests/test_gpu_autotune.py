"""The tuner stores a choice only where there is one: passes that a box does not
launch (a small box's y and z passes are one kernel) and second names of the same
kernel are neither timed nor stored."""
import pytest

pytestmark = pytest.mark.gpu


def test_tune_of_a_box_on_the_plane_kernel():
    from spectraldns_amd.autotune import tune
    res = tune((32, 32, 32), precision="double", dealias="2/3-rule", steps=1)
    assert set(res["variants"]) == {"x_inverse", "x_forward_rk", "transforms"}
    assert all(t > 0 for ms in res["ms"].values() for t in ms)
    assert len(res["ms"]["x_forward_rk"]) == 2


def test_tune_of_a_box_on_the_passes():
    from spectraldns_amd.autotune import PASSES, tune
    res = tune((96, 96, 64), precision="single", dealias="2/3-rule", steps=1)
    assert set(res["variants"]) == set(PASSES)
    assert all(t > 0 for ms in res["ms"].values() for t in ms)
    assert len(res["ms"]["x_forward_rk"]) == 2 and len(res["ms"]["z_cross"]) == 6
    assert set(res["variants"].values()) <= {0, 1, 2, 3, 4, 5}


def test_tune_of_an_ensemble_on_the_plane_kernel():
    from spectraldns_amd.autotune import tune_batch
    res = tune_batch([32, 32, 16], precision="single", steps=2)
    assert set(res["ms"]) == {"0/16", "0/32", "4/16", "4/32"}
    assert {k for k, length, v in res["variants"]} <= {0, 4}


def test_launches():
    import math
    from spectraldns_amd._abi import Plan
    L = (2 * math.pi,) * 3
    assert [Plan((32, 32, 32), L, "double", "2/3-rule").launches(k) for k in range(-1, 6)] == [0, 1, 0, 0, 0, 1, 0]
    assert [Plan((96, 96, 64), L, "double", "2/3-rule").launches(k) for k in range(-1, 6)] == [0, 1, 1, 1, 1, 1, 0]
