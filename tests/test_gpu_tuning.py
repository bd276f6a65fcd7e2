"""Launch shapes: every one accepted, none changes a result.

The flux shapes apply where each class has a launch of its own, so the cloud
here is above the joint launch's sizes (flux_small in kernels_flux_fused.hip).
"""

import numpy as np
import pytest

from conftest import PKG

pytestmark = pytest.mark.gpu
solver = PKG.solver
pc = PKG.pointcloud


def shells(n):
    return pc.ellipsoid_cloud(n * 8 // 100, n * 4 // 100, n - n * 12 // 100, seed=9, order="morton", workers=8)


@pytest.fixture(scope="module")
def large():
    return shells(560000)


# caps the FP64 kernels have no variant for (3 and more) run the default one
@pytest.mark.parametrize("precision,shapes", [
    ("fp64", [(64, 1), (128, 2), (256, 3), (64, 4), (128, 6), (256, 0)]),
    ("mixed", [(64, 1), (256, 1), (128, 2), (128, 3), (256, 4), (64, 4), (128, 5), (256, 6), (64, 6), (256, 0)]),
])
def test_every_class_launch_variant_agrees(large, precision, shapes):
    r = np.random.default_rng(4)
    prim = np.tile(pc.freestream_prim(0.6, 2.0), (large.n, 1)) * (1.0 + 0.01 * r.standard_normal((large.n, 5)))
    s = solver.Solver(large, 0.6, 2.0, 0.2, precision=precision)
    want = None
    for block, waves in [(0, 0)] + shapes:
        print(f"[gpu] {precision}, {large.n} points, block {block}, waves {waves}", flush=True)
        s.set_tuning({"flux_interior_block": block, "flux_interior_waves": waves,
                      "flux_wall_block": block, "flux_wall_waves": waves})
        s.upload("prim", prim)
        s.run(1, 2)
        got = s.download("prim"), s.download("flux_res")
        assert np.isfinite(got[0]).all()
        if want is None:
            want = got
        assert np.array_equal(got[0], want[0]) and np.array_equal(got[1], want[1])
    s.close()


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
def test_autotuner_reports_the_joint_launch_as_the_default(precision):
    """One launch takes both classes of a small cloud, whatever the shapes:
    there is nothing to choose, and no time of a shape that never ran."""
    cl = shells(30000)
    print(f"[gpu] autotune {precision}, {cl.n} points", flush=True)
    s = solver.Solver(cl, 0.6, 2.0, 0.2, precision=precision)
    s.upload("prim", np.tile(pc.freestream_prim(0.6, 2.0), (cl.n, 1)))
    t = s.autotune(2)
    s.close()
    for part in ("flux_interior", "flux_wall"):
        assert (t[f"{part}_block"], t[f"{part}_waves"], t[f"{part}_lds"]) == (256, 0, 0)
        assert 0.0 < t[f"{part}_ms"] == t[f"{part}_default_ms"]


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
def test_autotuner_chooses_among_the_class_launches(large, precision):
    print(f"[gpu] autotune {precision}, {large.n} points", flush=True)
    s = solver.Solver(large, 0.6, 2.0, 0.2, precision=precision)
    s.upload("prim", np.tile(pc.freestream_prim(0.6, 2.0), (large.n, 1)))
    t = s.autotune(1)
    s.close()
    for part in ("flux_interior", "flux_wall"):
        assert t[f"{part}_block"] in (64, 128, 256)
        assert 1 <= t[f"{part}_waves"] <= (2 if precision == "fp64" else 6)
        assert 0.0 < t[f"{part}_ms"] <= t[f"{part}_default_ms"]


@pytest.mark.parametrize("precision,power,waves", [("fp64", 0.0, {2}), ("fp64", 2.0, {2}), ("mixed", 0.0, {2, 4, 6}),
                                                   ("mixed", 2.0, {4})])
def test_autotuner_starts_from_the_default_q_derivatives(precision, power, waves):
    """The forms with one register cap report that one, and the default's time
    is that of the shape that runs by default: the tuned and the default shape
    agree in every result, and the choice is not slower than the default."""
    cl = pc.fixture_cloud(3000, seed=6, order="morton", k=25 if power == 0.0 else 22)
    print(f"[gpu] autotune {precision}, power {power}, {cl.n} points", flush=True)
    prim = np.tile(pc.freestream_prim(0.6, 2.0), (cl.n, 1))
    s = solver.Solver(cl, 0.6, 2.0, 0.2, precision=precision, power=power)
    s.upload("prim", prim)
    s.run(1, 2)
    want = s.download("dq")
    t = s.autotune(2)
    assert t["qderiv_block"] in (64, 128, 256) and t["qderiv_waves"] in waves
    assert 0.0 < t["qderiv_ms"] <= t["qderiv_default_ms"]
    for lds in (t["qderiv_lds"], 0, 65536):
        for block in (0, t["qderiv_block"]):
            s.set_tuning({**t, "qderiv_block": block, "qderiv_lds": lds})
            s.upload("prim", prim)
            s.run(1, 2)
            assert np.array_equal(s.download("dq"), want)
    s.close()
