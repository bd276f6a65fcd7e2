"""Lanes per point of the fused flux kernel.

flux_small (kernels_flux_fused.hip) picks the lanes that share a point, and
whether the two classes share a launch, from the number of points bound.  A
point's sums must not depend on that: a cloud's state is compared, bit for
bit, between a run by itself (32 lanes per point) and a run beside another
cloud large enough for each of the other rules.  The cloud by itself is held
to the oracle by the fixtures' tests.
"""

import numpy as np
import pytest

from conftest import PKG

pytestmark = pytest.mark.gpu
solver = PKG.solver
pc = PKG.pointcloud


def shells(n, k=25):
    return pc.ellipsoid_cloud(n * 8 // 100, n * 4 // 100, n - n * 12 // 100, k=k, seed=9, order="morton", workers=8)


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
@pytest.mark.parametrize("power,fillers", [
    (0.0, [4000]),                 # 32 lanes (general) and 16 (interior)
    (0.0, [4000] * 5),             # 16 and 16
    (0.0, [40000]),                # 16 and 4
    (0.0, [220000]),               # 4 and 4
    (0.0, [560000]),               # a launch per class
    (2.0, [4000]),                 # 16 and 16, weighted least squares
    (2.0, [40000]),                # 16 and 4
    (2.0, [220000]),               # a launch per class
])
def test_sums_do_not_depend_on_the_lanes(precision, power, fillers):
    k = 25 if power == 0.0 else 22
    cl = pc.fixture_cloud(500, seed=3, order="morton", k=k)
    others = [shells(n, k) if n > 20000 else pc.fixture_cloud(n * 62 // 100, seed=4 + i, order="blocks", k=k)
              for i, n in enumerate(fillers)]
    clouds = [cl] + others
    r = np.random.default_rng(8)
    prim = [np.tile(pc.freestream_prim(0.6, 2.0), (c.n, 1)) * (1.0 + 0.01 * r.standard_normal((c.n, 5)))
            for c in clouds]
    print(f"[gpu] {precision}, power {power}, clouds of {[c.n for c in clouds]}", flush=True)
    bs = solver.BatchSolver(clouds, [0.6] * len(clouds), [2.0] * len(clouds), 0.2, precision=precision, power=power)
    bs.upload("prim", np.concatenate(prim))
    bs.run(1, 3)
    got = bs.split(bs.download("prim"))[0], bs.split(bs.download("flux_res"))[0]
    bs.close()
    s = solver.Solver(cl, 0.6, 2.0, 0.2, precision=precision, power=power)
    s.upload("prim", prim[0])
    s.run(1, 3)
    assert np.isfinite(got[0]).all()
    assert np.array_equal(got[0], s.download("prim"))
    assert np.array_equal(got[1], s.download("flux_res"))
    s.close()


def test_autotuned_class_launches_fit_the_lds():
    """Above the joint launch's sizes the autotuner reserves up to a CU's whole
    LDS for a workgroup of the class kernels; the FP64 ones hold a table there."""
    cl = shells(560000)
    prim = np.tile(pc.freestream_prim(0.6, 2.0), (cl.n, 1))
    print(f"[gpu] autotune, {cl.n} points", flush=True)
    s = solver.Solver(cl, 0.6, 2.0, 0.2)
    s.upload("prim", prim)
    s.run(1, 2)
    want = s.download("prim")
    t = s.autotune(1)
    for lds in (t["flux_interior_lds"], 163840):
        s.set_tuning({**t, "flux_interior_lds": lds, "flux_wall_lds": lds})
        s.upload("prim", prim)
        s.run(1, 2)
        assert np.array_equal(s.download("prim"), want)
    s.close()
