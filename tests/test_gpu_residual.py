"""The residual's reduction over the state update's workgroups (256 points
each), at the edges of the final workgroup's waves and threads."""

import math

import numpy as np
import pytest

from conftest import PKG

pytestmark = pytest.mark.gpu
solver = PKG.solver
pc = PKG.pointcloud


@pytest.mark.parametrize("partials,extra", [(32, 0), (64, 0), (64, 1), (1024, 0), (1024, 1)])
def test_residual_over_workgroups(partials, extra):
    n = 256 * partials + extra
    cl = pc.ellipsoid_cloud(n * 8 // 100, n * 4 // 100, n - n * 8 // 100 - n * 4 // 100, k=25, seed=9,
                            order="morton", workers=8)
    r = np.random.default_rng(partials + extra)
    prim = np.tile(pc.freestream_prim(0.6, 2.0), (n, 1)) * (1.0 + 0.01 * r.standard_normal((n, 5)))
    print(f"[gpu] residual over {n} points", flush=True)
    s = solver.Solver(cl, 0.6, 2.0, 0.2)
    s.upload("prim", prim)
    for t in (1, 2):
        rho = s.download("prim")[:, 0]
        res_new, _ = s.fpi_solver(t)
        # a term is two roundings of the densities on both sides, in the same
        # order; a sum's error is at most its longest chain of additions
        # (butterflies of 6, 6 and 4, 3 waves, 2 strides: under 24) half-ulps
        term = np.where(cl.status < 2, (s.download("prim")[:, 0] - rho) ** 2, 0.0)
        total = math.fsum(term)
        rec = s.residual()
        assert abs(rec["sum_res_sqr"] - total) <= 24 * 1.2e-16 * total
        assert abs(res_new - math.sqrt(total) / n) <= 16 * 1.2e-16 * res_new
        assert rec["max_res"] == term.max()
        assert rec["max_res_point"] == int(term.argmax()) + 1
        assert rec["res_new"] == res_new
    s.upload("prim", prim)
    hist, _ = s.run(1, 2)
    assert hist[1] == res_new
    s.close()
