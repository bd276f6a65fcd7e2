"""The fused FP64 flux kernel over the range of split-flux arguments.

erf and exp of one argument come from a table up to 6 and from a series
beyond (erf_exp.h): states from rest to Mach 8, where S = u*sqrt(beta) runs
from 0 to about 7, against the oracle.  The tolerance is that of the parity
tests' flux residual, 1e-11 of each component's largest magnitude: the
residual's terms cancel to a few hundredths of their size, and each carries
some ten roundings.
"""

import sys

import numpy as np
import pytest

from conftest import PKG, ROOT

pytestmark = pytest.mark.gpu
solver = PKG.solver
pc = PKG.pointcloud
sys.path.insert(0, ROOT + "/oracle")


@pytest.mark.parametrize("mach", [0.0, 0.6, 3.0, 6.5, 8.0])
def test_flux_residual_from_rest_to_mach_8(mach):
    import orc

    cl = pc.fixture_cloud(700, seed=6, order="morton")
    r = np.random.default_rng(2)
    prim = np.tile(pc.freestream_prim(mach, 2.0), (cl.n, 1)) * (1.0 + 0.01 * r.standard_normal((cl.n, 5)))
    print(f"[gpu] Mach {mach}, {cl.n} points", flush=True)
    o = orc.Oracle(cl, mach, 2.0, 0.2, prim=prim.copy())
    o.run(1, 1, "explicit")
    want = np.asarray(o.flux_res).reshape(cl.n, 5)
    s = solver.Solver(cl, mach, 2.0, 0.2)
    s.upload("prim", prim)
    s.run(1, 1)
    got = s.download("flux_res")
    s.close()
    assert np.isfinite(want).all()
    assert np.max(np.abs(got - want) / np.max(np.abs(want), axis=0)) < 1e-11
