"""The band's diagonal-tile inverses: what the folded tiles leave of the residual.

Folds multiply by Y = U^-1 from the right side of U, so Y has to satisfy Y U = I.
The solve of the third Newton iteration, without refinement, leaves in a plain
NumPy band LU with 64 x 64 tiles |K du + r| / |r| of 1.5e-14, 7.7e-15 and 3.3e-14 on
the three patches below with the inverses formed by substitution; with their
diagonal blocks multiplied instead it is 6.5e-14, 1.5e-13 and 5.5e-13.  The bound is
three times the former.
"""
import numpy as np
import pytest

import mafem
from mafem.analysis import DeviceMesh

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("motion,n1,n2,bound", [(mafem.ALEVB, 17, 13, 4.6e-14), (mafem.ALEV, 17, 13, 2.3e-14),
                                                (mafem.LAG, 20, 17, 1e-13)])
def test_unrefined_residual_of_the_band_solve(motion, n1, n2, bound):
    print(f"tile inverses {motion.name} {n1}x{n2}", flush=True)
    rng = np.random.default_rng(1)
    p = mafem.Params(motion=motion, num1el=n1, num2el=n2, length=1.0, kb=1.0, kg=-0.5, zv=1.0,
                     enr=1e-10, output=False)
    speed = 0.01 * float(rng.uniform(0.9, 1.1))
    mesh = mafem.make_mesh(p, pull_speed=speed)
    xms, cps = mafem.prepare_input(p, mesh, pull_speed=speed)
    xms[:, 2] += rng.normal(0.0, 1e-6, mesh.numnp)
    dev = DeviceMesh(mesh, p)
    dev.set_ordering("band")
    dev.set_solver("direct", refine_sweeps=0)
    dev.set_state(xms, cps)
    dev.predict(1e-3)
    rc, eps = dev.time_step(1e-3, 1e-3)
    assert rc == 0 and len(eps) == 3
    s = dev.stats()
    rel = s["last_relres"] if isinstance(s, dict) else s.last_relres
    print(f"|K du + r| / |r| = {rel:.2e}", flush=True)
    assert rel < bound
