"""Residual and tangent where the area kernel's launch changes its split: one
round of nine, three or two lanes per column, one lane, and full rounds of 256
blocks with the rest split (1820 LAG or 910 ALEVB elements a round), against the
oracle.  Every entry is a sum of at most 4 x 9 Gauss-point terms in 64 bits, so the
matrices agree to 1e-12 in norm, as at the sizes the other parity tests use."""
import numpy as np
import pytest

import mafem
from oracle import fem, mesh as om

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("motion,n1,n2", [
    ("LAG", 14, 14), ("LAG", 15, 14), ("LAG", 25, 24), ("LAG", 26, 24), ("LAG", 30, 30), ("LAG", 31, 30),
    ("LAG", 43, 43), ("EUL", 13, 13), ("ALEVB", 10, 10), ("ALEVB", 18, 17), ("ALEVB", 31, 30),
    ("STATIC", 28, 27),
])
def test_residual_and_tangent_at_the_splits(motion, n1, n2):
    print(f"area split {motion} {n1}x{n2}", flush=True)
    mo = getattr(mafem, motion)
    scen = "F_CAVI" if motion == "STATIC" else "F_PULL"
    p = mafem.Params(motion=mo, scenario=getattr(mafem, scen), num1el=n1, num2el=n2, length=1.0,
                     enr=1e-10, output=False)
    po = om.Params(motion=getattr(om, motion), scenario=getattr(om, scen), num1el=n1, num2el=n2,
                   length=1.0, enr=1e-10)
    kw = {} if motion == "STATIC" else {"pull_speed": 0.5}
    mesh = mafem.make_mesh(p, **kw)
    xms, cps = mafem.prepare_input(p, mesh, **kw)
    rng = np.random.default_rng(3)
    if motion != "STATIC":
        xms[:, 2] += rng.normal(0, 1e-3, mesh.numnp)
    cps += np.where(mesh.ID.T != 0, rng.normal(0, 1e-2, cps.shape), 0.0)
    r, K = mafem.calc_r_K(mesh, xms, cps, 1e-3, 1e-3, p)
    o, _, _ = fem.build(po, **kw)
    r_o, K_o = fem.calc_r_K(o, xms, cps, 1e-3, 1e-3)
    d = (K - K_o)
    assert np.linalg.norm(r - r_o) <= 1e-12 * np.linalg.norm(r_o)
    assert np.linalg.norm(d.data) <= 1e-12 * np.linalg.norm(K_o.data)
