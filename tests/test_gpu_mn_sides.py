"""Solves on both sides of the sizes where patches stop keeping M = L21 W and N = Z
U12: the factors alone solve the tangent to the accuracy of the tile-local pivoting
(the bound of the other front tests), and as an FP32 preconditioner they leave
FGMRES few iterations."""
import numpy as np
import pytest

import mafem
from mafem.analysis import DeviceMesh

pytestmark = pytest.mark.gpu


def _tangent(motion, n):
    p = mafem.Params(motion=motion, num1el=n, num2el=n, length=1.0, enr=1e-10, output=False)
    mesh = mafem.make_mesh(p, pull_speed=0.5)
    xms, cps = mafem.prepare_input(p, mesh, pull_speed=0.5)
    xms[:, 2] += np.random.default_rng(5).normal(0, 1e-6, mesh.numnp)
    dev = DeviceMesh(mesh, p)
    dev.set_state(xms, cps)
    return dev, *dev.assemble(1e-3, 1e-3)


@pytest.mark.parametrize("motion,n,precision", [
    ("LAG", 7, 64), ("LAG", 48, 64), ("LAG", 49, 64), ("EUL", 34, 64), ("EUL", 35, 64), ("ALEVB", 22, 64),
    ("ALEVB", 23, 64), ("ALEVB", 30, 64), ("ALEVB", 31, 64), ("ALEVB", 66, 32), ("ALEVB", 67, 32)])
def test_solves_with_and_without_the_products(motion, n, precision):
    print(f"M and N {motion} {n}x{n} FP{precision}", flush=True)
    dev, r, K = _tangent(getattr(mafem, motion), n)
    try:
        if precision == 64:
            dev.set_solver("direct", refine_sweeps=0, rtol=1e-13)
        else:
            dev.set_solver("krylov", precision=32, rtol=1e-12)
        du, _ = dev.solve(-r)
        its = dev.stats()["gmres_iters"]
    finally:
        dev.close()
    true = np.linalg.norm(K @ du + r) / np.linalg.norm(r)
    print(f"  residual {true:.2e}, {its} iterations", flush=True)
    assert true <= (1e-9 if precision == 64 else 1e-11)
    assert precision == 64 or its <= 60


def test_mode_change_keeps_the_solution():
    """A context whose solver changes (the other form of storage) solves the same."""
    dev, r, K = _tangent(mafem.ALEVB, 26)
    try:
        for mode, precision in (("direct", 64), ("krylov", 64), ("krylov", 32), ("direct", 64)):
            dev.set_solver(mode, precision=precision, rtol=1e-12)
            du, _ = dev.solve(-r)
            assert np.linalg.norm(K @ du + r) <= 1e-11 * np.linalg.norm(r)
    finally:
        dev.close()
