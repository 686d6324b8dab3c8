"""What the fronts' tile inverses leave of a solve's residual.

Panels and solves multiply by inverses of the diagonal tiles' factors.  Formed by
substitution, or with its residual, the factorization alone leaves about what
triangular solves leave; formed as plain block products it leaves several times as
much, and FP32 factors stop preconditioning the worst conditioned tangents.
The third Newton iteration's |K du + r| / |r| without refinement, 64x64 LAG, with
triangular solves in the upper levels: 2.6e-12 in FP64, 1.1e-3 in FP32 (geometric
means); with block products 1.0e-11 and 6.7e-3.  The bounds are three times the
former.  A 64x64 EUL step with FP32 factors takes 3 iterations there and ends
unconverged after 14 with block products.
"""
import numpy as np
import pytest

import mafem
from mafem.analysis import DeviceMesh

pytestmark = pytest.mark.gpu

DT = 1e-3


def _patch(motion, n, seed):
    rng = np.random.default_rng(seed)
    p = mafem.Params(motion=motion, num1el=n, num2el=n, length=1.0, kb=1.0, kg=-0.5, zv=1.0,
                     enr=1e-10, output=False)
    speed = 0.01 * float(rng.uniform(0.9, 1.1))
    mesh = mafem.make_mesh(p, pull_speed=speed)
    xms, cps = mafem.prepare_input(p, mesh, pull_speed=speed)
    xms[:, 2] += rng.normal(0.0, 1e-6, mesh.numnp)
    dev = DeviceMesh(mesh, p)
    dev.set_state(xms, cps)
    dev.predict(DT)
    return dev


@pytest.mark.parametrize("seed", [1, 2, 3])
@pytest.mark.parametrize("precision,bound", [(64, 7.8e-12), (32, 3.3e-3)])
def test_unrefined_residual_of_the_fronts(precision, bound, seed):
    print(f"front inverses LAG 64x64 FP{precision} seed {seed}", flush=True)
    dev = _patch(mafem.LAG, 64, seed)
    try:
        dev.time_step(DT, DT, 2)
        dev.set_solver("direct", precision=precision, refine_sweeps=0, rtol=1e-3)
        dev.time_step(DT, DT, 1)
        rel = dev.stats()["last_relres"]
    finally:
        dev.close()
    print(f"  |K du + r| / |r| = {rel:.2e}", flush=True)
    assert rel < bound


@pytest.mark.parametrize("seed", [1, 2, 3])
def test_fp32_factors_precondition_the_eulerian_tangent(seed):
    print(f"front inverses EUL 64x64 FP32 factors seed {seed}", flush=True)
    dev = _patch(mafem.EUL, 64, seed)
    try:
        dev.set_solver("krylov", precision=32, refactor_iters=0, rtol=1e-13)
        rc, eps = dev.time_step(DT, DT)
    finally:
        dev.close()
    print(f"  status {rc}, eps {eps}", flush=True)
    assert rc == 0 and len(eps) <= 4
