"""The leaf size that a patch's elimination tree takes costs no accuracy.

The second Newton iteration's |K du + r| / |r| without refinement, against the
same with leaves of four nodes: over a sweep of Eulerian patches leaves of five
left at most 3.3 times as much, larger ones up to five digits more at sizes such as
the first three.  The bound is 8, which the other motions keep at every size."""
import numpy as np
import pytest

import mafem
from mafem.analysis import DeviceMesh

pytestmark = pytest.mark.gpu

DT = 1e-3


def _unrefined(motion, n1, n2):
    rng = np.random.default_rng(1)
    p = mafem.Params(motion=motion, num1el=n1, num2el=n2, length=1.0, kb=1.0, kg=-0.5, zv=1.0,
                     enr=1e-10, output=False)
    speed = 0.01 * float(rng.uniform(0.9, 1.1))
    mesh = mafem.make_mesh(p, pull_speed=speed)
    xms, cps = mafem.prepare_input(p, mesh, pull_speed=speed)
    xms[:, 2] += rng.normal(0.0, 1e-6, mesh.numnp)
    dev = DeviceMesh(mesh, p)
    try:
        dev.set_state(xms, cps)
        dev.predict(DT)
        dev.time_step(DT, DT, 1)
        dev.set_solver("direct", refine_sweeps=0, rtol=1e-3)
        dev.time_step(DT, DT, 1)
        return dev.stats()["last_relres"]
    finally:
        dev.close()


@pytest.mark.parametrize("motion,n1,n2", [("EUL", 31, 27), ("EUL", 56, 56), ("EUL", 60, 60),
                                          ("EUL", 24, 24), ("LAG", 60, 60), ("ALEVB", 26, 26)])
def test_chosen_leaf_keeps_the_accuracy(monkeypatch, motion, n1, n2):
    print(f"leaf accuracy {motion} {n1}x{n2}", flush=True)
    monkeypatch.delenv("MAFEM_ND_LEAF", raising=False)
    chosen = _unrefined(getattr(mafem, motion), n1, n2)
    monkeypatch.setenv("MAFEM_ND_LEAF", "4")
    least = _unrefined(getattr(mafem, motion), n1, n2)
    print(f"  {chosen:.1e}, with leaves of four {least:.1e}", flush=True)
    assert chosen <= 8 * least
