"""Batch members whose state is undefined or overflows: their step is reported as
not converged, and their neighbours take theirs as they do without them, bit for
bit (every batched kernel computes a patch from that patch's data alone)."""
import numpy as np
import pytest

import mafem
from mafem.patches import Patch, PatchSpec

pytestmark = pytest.mark.gpu

DT = 1e-3


def _step(spoil, alone, graphs):
    """One batch step of good, spoiled, good; `alone`: of the good ones only."""
    specs = [PatchSpec(mafem.LAG, 6, 1.0, 1.0, 0.4, 3), PatchSpec(mafem.ALEVB, 8, 1.0, 1.0, 0.4, 4),
             PatchSpec(mafem.EUL, 9, 2.0, 0.5, 0.4, 5)]
    pts = [Patch(s) for k, s in enumerate(specs) if k != 1 or not alone]
    b = mafem.Batch([pt.dev for pt in pts], precision=32, use_graphs=graphs)
    try:
        for pt in pts:
            pt.set_pull(pt.spec.speed_at(0))
        if not alone:
            x, c = pts[1].dev.get_state()
            spoil(pts[1].mesh, x, c)
            pts[1].dev.set_state(x, c)
        iters, eps, st = b.time_step(DT, DT)
        return list(st), eps, [pt.dev.get_state() for pt in pts]
    finally:
        b.close()
        for pt in pts:
            pt.close()


def _nan_position(mesh, x, c):
    x[x.shape[0] // 2, 2] = np.nan


def _nan_everywhere(mesh, x, c):
    x[:] = np.nan


def _folded(mesh, x, c):  # every element of area zero: 1 / J
    x[:, 1] = 0.0


def _overflow(mesh, x, c):  # |r|^2 beyond the range of 64 bits
    free = np.asarray(mesh.ID).T != 0
    c[free] = 1e200


def _far(mesh, x, c):  # finite norms, FP32 factors out of range, then a diverging iteration
    free = np.asarray(mesh.ID).T != 0
    c[free] = 1e100


def _infinite(mesh, x, c):
    free = np.argwhere(np.asarray(mesh.ID).T != 0)
    node, dof = free[len(free) // 2]
    c[node, dof] = np.inf


@pytest.mark.parametrize("graphs", [True, False])
@pytest.mark.parametrize("spoil", [_nan_position, _nan_everywhere, _folded, _overflow, _far, _infinite])
def test_undefined_member_fails_and_its_neighbours_do_not(spoil, graphs):
    print(f"batch member {spoil.__name__} graphs={graphs}", flush=True)
    _, _, good = _step(spoil, True, graphs)
    st, eps, states = _step(spoil, False, graphs)
    print("  status", st, "eps", eps[1][:3], flush=True)
    assert st[0] == 0 and st[1] == 1 and st[2] == 0
    for (x, c), (xa, ca) in zip((states[0], states[2]), good):
        assert np.array_equal(x, xa) and np.array_equal(c, ca)
