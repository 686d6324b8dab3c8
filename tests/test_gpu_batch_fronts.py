"""Batches factor into their members' nested-dissection fronts, which a member's
own solves use too.  A member that solves for itself between two batch steps, in
the batch's precision or in the other one (its fronts are then allocated
afresh), leaves the batch's next step what it is without that solve, to the
batch's solve tolerance; sizes around a single front, one level and several,
unequal in depth, unknowns and precision."""
import numpy as np
import pytest

import mafem
from mafem.patches import Patch, PatchSpec

pytestmark = pytest.mark.gpu

DT = 1e-3


def _specs():
    return [PatchSpec(mafem.LAG, 4, 1.0, 1.0, 0.4, 3), PatchSpec(mafem.ALEVB, 7, 1.0, 1.0, 0.5, 4),
            PatchSpec(mafem.EUL, 13, 2.0, 0.5, 0.4, 5), PatchSpec(mafem.LAG, 21, 0.5, 2.0, 0.6, 6)]


def _run(precision, own):
    pts = [Patch(s) for s in _specs()]
    b = mafem.Batch([pt.dev for pt in pts], precision=precision, refactor_iters=20)
    try:
        for k in range(2):
            for pt in pts:
                pt.set_pull(pt.spec.speed_at(k))
            if k == 1 and own:
                for pt in pts[1:]:
                    x, c = pt.dev.get_state()
                    pt.dev.set_solver("krylov", precision=own, refactor_iters=0)
                    pt.dev.time_step((k + 1) * DT, DT)
                    pt.dev.set_state(x, c)
            _, _, st = b.time_step((k + 1) * DT, DT)
            assert (st == 0).all()
        assert b.stats()["hard_failures"] == 0
        return [pt.dev.get_state() for pt in pts], b.stats()["fp64_patches"]
    finally:
        b.close()
        for pt in pts:
            pt.close()


@pytest.mark.parametrize("precision,own", [(32, 32), (32, 64), (64, 32)])
def test_members_own_solves_between_steps(precision, own):
    print(f"batch in FP{precision}, members' own solves in FP{own}", flush=True)
    ref, n64 = _run(precision, 0)
    got, m64 = _run(precision, own)
    assert n64 == m64
    for (x, c), (xr, cr) in zip(got, ref):
        # Newton's last correction is below 1e-10 a free unknown, its solve at 1e-10 of that
        assert np.linalg.norm(c - cr) <= 1e-8 * np.linalg.norm(cr)
        assert np.linalg.norm(x - xr) <= 1e-8 * np.linalg.norm(xr)
