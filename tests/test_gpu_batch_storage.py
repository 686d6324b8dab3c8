"""A member of a batch that solves for itself between two batch steps leaves the
batch's factorizations alone: its own factors, in either precision, lie in storage of
their own.  The batch's next step takes as many factorizations and gives the same
bits as without those solves."""
import numpy as np
import pytest

import mafem
from mafem.patches import Patch, PatchSpec

pytestmark = pytest.mark.gpu

DT = 1e-3


def _run(precision, own):
    specs = [PatchSpec(mafem.LAG, 5, 1.0, 1.0, 0.4, 3), PatchSpec(mafem.ALEVB, 9, 1.0, 1.0, 0.5, 4),
             PatchSpec(mafem.EUL, 17, 2.0, 0.5, 0.4, 5)]
    pts = [Patch(s) for s in specs]
    b = mafem.Batch([pt.dev for pt in pts], precision=precision, refactor_iters=20)
    factors = []
    try:
        for k in range(3):
            for pt in pts:
                pt.set_pull(pt.spec.speed_at(k))
            if k and own:
                for pt in pts[:2]:
                    x, c = pt.dev.get_state()
                    pt.dev.set_solver(own[0], precision=own[1])
                    pt.dev.time_step((k + 1) * DT, DT)
                    pt.dev.set_state(x, c)
            _, _, st = b.time_step((k + 1) * DT, DT)
            assert (st == 0).all()
            factors.append(b.stats()["patch_factors"])
        return factors, [pt.dev.get_state() for pt in pts]
    finally:
        b.close()
        for pt in pts:
            pt.close()


@pytest.mark.parametrize("precision", [32, 64])
@pytest.mark.parametrize("own", [("direct", 64), ("krylov", 32), ("krylov", 64)])
def test_own_solves_leave_the_batch_factors_alone(precision, own):
    print(f"batch in FP{precision}, members' own solves {own}", flush=True)
    ref, states = _run(precision, None)
    got, mixed = _run(precision, own)
    print(f"  factorizations {ref} and {got}", flush=True)
    assert got == ref
    for (x, c), (xr, cr) in zip(mixed, states):
        assert np.array_equal(x, xr) and np.array_equal(c, cr)
