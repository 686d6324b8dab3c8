"""A patch's trajectory in a batch is the same bits alone and among copies of itself
that fill the levels of its elimination tree: a level of 512 tile rows and more is
solved with one block per tile row instead of four (two 64x64 EUL or eight 40x40
LAG patches reach that on their leaves, one does not)."""
import numpy as np
import pytest

import mafem
from mafem.patches import Patch, PatchSpec

pytestmark = pytest.mark.gpu

DT = 1e-3


def _run(spec, count, precision):
    pts = [Patch(spec) for _ in range(count)]
    b = mafem.Batch([pt.dev for pt in pts], precision=precision)
    try:
        for pt in pts:
            pt.set_pull(pt.spec.speed_at(0))
        iters, _, st = b.time_step(DT, DT)
        assert (st == 0).all()
        return iters, [pt.dev.get_state() for pt in pts]
    finally:
        b.close()
        for pt in pts:
            pt.close()


@pytest.mark.parametrize("precision", [32, 64])
@pytest.mark.parametrize("motion,n,count", [("EUL", 64, 2), ("LAG", 40, 8), ("LAG", 40, 7)])
def test_wide_levels_keep_a_patch_bits(motion, n, count, precision):
    print(f"{count} x {motion} {n}x{n} FP{precision}", flush=True)
    spec = PatchSpec(getattr(mafem, motion), n, 1.0, 1.0, 0.4, 3)
    it1, alone = _run(spec, 1, precision)
    its, mix = _run(spec, count, precision)
    for k, (x, c) in enumerate(mix):
        assert its[k] == it1[0]
        assert np.array_equal(x, alone[0][0]) and np.array_equal(c, alone[0][1])
