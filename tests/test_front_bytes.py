"""The memory bound that requests are admitted by covers the fronts that the
elimination trees lay out, for batches and for contexts' own factorizations, at
every size and for every number of unknowns a node."""
import os
import subprocess

import mafem
from mafem.patches import PatchSpec, device_bytes, front_bytes

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))),
                    "membranealefem.jl_amd", "csrc")


def test_bound_covers_the_laid_out_fronts(tmp_path):
    src = r'''
#include <cstdio>
#include "nd_plan.h"
using namespace mafem::nd;
int main() {
  for (int ndf : {4, 7, 8})
    for (int n = 1; n <= 132; ++n) {
      const Plan P = build_plan(n + 2, n + 2, ndf, choose_leaf(n + 2, n + 2, ndf, ndf == 7 ? 5 : 10));
      std::vector<int64_t> at;
      int64_t tiles = place_schur(P, at), mn = 0;
      for (const Front &F : P.fr) {
        tiles += (int64_t)F.fT * (F.FT + F.fT - 1) + (int64_t)(F.FT - F.fT) * F.fT + 2 * F.fT;
        mn += 2 * (int64_t)F.fT * (F.FT - F.fT);
      }
      const bool d = mn_saving(P, 2.0, 64) > 0.0, k = mn_saving(P, 5.0, 32) > 0.0;
      std::printf("%d %d %ld %ld %ld\n", ndf, n, (long)tiles, (long)(tiles + (d ? mn : 0)),
                  (long)(tiles + (k ? mn : 0)));
    }
}
'''
    cpp, exe = str(tmp_path / "c.cpp"), str(tmp_path / "c")
    with open(cpp, "w") as f:
        f.write(src)
    subprocess.run(["g++", "-O1", "-std=c++17", "-I", CSRC, cpp, "-o", exe], check=True)
    motion = {4: mafem.LAG, 7: mafem.EUL, 8: mafem.ALEVB}
    rows = [list(map(int, l.split())) for l in subprocess.run([exe], check=True, capture_output=True,
                                                              text=True).stdout.splitlines()]
    assert len(rows) > 200
    for ndf, n, batch, own64, own32 in rows:
        s = PatchSpec(motion[ndf], n, 1.0, 1.0, 0.4, 0)
        for precision, own, tiles in ((32, False, batch), (64, False, batch), (64, True, own64),
                                      (32, True, own32)):
            assert front_bytes(s, precision, own) >= tiles * 64 * 64 * precision // 8, (ndf, n, precision, own)
            assert device_bytes(s, precision, ordering="nd", own=own) > front_bytes(s, precision, own)
