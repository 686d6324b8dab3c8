"""Which patches keep M = L21 W and N = Z U12 of their fronts: mn_saving's sign agrees
with the time steps measured without and with them (ms, in its comment), and it
falls with the patch's size while the number of levels stays the same."""
import os
import subprocess

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))),
                    "membranealefem.jl_amd", "csrc")


def test_saving_agrees_with_the_measured_steps(tmp_path):
    src = r'''
#include "nd_plan.h"
using namespace mafem::nd;
double at(int n1, int n2, int ndf, double solves, int prec) {
  return mn_saving(build_plan(n1 + 2, n2 + 2, ndf, choose_leaf(n1 + 2, n2 + 2, ndf, ndf == 7 ? 5 : 10)),
                   solves, prec);
}
int main() {
  const int yes[][3] = {{24, 24, 4}, {40, 40, 4}, {48, 48, 4}, {32, 32, 7}, {8, 8, 4}, {48, 48, 3}};
  const int no[][3] = {{56, 56, 4}, {40, 40, 7}, {24, 24, 8}, {48, 48, 8}, {96, 80, 4}, {64, 64, 8}};
  for (auto &x : yes)
    if (at(x[0], x[1], x[2], 2.0, 64) <= 0.0) return 1;
  for (auto &x : no)
    if (at(x[0], x[1], x[2], 2.0, 64) > 0.0) return 2;
  if (at(32, 32, 8, 5.0, 32) <= 0.0 || at(48, 48, 4, 5.0, 32) <= 0.0) return 3;
  // one front has no boundary and no level below it: nothing to save
  const Plan one = build_plan(4, 4, 4, 4);
  if (one.fr.size() != 1 || mn_saving(one, 5.0, 32) > 0.0) return 4;
  for (int n = 64; n < 128; n += 8)  // leaves of four: nine levels throughout
    if (mn_saving(build_plan(n + 8, n + 8, 8, 4), 2.0, 64) > mn_saving(build_plan(n, n, 8, 4), 2.0, 64)) return 5;
}
'''
    cpp, exe = str(tmp_path / "c.cpp"), str(tmp_path / "c")
    with open(cpp, "w") as f:
        f.write(src)
    subprocess.run(["g++", "-O1", "-std=c++17", "-I", CSRC, cpp, "-o", exe], check=True)
    assert subprocess.run([exe]).returncode == 0
