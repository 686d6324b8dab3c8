"""Host logic of the nested-dissection front plan (csrc/nd_plan.h).

tests/nd_check.cpp builds the plan and runs a dense CPU emulation of the
multifrontal factorization and solve the device performs over it (same front
layout, entry ownership, child gather order and tile-local pivoting) on a
random matrix with the tangent's node-block pattern, prescribed identity rows
and a zero diagonal entry per node; its solution must match a dense
partial-pivoting LU solve.  The plan's structural invariants (every coupled
entry in exactly one front, children at lower levels, separators with two
children) are checked there too.
"""
import os
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(os.path.dirname(HERE), "membranealefem.jl_amd", "csrc")


@pytest.fixture(scope="module")
def nd_check(tmp_path_factory):
    exe = str(tmp_path_factory.mktemp("nd") / "nd_check")
    subprocess.run(["g++", "-O2", "-std=c++17", "-I", CSRC, os.path.join(HERE, "nd_check.cpp"),
                    "-o", exe], check=True)
    return exe


@pytest.mark.parametrize("n1,n2,ndf,leaf,seed", [
    (10, 10, 8, 4, 1),   # 8x8 elements, ALEVB-sized node blocks
    (12, 9, 4, 4, 2),    # rectangular, LAG
    (9, 14, 7, 4, 3),    # EUL
    (10, 10, 8, 6, 4),   # larger leaves
    (5, 5, 8, 4, 5),     # one separator level
    (3, 4, 8, 4, 6),     # a single leaf front
    (18, 18, 4, 4, 7),   # five levels
])
def test_multifrontal_emulation_solves(nd_check, n1, n2, ndf, leaf, seed):
    out = subprocess.run([nd_check, str(n1), str(n2), str(ndf), str(leaf), str(seed)],
                         capture_output=True, text=True)
    assert out.returncode == 0, out.stdout + out.stderr
    rel_nd, rel_dense, diff, fronts, levels, steps = out.stdout.split()
    assert float(rel_nd) <= 1e-10
    assert float(diff) <= 1e-9
    assert int(fronts) >= 1 and int(levels) >= 1 and int(steps) >= 1


def test_plan_chain_lengths(nd_check):
    """The dependent tile steps of the 64x64 ALEVB plan (66 x 66 nodes, 8
    unknowns): the level maxima of the fully-summed tile rows, 2, 1, 2, 2, 4,
    4, 8, 8, 17 from the leaves to the root."""
    src = r'''
#include <cstdio>
#include "nd_plan.h"
int main() {
  auto P = mafem::nd::build_plan(66, 66, 8);
  for (auto &l : P.by_level) printf("%d ", P.fr[l.front()].fT);
  printf("| %lld %zu\n", (long long)P.critical_steps(), P.fr.size());
}
'''
    d = os.path.dirname(nd_check)
    with open(os.path.join(d, "steps.cpp"), "w") as f:
        f.write(src)
    exe = os.path.join(d, "steps")
    subprocess.run(["g++", "-O2", "-std=c++17", "-I", CSRC, os.path.join(d, "steps.cpp"), "-o",
                    exe], check=True)
    out = subprocess.run([exe], capture_output=True, text=True, check=True).stdout
    levels, rest = out.split("|")
    assert [int(x) for x in levels.split()] == [2, 1, 2, 2, 4, 4, 8, 8, 17]
    steps, fronts = rest.split()
    assert int(steps) == 48 and int(fronts) == 511


def test_leaf_choice_prices_the_built_plan(tmp_path):
    """plan_cost counts what build_plan lays out: levels, dependent steps and tile
    products of every leaf size, on square, ragged, strip and single-front grids;
    choose_leaf takes the least."""
    src = r'''
#include <cmath>
#include <cstdio>
#include "nd_plan.h"
using namespace mafem::nd;
int main() {
  const int g[][3] = {{3, 3, 4}, {8, 8, 4}, {10, 10, 8}, {19, 15, 7}, {42, 9, 3}, {5, 60, 8}, {35, 29, 7}};
  for (auto &x : g) {
    double least = 1e300;
    for (int leaf = 4; leaf <= 10; ++leaf) {
      const Plan P = build_plan(x[0], x[1], x[2], leaf);
      double pr = 0.0;
      for (const Front &F : P.fr)
        for (int K = 0; K < F.fT; ++K) pr += (double)(F.FT - K - 1) * (F.FT - K);
      const double c = 33.0 * (P.critical_steps() + P.levels) + pr * 2 * 64 * 64 * 64 / 45e6;
      if (std::fabs(c - plan_cost(x[0], x[1], x[2], leaf)) > 1e-9 * c) return 1;
      least = std::fmin(least, c);
    }
    if (plan_cost(x[0], x[1], x[2], choose_leaf(x[0], x[1], x[2])) > least * (1 + 1e-12)) return 2;
  }
}
'''
    cpp, exe = str(tmp_path / "c.cpp"), str(tmp_path / "c")
    with open(cpp, "w") as f:
        f.write(src)
    subprocess.run(["g++", "-O1", "-std=c++17", "-I", CSRC, cpp, "-o", exe], check=True)
    assert subprocess.run([exe]).returncode == 0


def test_schur_complements_that_coexist_do_not_overlap(tmp_path):
    """place_schur: complements that are there on a common level (from their
    front's to its parent's) lie apart, inside the pool, and the pool is smaller
    than all of them once a tree has a few levels."""
    src = r'''
#include <cstdio>
#include "nd_plan.h"
using namespace mafem::nd;
int main() {
  const int g[][4] = {{3, 3, 4, 4}, {6, 5, 8, 4}, {8, 8, 4, 4}, {19, 15, 7, 4}, {42, 9, 3, 5}, {5, 60, 8, 4}, {35, 29, 7, 6}};
  for (auto &x : g) {
    const Plan P = build_plan(x[0], x[1], x[2], x[3]);
    std::vector<int64_t> at;
    const int64_t total = place_schur(P, at);
    int64_t sum = 0;
    auto size = [&](size_t t) { return (int64_t)(P.fr[t].FT - P.fr[t].fT) * (P.fr[t].FT - P.fr[t].fT); };
    for (size_t t = 0; t < P.fr.size(); ++t) {
      if (P.fr[t].parent < 0) continue;
      sum += size(t);
      if (at[t] < 0 || at[t] + size(t) > total) return 1;
      for (size_t u = 0; u < t; ++u) {
        if (P.fr[u].parent < 0) continue;
        const bool meet = P.fr[t].level <= P.fr[P.fr[u].parent].level && P.fr[u].level <= P.fr[P.fr[t].parent].level;
        if (meet && at[t] < at[u] + size(u) && at[u] < at[t] + size(t)) return 2;
      }
    }
    if (P.levels > 4 && total >= sum) return 3;
  }
}
'''
    cpp, exe = str(tmp_path / "c.cpp"), str(tmp_path / "c")
    with open(cpp, "w") as f:
        f.write(src)
    subprocess.run(["g++", "-O1", "-std=c++17", "-I", CSRC, cpp, "-o", exe], check=True)
    assert subprocess.run([exe]).returncode == 0
