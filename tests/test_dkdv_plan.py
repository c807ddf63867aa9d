"""The host plan of the dK/dV launch (csrc/dkdv_plan.hpp), compiled for the
CPU: every plan hands each unit to exactly one share, within the workgroups and
partial slots the launch has, and measured shapes get the share count that ran
fastest."""
import itertools
import subprocess
from pathlib import Path

import pytest

from kotflash_amd.build import hipcc

CSRC = Path(__file__).resolve().parents[1] / "kotflash_amd" / "csrc"
PROGRAM = r"""
#include "dkdv_plan.hpp"
#include <cstdio>
int main() {
  int ngroups, G, nqt, nkt, causal, cus, tile;
  while (scanf("%d %d %d %d %d %d %d", &ngroups, &G, &nqt, &nkt, &causal, &cus, &tile) == 7) {
    const kf::DkdvPlan& p = kf::dkdv_plan(ngroups, G, nqt, nkt, causal != 0, cus, kf::kFixupCost8[tile]);
    printf("%d %d", p.nwg, p.shared);
    for (int w = 0; w <= p.nwg; ++w) printf(" %d", p.split.start[w]);
    printf("\n");
  }
}
"""


@pytest.fixture(scope="module")
def plans(tmp_path_factory):
    where = tmp_path_factory.mktemp("plan")
    (where / "plan.cpp").write_text(PROGRAM)
    rocm = Path(hipcc()).resolve().parent.parent
    subprocess.run(["g++", "-O2", "-std=c++17", "-D__HIP_PLATFORM_AMD__", f"-I{CSRC}",
                    f"-isystem{rocm / 'include'}", "plan.cpp", "-o", "plan"], cwd=where, check=True)

    def run(problems):
        text = "".join(" ".join(str(int(x)) for x in p) + "\n" for p in problems)
        out = subprocess.run([str(where / "plan")], input=text, capture_output=True, text=True, check=True)
        rows = [[int(x) for x in line.split()] for line in out.stdout.splitlines()]
        assert len(rows) == len(problems)
        return [(r[0], r[1], r[2:]) for r in rows]

    return run


def _row_ends(ngroups, g, nqt, nkt, causal):
    """Unit numbers at which a tile row ends, in the launch's order."""
    units = [max(0, nqt - (2 * kt if causal else 0)) * g for kt in range(nkt)]
    seen = sum(u > 0 for u in units)
    order = [seen - 1 - pos // 2 if pos % 2 else pos // 2 for pos in range(seen)]
    return list(itertools.accumulate(units[kt] for _ in range(ngroups) for kt in order))


def test_plans_cover_every_unit_once(plans):
    problems = [(ngroups, g, nqt, nkt, causal, cus, tile)
                for ngroups, g in ((1, 1), (1, 8), (2, 4), (7, 1), (24, 2), (48, 1), (200, 1))
                for nqt in (1, 2, 3, 9, 16, 33, 64) for nkt in (1, 2, 5, 8, 17, 40)
                for causal in (0, 1) for cus, tile in ((256, 1), (256, 3), (304, 2), (6, 1))]
    for problem, (nwg, shared, start) in zip(problems, plans(problems)):
        ends = _row_ends(*problem[:5])
        assert 1 <= nwg <= problem[5] and (nwg % 8 == 0 or nwg == problem[5]), problem
        assert start[0] == 0 and start[-1] == ends[-1], problem
        assert all(a <= b for a, b in zip(start, start[1:])), problem
        # Rows that a boundary lies inside: what the fixup has to sum.
        inside = set(start) - set(ends) - {0}
        cut = sum(any(a < u < b for u in inside) for a, b in zip([0] + ends, ends)) if inside else 0
        assert cut == shared, problem


# B, Hq, Hkv, Sq, Sk, D, causal, shares (us for dK/dV and fixup: 256 shares, 8 units a share, 4)
MEASURED = [
    (3, 16, 8, 533, 533, 128, True, 256),    # 35.4, 40.5, 35.9: rows in 1.3 shares of 8 units
    (1, 16, 4, 433, 433, 64, True, 64),      # 4 units 26% ahead of 8
    (1, 8, 1, 1393, 467, 72, False, 88),     # 98.9, 34.0, 39.5: rows in 22 shares
    (1, 4, 1, 1739, 1739, 80, True, 112),    # 64.3, 34.5, 36.9
    (4, 4, 4, 872, 872, 112, True, 112),     # 34.0, 28.0, 35.6: whole rows
]


def test_shares_of_measured_shapes(plans):
    problems = [(b * hkv, hq // hkv, -(-sq // 64), -(-sk // 128), causal, 256, -(-d // 32) - 1)
                for b, hq, hkv, sq, sk, d, causal, _ in MEASURED]
    got = plans(problems)
    assert [nwg for nwg, _, _ in got] == [m[-1] for m in MEASURED]
    assert got[-1][1] == 0 and all(shared > 0 for _, shared, _ in got[:-1])
