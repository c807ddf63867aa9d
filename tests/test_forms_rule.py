"""The host rule that picks the forward's and dQ's form (attn_form in
csrc/kf_host.hpp), compiled for the CPU: the forms of measured shapes on each
side of its lines."""
import subprocess
from pathlib import Path

import pytest

from kotflash_amd.build import hipcc

CSRC = Path(__file__).resolve().parents[1] / "kotflash_amd" / "csrc"
NAMES = ("4x1", "4x2", "2x2", "2x4", "1x4", "1x8")
PROGRAM = r"""
#include "kf_host.hpp"
#include <cstdio>
int main() {
  int dq, tile, causal;
  long heads, sq, sk;
  while (scanf("%d %d %ld %ld %ld %d", &dq, &tile, &heads, &sq, &sk, &causal) == 6) {
    const auto& costs = dq ? kf::kDqCosts[tile] : kf::kFwdCosts[tile];
    const int f = kf::attn_form(costs, heads, sq, sk, causal != 0);
    printf("%d %d\n", f, costs[f].per_cu);
  }
}
"""


@pytest.fixture(scope="session")
def form_of(tmp_path_factory):
    """form_of([(kernel, d, heads, sq, sk, causal), ...]) -> form names, each
    checked to be built."""
    where = tmp_path_factory.mktemp("forms")
    (where / "forms.cpp").write_text(PROGRAM)
    rocm = Path(hipcc()).resolve().parent.parent
    subprocess.run(["g++", "-O2", "-std=c++17", "-D__HIP_PLATFORM_AMD__", f"-I{CSRC}",
                    f"-isystem{rocm / 'include'}", "forms.cpp", "-o", "forms"], cwd=where, check=True)

    def run(problems):
        text = "".join(f"{int(kernel == 'dq')} {max(0, -(-d // 32) - 1)} {heads} {sq} {sk} {int(causal)}\n"
                       for kernel, d, heads, sq, sk, causal in problems)
        out = subprocess.run([str(where / "forms")], input=text, capture_output=True, text=True, check=True)
        picked = [line.split() for line in out.stdout.splitlines()]
        assert len(picked) == len(problems) and all(int(built) > 0 for _, built in picked)
        return [NAMES[int(form)] for form, _ in picked]

    return run


# kernel, d, heads, sq, sk, causal, the form that measured fastest (us: 4x1, 4x2, 2x2)
MEASURED = [
    ("fwd", 128, 128, 384, 4343, False, "4x1"),  # 132, 155, 197
    ("fwd", 96, 8, 5999, 1986, False, "4x1"),    # 47.8, 55.3, 63.4
    ("fwd", 72, 32, 1536, 2340, False, "4x1"),   # 54.2, 60.2, 69.4
    ("dq", 80, 64, 710, 5854, False, "4x1"),     # 142, 156, 169
    ("dq", 64, 8, 6272, 4461, False, "4x1"),     # 94.0, 103, 106
    ("fwd", 64, 32, 1195, 3664, False, "2x2"),   # two per CU: 70.0, 73.1, 63.3
    ("fwd", 128, 32, 981, 1752, False, "4x2"),   # 256 tiles, one 4x1 workgroup per CU: 37.9 against 40.2
    ("fwd", 112, 32, 1291, 1291, True, "4x2"),   # causal, 352 tiles: 27.6 against 29.6
]


def test_forms_of_measured_shapes(form_of):
    assert form_of([m[:6] for m in MEASURED]) == [m[6] for m in MEASURED]


def test_form_limits(form_of):
    """4x1 past two 4x1 workgroups per CU, past one (non-causal) only forms
    with two workgroups per CU, and a form that is built everywhere."""
    lengths = [1, 31, 33, 128, 129, 300, 1000, 2049, 4096, 9000, 33000]
    problems = [(kernel, d, heads, sq, sk, causal) for kernel in ("fwd", "dq") for d in (32, 64, 80, 96, 128)
                for heads in (1, 2, 7, 16, 64, 257, 513) for sq in lengths for sk in lengths
                for causal in (False, True)]
    for (kernel, d, heads, sq, _, causal), form in zip(problems, form_of(problems)):
        # Not built: never priced ahead of 4x1.
        assert (kernel, d, causal, form) != ("dq", 128, False, "4x2")
        tiles = -(-sq // 128) * heads
        if tiles > 512 or (tiles > 256 and not causal and d > 64):
            assert form == "4x1"
        elif tiles > 256 and not causal:
            assert form in ("4x1", "2x2")


def test_gpu_shapes_reach_every_form(form_of):
    """The shapes that tests/test_gpu_forms.py runs reach every form that the
    rule gives either kernel, at every head-dim tile, causal and not."""
    from tests.test_gpu_forms import HEAD_DIMS, SHAPES

    def reach(problems):
        return {(p[0], p[1], p[5], form) for p, form in zip(problems, form_of(problems))}

    kinds = [(kernel, d, causal) for kernel in ("fwd", "dq") for d in HEAD_DIMS for causal in (False, True)]
    sizes = [int(20 * 1.3 ** i) for i in range(29)]
    every = reach([(kernel, d, heads, sq, sk, causal) for kernel, d, causal in kinds
                   for heads in (1, 2, 3, 4, 6, 8, 12, 16, 24, 32, 48, 64, 96, 128, 192, 256)
                   for sq in sizes for sk in sizes])
    run = reach([(kernel, d, b * hq, sq, sk, causal) for kernel, d, causal in kinds
                 for b, hq, _, sq, sk, c in SHAPES if c == causal])
    assert every - run == set()
