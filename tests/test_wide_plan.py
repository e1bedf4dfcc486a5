"""How a prompt chunk's projections share their work (ops::Linear::wideSplit). No GPU."""
import pathlib
import shutil
import subprocess

import pytest

import splash_amd  # noqa: F401  (the library the program links)

ROOT = pathlib.Path(__file__).resolve().parent.parent
HIP = pathlib.Path("/opt/rocm/include")

PROGRAM = r"""
#include "ops/Linear.hpp"
#include <cstdio>
int main() {
  unsigned units, groups, blocks, rows, splittable;
  while (std::scanf("%u %u %u %u %u", &units, &groups, &blocks, &rows, &splittable) == 5) {
    splash::ops::KernelCalibration calibration{units};
    const auto plan = splash::ops::Linear(calibration).wideSplit(groups, blocks, rows, splittable);
    std::printf("%u %u %u %u %u\n", plan.rowGroups, plan.tiles, plan.splits, plan.tailGroups, plan.tailRowGroups);
  }
}
"""


@pytest.fixture(scope="module")
def program(tmp_path_factory):
    if not shutil.which("g++") or not (HIP / "hip" / "hip_runtime.h").exists():
        pytest.skip("no host compiler or no HIP headers")
    folder = tmp_path_factory.mktemp("plan")
    (folder / "plan.cpp").write_text(PROGRAM)
    library = ROOT / "splash_amd" / "lib"
    subprocess.run(["g++", "-std=c++20", "-w", "-fno-access-control", "-D__HIP_PLATFORM_AMD__", f"-I{HIP}", f"-I{ROOT / 'include'}",
                    f"-I{ROOT / 'splash_amd' / 'csrc'}", str(folder / "plan.cpp"), "-o", str(folder / "plan"), f"-L{library}",
                    "-lsplash_hip", f"-Wl,-rpath,{library}", "-Wl,--unresolved-symbols=ignore-in-shared-libs"], check=True, timeout=240)
    return folder / "plan"


def parts_of_whole_rounds(units, groups, blocks, rows, splittable):
    """The parts of K that workgroups of one height leave: the fastest plan of those without a tail."""
    live, slots, best = -(-rows // 16), 2 * units, None
    for tallest in (8, 7, 6, 4):
        items = -(-live // tallest) * groups
        for s in range(1, 9):
            if s > 1 and (not splittable or s * 2 > blocks):
                break
            cost = -(-items * s // slots) / s * (2.2 + tallest) * blocks * 0.55
            cost += 5.0 + s * rows * groups * 128 * 8 / 4.5e6 if s > 1 else 0.0
            if best is None or cost < best[0]:
                best = (cost, s)
    return best[1]


def test_a_tail_never_takes_the_place_of_parts_of_k(program):
    """Which parts a row's sum is added in decides its rounding: columns in shorter workgroups leave it as it is."""
    cases = [(units, groups, blocks, rows, splittable) for units in (64, 256) for groups in (3, 16, 40, 80, 81, 97, 200, 400) for blocks in (4, 8, 20, 32, 100)
             for rows in (*range(16, 2049, 112), 777, 1536) for splittable in (0, 1)]
    out = subprocess.run([str(program)], input="\n".join(" ".join(map(str, c)) for c in cases), capture_output=True, text=True, timeout=60, check=True)
    plans = [tuple(map(int, line.split())) for line in out.stdout.splitlines()]
    assert len(plans) == len(cases)
    tails = split = 0
    for case, (row_groups, tiles, splits, tail, tail_row_groups) in zip(cases, plans):
        assert splits == parts_of_whole_rounds(*case), case
        live = -(-case[3] // 16)
        assert row_groups * tiles >= live and (not tail or (splits == 1 and tiles > 4 and tail <= case[1] and tail_row_groups == -(-live // 4))), case
        tails += tail > 0
        split += splits > 1
    assert tails > 50 and split > 50
