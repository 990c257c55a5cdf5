"""bench.py's roofline on a step of two launches (RK3's last two stages
together): bytes a cell and the words of the line; and the sources that date its
profiles: every header that the stage launchers take kernels from."""
import os
import re

import bench

CSRC = os.path.join(os.path.dirname(os.path.abspath(bench.__file__)), "alsvinn_amd", "csrc")


def test_bytes_of_two_launches():
    # stage 1: U0 read, L0 and the copy of U0 written; then L0 and the copy
    # read, the state written
    assert bench.stage_bytes_per_cell(4, 2) == [96, 96]
    assert bench.stage_bytes_per_cell(4, 3) == bench.stage_bytes_per_cell(4) == [64, 96, 96]
    assert "2 launches" in bench.step_description(2) and "3 fused stage launches" in bench.step_description(3)


def test_every_stage_kernel_dates_the_profiles():
    found, todo = set(), ["avh_stage_inst.hpp"]
    while todo:
        name = todo.pop()
        if name in found:
            continue
        found.add(name)
        text = open(os.path.join(CSRC, name)).read()
        todo += re.findall(r'#include "(avh_\w+\.hpp)"', text)
    # whole steps of small 1D grids: no workload of bench.py runs them
    assert found - {"avh_line.hpp"} <= set(bench.KERNEL_SOURCES)
