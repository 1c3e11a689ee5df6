"""CPU: the walk's short cuts give the plain tests' answers. The device
headers, compiled for one lane (`tests/cpu/walk_bounds.cpp`), settle boxes
from their centres and half extents, cut polygons and hulls in the LDS layout,
and are compared with the eight-corner tests, `in_bound`, the exact projected
extent and the general clips: the same answer for every box, the same bits for
every draw. Boxes and triangles are made to touch what decides them (a window,
near, far or horizon plane, the bounding sphere, the prefilter's threshold)."""
import os
import re
import subprocess
from pathlib import Path

import pytest

ROOT = Path(__file__).resolve().parent.parent
ROCM = Path(os.environ.get("ROCM_PATH", "/opt/rocm"))


@pytest.fixture(scope="module")
def walk_bounds(tmp_path_factory):
    exe = tmp_path_factory.mktemp("walk_bounds") / "walk_bounds"
    # (warnings off: device attributes mean nothing to a host compiler)
    subprocess.run(["g++", "-O2", "-std=c++17", "-ffp-contract=off", "-w", "-D__HIP_PLATFORM_AMD__",
                    f"-I{ROCM / 'include'}", f"-I{ROOT / 'continuum_amd' / 'csrc'}",
                    str(ROOT / "tests" / "cpu" / "walk_bounds.cpp"), "-o", str(exe)], check=True)

    def run(mode, count, seed):
        out = subprocess.run([str(exe), mode, str(count), str(seed)], capture_output=True, text=True, check=True).stdout
        cases, wrong, settled = map(int, re.search(r"cases (\d+) wrong (\d+) settled (\d+)", out).groups())
        assert wrong == 0, out
        return cases, settled
    return run


@pytest.mark.parametrize("seed", [1, 2])
@pytest.mark.parametrize("mode,count", [("light", 200000), ("object", 100000), ("apex", 200000), ("any", 100000)])
def test_boxes_are_settled_as_by_their_corners(walk_bounds, mode, count, seed):
    """Light cones, the same in a turned and scaled object's space, and boxes
    by an apex up to 10^6 m from the origin, where the bounding sphere's centre
    is rounded by more than the box is wide; cones of any window and far plane
    over boxes that may be empty, unbounded or not a number."""
    cases, settled = walk_bounds(mode, count, seed)
    assert settled > cases / 4  # (two checks a box: the short cut did settle boxes)


def test_sky_boxes_are_settled_by_the_horizon_of_any_normal(walk_bounds):
    """Normals of length 1 and of 10^-3 to 10^6, boxes with corners in the horizon's plane."""
    cases, settled = walk_bounds("sky", 200000, 1)
    assert settled > cases / 4


@pytest.mark.parametrize("mode,count", [("triangle", 200000), ("hull", 500000)])
def test_draws_are_the_general_clips(walk_bounds, mode, count):
    cases, settled = walk_bounds(mode, count, 3)
    assert settled > cases / 4
