"""CPU: the cloud weight's fixed-point cells against the reference's, over cells
of 0.05 to 1,000 units, with the library's own grid metadata (a host program
linked against the library), and which grids have them at all."""
import os
import subprocess

import numpy as np
import pytest

from amcl3d_amd import _lib

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.fixture(scope="session")
def compare(tmp_path_factory):
    lib = os.path.dirname(os.path.abspath(_lib.LIB_PATH))
    exe = str(tmp_path_factory.mktemp("host") / "fixed_cells")
    subprocess.run(["g++", "-O2", "-std=c++17", "-ffp-contract=off", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include",
                    "-o", exe, os.path.join(ROOT, "tests", "host", "fixed_cells.cpp"), "-L" + lib, "-lamcl3d_gpu",
                    "-Wl,-rpath," + lib, "-L/opt/rocm/lib", "-Wl,-rpath-link,/opt/rocm/lib"], check=True)

    def run(grids):
        text = "".join("%d %d %d %.17g %.17g %.17g %.17g %.17g %d %d\n" % g for g in grids)
        out = subprocess.run([exe], input=text, capture_output=True, text=True, check=True, timeout=300).stdout
        rows = [line.split() for line in out.splitlines()]
        assert len(rows) == len(grids)
        return [(int(f), float(near), int(j), int(w), int(o)) for f, near, j, w, o in rows]

    return run


# units per cell, cells per axis, min
CELLS = [(0.05, (900, 40, 70), (-17.35, 3.1, -0.4)), (0.05, (2000, 2000, 600), (0.0, 0.0, 0.0)),
         (0.05, (4000, 900, 60), (-100.0, 0.0, 0.0)), (0.1, (200, 200, 60), (0.0, 0.0, 0.0)),
         (0.1, (199, 199, 60), (0.0, 0.0, 0.0)), (0.1, (233, 171, 47), (-3.7, 0.2, -1.0)),
         (0.2, (90, 300, 33), (-9.0, 1e-3, 5.0)), (0.25, (64, 128, 20), (-8.0, -16.0, 0.0)),
         (0.3, (100, 77, 25), (2.7, -11.0, -3.0)), (1.0, (500, 300, 40), (-250.0, 0.0, 3.0)),
         (3.3, (700, 300, 40), (-250.0, 0.5, 3.0)), (9.0, (2000, 700, 90), (0.0, -4.0, 1.0)),
         (40.0, (600, 500, 120), (0.0, -7000.0, 11.0)), (50.0, (1000, 800, 60), (0.0, 0.0, 0.0)),
         (250.0, (200, 2000, 60), (1.0, -3.0, 0.0)), (1000.0, (400, 90, 30), (0.0, 0.0, 0.0)),
         (1000.0, (4000, 90, 30), (0.0, 0.0, 0.0)), (3e4, (300, 90, 30), (0.0, 0.0, 0.0))]


@pytest.mark.parametrize("part", range(3))
def test_cells_match_the_reference(compare, part):
    grids = [n + (res,) + mn + (0.0, 3_000_000, 11 + part) for res, n, mn in CELLS[part::3]]
    for g, (fixed, near, compared, wrong, _) in zip(grids, compare(grids)):
        assert wrong == 0, (g, near, compared, wrong)
        if fixed:
            assert compared > 300_000, (g, compared)  # a third of the draws are away from the faces
            assert near <= 2.0 ** -11 * 1.01


def test_random_extents(compare):
    """Whole-cell maps of any extent: the bound of the map, a float, is a face only to within its rounding."""
    rng = np.random.default_rng(5)
    grids = []
    for k in range(120):
        res = float(rng.choice([0.05, 0.1, 0.15, 0.2, 0.5, 1.0, 7.0, 60.0, 333.0]))
        n = tuple(int(v) for v in rng.integers(20, 1200, 3))
        mn = tuple(float(v) for v in np.round(rng.uniform(-50, 50, 3), 2))
        grids.append(n + (res,) + mn + (0.0, 100_000, k))
    for g, (fixed, near, compared, wrong, _) in zip(grids, compare(grids)):
        assert wrong == 0, (g, near, compared, wrong)


def test_which_grids_are_fixed(compare):
    """The mode of the grids the GPU tests weight on: a rule that turned the
    form off everywhere, or on for a grid outside it, would show here."""
    want = {((200, 180, 60), 0.1, (0.0, 0.0, 0.0), 0.0): 1, ((900, 40, 70), 0.05, (-17.35, 3.1, -0.4), 0.0): 1,
            ((64, 128, 20), 0.25, (-8.0, -16.0, 0.0), 0.0): 1, ((199, 199, 60), 0.1, (0.0, 0.0, 0.0), 0.0): 1,
            ((90, 300, 33), 0.2, (-9.0, 1e-3, 5.0), 0.0): 1, ((100, 77, 25), 0.3, (2.7, -11.0, -3.0), 0.0): 1,
            ((4000, 9, 8), 0.05, (-100.0, 0.0, 0.0), 0.0): 1, ((600, 50, 20), 40.0, (0.0, -700.0, 11.0), 0.0): 1,
            ((200, 90, 20), 250.0, (1.0, -3.0, 0.0), 0.0): 1,
            ((9000, 8, 9), 0.05, (-100.0, 0.0, 0.0), 0.0): 0, ((4000, 9, 8), 1000.0, (0.0, 0.0, 0.0), 0.0): 0,
            ((120, 80, 30), 0.1, (0.0, 0.0, 0.0), 0.5): 0, ((150, 90, 40), 0.07, (0.0, -2.0, 0.0), 0.0): 0}
    grids = [n + (res,) + mn + (cut, 1000, 1) for n, res, mn, cut in want]
    got = [r[0] for r in compare(grids)]
    assert dict(zip(want, got)) == want


def test_outside_points_are_not_redone(compare):
    """The point staged for padding and for non-finite points: out of the map
    and away from every face under any pose, so that no lane repeats it."""
    grids = [n + (res,) + mn + (0.0, 1000, 2) for res, n, mn in CELLS]
    rows = compare(grids)
    assert sum(r[0] for r in rows) > len(rows) // 2
    for g, (fixed, near, compared, wrong, outside) in zip(grids, rows):
        assert outside == 0, (g, outside)
