"""The LU-SGS sweeps' schedule and tables, checked on the host (no GPU) from
their definitions by sweep_layout.cpp."""
import os
import subprocess

import pytest

import minifs_amd as mfs

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
PKG = os.path.dirname(mfs.__file__)
CELLS = {"tet": 0, "hex": 1, "prism": 2}


@pytest.fixture(scope="module")
def sweep_layout(tmp_path_factory):
    exe = str(tmp_path_factory.mktemp("layout") / "sweep_layout")
    subprocess.run(["g++", "-std=c++17", "-O2", "-I", os.path.join(PKG, "csrc"), "-o", exe,
                    os.path.join(ROOT, "tests", "sweep_layout.cpp"), "-L", PKG, "-lmfs_hip", f"-Wl,-rpath,{PKG}"],
                   check=True)

    def run(cells, dims, tree, tile, *more):
        cmd = [exe, CELLS[cells], *dims, *tree, tile, *more]
        return subprocess.run([str(x) for x in cmd], capture_output=True, text=True, timeout=60).stdout.strip()

    return run


@pytest.mark.parametrize("tile", [64, 1000, 4096])
@pytest.mark.parametrize("tree", [(4, 512), (2, 16), (2, 128)])
@pytest.mark.parametrize("cells,dims", [("tet", (1, 1, 1)), ("tet", (7, 5, 6)), ("tet", (31, 29, 33)), ("hex", (1, 2, 1)),
                                        ("hex", (9, 8, 11)), ("hex", (41, 43, 40)), ("prism", (3, 1, 2)),
                                        ("prism", (33, 30, 31))])
def test_tables_follow_from_the_mesh(sweep_layout, cells, dims, tree, tile):
    """Chunks cover the cells once, in level order, within their limits of
    cells and dependencies; every dependency comes earlier in both schedules;
    dependency counts and waits are those of the mesh's faces.  Meshes of one
    chunk up to ones laid out on several threads."""
    assert sweep_layout(cells, dims, tree, tile) == "ok"


@pytest.mark.parametrize("direction", [0, 1])
@pytest.mark.parametrize("spoil", ["dependency", "level", "order", "cells", "position"])
def test_order_that_cannot_progress_is_refused(sweep_layout, spoil, direction):
    """A schedule in which a wave could wait for a chunk that comes later, or
    that no wave takes, is an error when the context is created."""
    said = sweep_layout("tet", (14, 12, 13), (2, 64), 1000, spoil, direction)
    assert said == ("forward", "backward")[direction] + " sweep chunks are not topological"
