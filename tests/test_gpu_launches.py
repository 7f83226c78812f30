"""GPU tests of what a context's steps launch (mfs_ctx_get_launches), and of
the gradient on each path that those launches take."""
import numpy as np
import pytest

import minifs_amd as mfs
from minifs_amd._lib import MFS_GRADIENT_INSIDE
from minifs_amd.serve import Server

pytestmark = pytest.mark.gpu

FIELDS = ("rho", "u", "v", "w", "p", "res", "dt", "dq", "dqdx", "dqdy", "dqdz", "qnode")


def _grid(cells, dims, tree, seed=4):
    p = mfs.make_params(mach=0.8, alpha=1.25, cfl=10.0)
    return mfs.Grid.box_bump(*dims, seed=seed, cells=cells).decouple(*tree).preprocess(p), p


@pytest.mark.parametrize("cells,n,opts,thin,workgroups,gradient",
                         [("tet", 20, {}, 1, 32, MFS_GRADIENT_INSIDE),
                          ("tet", 20, {"sweep_tail_grid": 1}, 1, 1, MFS_GRADIENT_INSIDE),
                          ("tet", 20, {"sweep_tail_grid": 2}, 1, 1, MFS_GRADIENT_INSIDE),
                          ("tet", 20, {"sweep_tail_grid": 7, "gradient_stream": 3}, 1, 4, 3),
                          ("tet", 20, {"sweep_tail_grid": 100000}, 1, None, MFS_GRADIENT_INSIDE),
                          ("tet", 20, {"sweep_tail_grid": -1}, 0, 0, 5),
                          ("tet", 20, {"sweep_by_tiles": 1}, 0, 0, 5),
                          ("tet", 10, {}, 2, 32, MFS_GRADIENT_INSIDE),
                          ("tet", 10, {"sweep_tail_grid": -1, "gradient_stream": 1}, 2, 32, 1),
                          ("tet", 1, {}, 2, 1, MFS_GRADIENT_INSIDE)])
def test_launches(cells, n, opts, thin, workgroups, gradient):
    """The launches of thin levels, on tetrahedra: none, the tails or both
    sweeps whole, with the option's waves (two each, rounded up to workgroups
    of four), and the gradient's place."""
    print(f"[launches] {cells} {n} {opts}", flush=True)
    g, p = _grid(cells, (n, n, n), (4, 512))
    s = mfs.Solver(g, p, **opts)
    a, info = s.launches(), s.info()
    if workgroups is None:  # as many as the tail has work for
        workgroups = (2 * info["sweep_tail_workgroups"] + 3) // 4
        assert workgroups > 32
    assert (a["thin_launch"], a["thin_workgroups"], a["gradient"]) == (thin, workgroups, gradient), a
    assert (a["wide_workgroups"] > 0) == (thin != 2)
    for chunks, tail in zip(a["chunks"], a["thin_chunks"]):
        if thin == 1:
            assert 0 < tail < chunks and info["sweep_tail_cells"] <= 12 * tail
        else:
            assert tail == (chunks if thin == 2 else 0)
    assert (a["thin_levels"] == info["sweep_levels"]) == (thin == 2) and (a["thin_levels"] > 0) == (thin > 0)
    s.enable_timing(1)  # every kernel group apart: no gradient inside
    assert s.launches()["gradient"] == min(gradient, 5)
    s.close()
    g.close()


def _remapped(tmp_path, dims, tree, bc_text, p):
    """A tetrahedral box whose two patches take other boundary types."""
    g0 = mfs.Grid.box_bump(*dims, seed=4).decouple(*tree)
    mesh, bc = str(tmp_path / "m.mfl"), str(tmp_path / "m.bc")
    g0.save(mesh, bc)
    g0.close()
    open(bc, "w").write(bc_text)
    return mfs.Grid.load(mesh, bc).preprocess(p)


@pytest.mark.parametrize("precision", [mfs.MFS_FP64, mfs.MFS_MIXED], ids=["fp64", "mixed"])
@pytest.mark.parametrize("cells,dims,tree,ghosts,thin", [("tet", (1, 1, 1), (4, 512), False, 2),
                                                         ("tet", (9, 7, 8), (4, 512), True, 2),
                                                         ("tet", (23, 20, 22), (4, 512), True, 1),
                                                         ("tet", (40, 40, 40), (4, 512), False, 1),
                                                         ("tet", (40, 40, 40), (2, 64), False, 1),
                                                         ("symm", (22, 21, 20), (4, 512), False, 1),
                                                         ("hex", (8, 9, 7), (4, 512), False, 2),
                                                         ("hex", (43, 41, 40), (4, 512), True, 1),
                                                         ("hex", (72, 70, 71), (2, 32), False, 1),
                                                         ("prism", (33, 30, 31), (4, 512), False, 1)])
def test_gradient_written_inside_the_thin_launches(tmp_path, cells, dims, tree, ghosts, thin, precision):
    """The node values and gradients that the side work of the thin launches
    writes, left by calls without their last gradient, are those of the
    iteration before as launches of their own write them: bit for bit, for
    tails and sweeps run whole, few and many cells per thin level, symmetry
    nodes, and calls of different lengths after one another."""
    print(f"[launches] gradient inside {cells} {dims} {tree} ghosts={ghosts} precision={precision}", flush=True)
    p = mfs.make_params(mach=0.8, alpha=1.25, cfl=10.0)
    if cells == "symm":
        g = _remapped(tmp_path, dims, tree, "2\n1 4\n2 6\n", p)
    else:
        g, p = _grid(cells, dims, tree)
    a, b = mfs.Solver(g, p, precision=precision), mfs.Solver(g, p, precision=precision, gradient_stream=1)
    assert a.launches()["gradient"] == MFS_GRADIENT_INSIDE and a.launches()["thin_launch"] == thin
    assert b.launches()["gradient"] == 1
    a.last_gradient(False)
    for s in (a, b):
        s.ghost_refresh(ghosts)
    before = a.field("dqdx")
    a.step(1)  # has no gradient but its last
    b.step(1)
    np.testing.assert_array_equal(a.field("dqdx"), before)
    for n in (2, 3, 5, 2):
        a.step(n)
        b.step(n - 1)
        for nm in ("qnode", "dqdx", "dqdy", "dqdz"):
            np.testing.assert_array_equal(a.field(nm), b.field(nm), err_msg=f"{n}: {nm}")
        assert not np.array_equal(a.field("dqdx"), before)
        before = a.field("dqdx")
        b.step(1)
        np.testing.assert_array_equal(a.field("rho"), b.field("rho"), err_msg=f"{n}")
    a.last_gradient(True)
    a.step(2)
    b.step(2)
    for nm in FIELDS:
        np.testing.assert_array_equal(a.field(nm), b.field(nm), err_msg=nm)
    a.close()
    b.close()
    g.close()


@pytest.mark.parametrize("stream", [1, 2, 3, 4, 5])
def test_last_gradient_left_out_on_every_stream(stream):
    """Without its last gradient a call on any of the gradient's streams ends
    with the iteration before's gradient, and everything else as with it."""
    print(f"[launches] last gradient left out, stream {stream}", flush=True)
    g, p = _grid("tet", (12, 11, 13), (4, 512))
    a = mfs.Solver(g, p, gradient_stream=stream, sweep_by_tiles=1 if stream == 5 else 0)
    b = mfs.Solver(g, p, gradient_stream=1)
    assert a.launches()["gradient"] == stream
    a.last_gradient(False)
    for n in (1, 4, 2):
        a.step(n)
        b.step(n - 1)
        if n > 1:
            for nm in ("qnode", "dqdx", "dqdy", "dqdz"):
                np.testing.assert_array_equal(a.field(nm), b.field(nm), err_msg=f"{n}: {nm}")
        b.step(1)
        for nm in ("rho", "u", "v", "w", "p", "res", "dq"):
            np.testing.assert_array_equal(a.field(nm), b.field(nm), err_msg=f"{n}: {nm}")
    np.testing.assert_array_equal(a.history(), b.history())
    a.close()
    b.close()
    g.close()


@pytest.mark.parametrize("cells,dims,tree,precision,ghosts",
                         [("tet", (57, 55, 56), (2, 64), mfs.MFS_FP64, False),
                          ("tet", (57, 55, 56), (2, 64), mfs.MFS_MIXED, False),
                          ("tet", (57, 55, 56), (2, 64), mfs.MFS_MIXED, True),
                          ("tet", (57, 55, 56), (2, 64), mfs.MFS_FP64, True),
                          ("hex", (100, 99, 101), (2, 32), mfs.MFS_MIXED, True),
                          ("prism", (80, 81, 79), (2, 16), mfs.MFS_FP64, False)])
def test_second_stream_gradient_beside_a_split_sweep(cells, dims, tree, precision, ghosts):
    """Shallow orders, whose tails are too short to hide the gradient: it
    starts on the second stream between a sweep's wide launch and its tail.
    Every field and history record equals the solver stream's, across calls
    and with the entry points in between."""
    print(f"[launches] second stream {cells} {dims} {tree} precision={precision} ghosts={ghosts}", flush=True)
    g, p = _grid(cells, dims, tree)
    a, b = (mfs.Solver(g, p, precision=precision, gradient_stream=k) for k in (5, 1))
    assert a.launches()["gradient"] == 5 and a.launches()["thin_launch"] == 1
    for s in (a, b):
        s.ghost_refresh(ghosts)
        s.step(3)
        s.step(1)
        s.iterate_reference_order(1)
        s.step(2)
    for nm in FIELDS:
        np.testing.assert_array_equal(a.field(nm), b.field(nm), err_msg=nm)
    np.testing.assert_array_equal(a.history(), b.history())
    a.last_gradient(False)
    a.step(3)
    b.step(2)
    for nm in ("qnode", "dqdx", "dqdy", "dqdz"):
        np.testing.assert_array_equal(a.field(nm), b.field(nm), err_msg=nm)
    a.close()
    b.close()
    g.close()


@pytest.mark.parametrize("precision", [mfs.MFS_FP64, mfs.MFS_MIXED], ids=["fp64", "mixed"])
@pytest.mark.parametrize("cells,dims,tree,thin", [("hex", (17, 16, 18), (2, 16), 2), ("hex", (20, 20, 20), (4, 512), 2),
                                                  ("hex", (22, 21, 23), (2, 16), 1), ("prism", (16, 16, 16), (2, 128), 2),
                                                  ("prism", (18, 17, 18), (2, 16), 1)])
def test_thin_levels_of_small_six_face_meshes(cells, dims, tree, thin, precision):
    """Levels of up to 128 groups of 8 cells are thin on meshes of every size:
    those of a few thousand cells, some of whose sweeps run whole on one XCD,
    give the tile schedule's bits."""
    print(f"[launches] small six-face mesh {cells} {dims} {tree} precision={precision}", flush=True)
    p = mfs.make_params(mach=0.8, alpha=1.25, cfl=10.0)
    g = mfs.Grid.box_bump(*dims, cells=cells).decouple(*tree).preprocess(p)
    a, b = mfs.Solver(g, p, precision=precision), mfs.Solver(g, p, precision=precision, sweep_by_tiles=1)
    assert a.launches()["thin_launch"] == thin
    for s in (a, b):
        s.step(4)
        s.iterate_reference_order(1)
    for nm in FIELDS:
        np.testing.assert_array_equal(a.field(nm), b.field(nm), err_msg=nm)
    a.close()
    b.close()
    g.close()


@pytest.mark.parametrize("precision", [mfs.MFS_FP64, mfs.MFS_MIXED], ids=["fp64", "mixed"])
@pytest.mark.parametrize("cells,sizes", [("tet", (3,)), ("tet", (36,)), ("tet", (24, 30)), ("hex", (65,)),
                                         ("tet", (10, 3, 12, 8, 5, 9, 2, 11, 4, 6, 7, 3, 5, 4, 2, 8, 9))])
def test_clamp_of_few_and_many_solves(cells, sizes, precision):
    """The ratio_dtmax clamp on in every solve: one small solve (fewer blocks
    than the least), one and two of more blocks than their share, more solves
    than get more than the least.  Each equals the solve alone."""
    print(f"[launches] clamp {cells} {sizes} precision={precision}", flush=True)
    p = mfs.make_params(mach=0.8, alpha=1.25, cfl=10.0, ratio_dtmax=1.2)
    grids = [mfs.Grid.box_bump(n, seed=k + 1, cells=cells).decouple().preprocess(p) for k, n in enumerate(sizes)]
    b = mfs.Batch(precision)
    members = [b.add(g, p) for g in grids]
    b.step(3)
    for m, g in zip(members, grids):
        s = mfs.Solver(g, p, precision=precision)
        s.step(3)
        for nm in FIELDS:
            np.testing.assert_array_equal(m.field(nm), s.field(nm), err_msg=nm)
        np.testing.assert_array_equal(m.history(), s.history())
        s.close()
    b.close()
    for g in grids:
        g.close()


@pytest.mark.parametrize("cells,precision,per_cell", [("tet", mfs.MFS_FP64, 940), ("tet", mfs.MFS_MIXED, 1122),
                                                      ("hex", mfs.MFS_FP64, 1300)])
def test_device_memory_of_a_context(cells, precision, per_cell):
    """A context holds what its steps read: bytes per cell, with room of 2%,
    without the arrays that only its creation reads (36 bytes per tetrahedron,
    52 per hexahedron)."""
    n = 40 if cells == "tet" else 64
    g, p = _grid(cells, (n, n, n), (4, 512))
    s = mfs.Solver(g, p, precision=precision)
    held = s.info()["device_bytes"] / g.info["nTCell"]
    print(f"[launches] {held:.1f} bytes per {cells} cell", flush=True)
    assert held < per_cell
    s.close()
    g.close()


@pytest.mark.parametrize("precision", [mfs.MFS_FP64, mfs.MFS_MIXED], ids=["fp64", "mixed"])
@pytest.mark.parametrize("n", [15, 40])
def test_server_reserves_what_a_request_takes(n, precision):
    """The serving loop's first reservation covers the context of its smallest
    requests and of larger ones, so that the budget holds from the start."""
    print(f"[launches] reservation {n} precision={precision}", flush=True)
    g, p = _grid("tet", (n, n, n), (4, 512))
    s = mfs.Solver(g, p, precision=precision)
    assert s.info()["device_bytes"] <= Server(precision, hbm_budget=1e9).bytes_per_cell * g.info["nTCell"]
    s.close()
    g.close()
