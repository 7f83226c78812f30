"""GPU tests of device tables that depend on a mesh's face and node order."""
import numpy as np
import pytest

import minifs_amd as mfs
from oracle import Oracle

pytestmark = pytest.mark.gpu

FIELDS = ("rho", "u", "v", "w", "p", "res", "dt", "dq", "dqdx", "dqdy", "dqdz")


@pytest.mark.parametrize("seed", [1, 2, 3])
def test_gradient_with_permuted_face_nodes(tmp_path, seed):
    """The tetrahedra's gradient adds a face's node values in the order of the
    face's own node list.  A mesh whose faces list their nodes in rotated
    order (every rotation occurs; the orientation stays) must give the
    oracle's gradients bit for bit."""
    print(f"[layout] rotated face nodes seed={seed}", flush=True)
    g0 = mfs.Grid.box_bump(4, 5, 3, seed=seed).decouple(2, 16)
    mesh, bc = str(tmp_path / "m.mfl"), str(tmp_path / "m.bc")
    g0.save(mesh, bc)
    raw = np.fromfile(mesh, dtype=np.int32)
    nN, nF, nC = raw[:3]
    at = 3 + 6 * nN  # header, three coordinate blocks of doubles
    assert np.all(raw[at:at + nF] == 3)
    f2n = raw[at + nF:at + nF + 3 * nF].reshape(nF, 3)
    turn = np.random.default_rng(seed).integers(0, 3, nF)
    f2n[:] = np.take_along_axis(f2n, (np.arange(3)[None, :] + turn[:, None]) % 3, axis=1)
    raw.tofile(mesh)
    mach, alpha, cfl, iters = 0.7, 1.5, 10.0, 3
    g = mfs.Grid.load(mesh, bc).preprocess(mfs.make_params(mach=mach, alpha=alpha, cfl=cfl))
    o = Oracle(mesh, bc, mach, alpha, cfl)
    o.run(iters, 0)
    s = mfs.Solver(g, mfs.make_params(mach=mach, alpha=alpha, cfl=cfl))
    s.step(iters)
    for nm in FIELDS:
        np.testing.assert_array_equal(s.field(nm), o.get(nm), err_msg=nm)
    s.close()
    o.close()
    g.close()
    g0.close()


@pytest.mark.parametrize("cells,dims,tree", [("tet", (9, 7, 8), (4, 512)), ("tet", (3, 2, 4), (2, 8)),
                                             ("hex", (13, 9, 11), (4, 512)), ("hex", (2, 1, 3), (2, 8)),
                                             ("prism", (8, 9, 5), (2, 64)), ("tet", (1, 1, 1), (4, 512))])
@pytest.mark.parametrize("opts", [{}, {"tile_cells": 64, "sweep_waves": 8}, {"sweep_by_tiles": 1}],
                         ids=["default", "tile64", "tiles"])
def test_sweep_chunks_bitwise(tmp_path, cells, dims, tree, opts):
    """Sweep chunks of 64 dependencies at their edges: cells without
    dependencies, chunks cut by the dependency and by the cell limit, levels
    of one chunk, meshes of a few cells, each schedule; bit for bit against
    the oracle."""
    print(f"[layout] sweep chunks {cells} {dims} {tree} {opts}", flush=True)
    mach, alpha, cfl, iters = 0.8, 1.25, 10.0, 3
    p = mfs.make_params(mach=mach, alpha=alpha, cfl=cfl)
    g = mfs.Grid.box_bump(*dims, seed=5, cells=cells).decouple(*tree)
    mesh, bc = str(tmp_path / "m.mfl"), str(tmp_path / "m.bc")
    g.save(mesh, bc)
    o = Oracle(mesh, bc, mach, alpha, cfl)
    o.run(iters, 0)
    g.preprocess(p)
    s = mfs.Solver(g, p, **opts)
    s.step(iters)
    for nm in FIELDS:
        np.testing.assert_array_equal(s.field(nm), o.get(nm), err_msg=nm)
    s.close()
    o.close()
    g.close()


@pytest.mark.parametrize("n,amp,opts", [(8, 0.5, {}), (8, 0.1, {}), (8, 0.5, {"sweep_by_tiles": 1}), (20, 0.5, {}),
                                        (20, 0.02, {}), (20, 0.5, {"sweep_tail_grid": -1})])
def test_limiter_paths_bitwise(tmp_path, n, amp, opts):
    """The DQ limiter in every sweep path (all levels thin, wide levels with a
    thin tail, one launch, tiles) on states far from and near the freestream
    with tightened limits, where thin chunks decide by bounds on single
    values whether the cells' five values are exchanged: bit for bit against
    the oracle, whose counters show the limiter's stages (large amplitude);
    and the FP32 operator gives the same bits in every path."""
    from tests import guards

    print(f"[layout] limiter n={n} amp={amp} {opts}", flush=True)
    p = guards.params()
    g0 = mfs.Grid.box_bump(n).decouple()
    mesh, bc = str(tmp_path / "m.mfl"), str(tmp_path / "m.bc")
    g0.save(mesh, bc)
    i = g0.info
    st = guards.perturbed_state(i["nTCell"] + i["nBFace"], p, amp=amp)
    if amp < 0.5:
        st["p"] *= amp
    g = g0.preprocess(p)
    o = Oracle(mesh, bc, guards.MACH, guards.ALPHA, guards.CFL, limits=guards.LIMITS)
    s = mfs.Solver(g, p, **opts)
    for k, a in st.items():
        o.set(k, a)
        s.upload(k, a)
    for it in range(guards.ITERS):
        o.run(1, 0)
        s.step(1)
        for nm in FIELDS:
            np.testing.assert_array_equal(s.field(nm), o.get(nm), err_msg=f"iteration {it}: {nm}")
    c = o.counts()
    if amp == 0.5:
        assert all(c[k] > 0 for k in ("fwd_limit1", "fwd_limit2", "fwd_limit3", "bwd_limit1", "bwd_limit3")), c
    s.close()
    m = [mfs.Solver(g, p, precision=mfs.MFS_MIXED, **kw) for kw in (opts, {"sweep_by_tiles": 1, "tile_cells": 512})]
    for x in m:
        for k, a in st.items():
            x.upload(k, a)
        x.step(guards.ITERS)
    for nm in FIELDS:
        np.testing.assert_array_equal(m[0].field(nm), m[1].field(nm), err_msg=f"mixed {nm}")
        assert np.isfinite(m[0].field(nm)).all()
    for x in m:
        x.close()
    o.close()
    g.close()


@pytest.mark.parametrize("cells,dims", [("tet", (1, 1, 1)), ("hex", (3, 2, 4)), ("hex", (8, 8, 33)),
                                        ("tet", (22, 23, 22)), ("hex", (63, 65, 32)), ("hex", (64, 65, 32))])
@pytest.mark.parametrize("mixed", [False, True])
def test_history_of_the_residual_pass_and_of_its_own_launch(cells, dims, mixed):
    """Up to 512 blocks of 256 cells, the residual pass's last block sums the
    norms and the time step range; above, and with each kernel group timed, a
    launch of its own does.  Both give the same history, bit for bit: meshes
    of one block, with an odd last block, more than 256 blocks, 512 blocks
    and more."""
    print(f"[layout] history {cells} {dims} mixed={mixed}", flush=True)
    out = []
    for level in (0, 1):
        g = mfs.Grid.box_bump(*dims, seed=3, cells=cells).decouple(2, 512)
        p = mfs.make_params(mach=0.8, alpha=1.25, cfl=10.0, ratio_dtmax=1.5)
        g.preprocess(p)
        s = mfs.Solver(g, p, precision=mfs.MFS_MIXED if mixed else mfs.MFS_FP64)
        s.enable_timing(level)
        s.step(2)
        s.step(3)
        out.append((s.history(), s.field("rho"), s.field("dt")))
        s.close()
        g.close()
    assert out[0][0].shape == (5, 7) and np.isfinite(out[0][0]).all()
    for a, b in zip(*out):
        np.testing.assert_array_equal(a, b)


@pytest.mark.parametrize("cells,dims", [("tet", (4, 3, 5)), ("hex", (7, 5, 6)), ("prism", (4, 6, 3))])
@pytest.mark.parametrize("jump", [0.0998, 0.0999, 0.09995, 0.1, 0.1001, 0.5])
def test_pressure_jump_test_near_its_limit(tmp_path, cells, dims, jump):
    """The time step takes the smaller CFL where a face's pressure jump,
    |dp| / (sum of both), exceeds 0.1; away from the limit the residual pass
    decides that without the division.  Two pressures whose jump lies below,
    at and above the limit (and a rounding around it), cell by cell at random:
    bit for bit against the oracle."""
    print(f"[layout] pressure jump {cells} {dims} {jump}", flush=True)
    mach, alpha, cfl = 0.8, 1.25, 10.0
    p = mfs.make_params(mach=mach, alpha=alpha, cfl=cfl)
    g = mfs.Grid.box_bump(*dims, seed=2, cells=cells).decouple(2, 64)
    mesh, bc = str(tmp_path / "m.mfl"), str(tmp_path / "m.bc")
    g.save(mesh, bc)
    n = g.info["nTCell"] + g.info["nBFace"]
    g.preprocess(p)
    rng = np.random.default_rng(11)
    ratio = (1.0 + jump) / (1.0 - jump)
    total = p.p_bar * np.where(rng.random(n) < 0.3, ratio, 1.0) * (1.0 + rng.integers(-2, 3, n) * 2.0**-52)
    st = {"rho": np.full(n, p.rho_s), "u": np.full(n, p.u_s), "v": np.full(n, p.v_s), "w": np.full(n, p.w_s),
          "p": total - p.p_bar}
    o = Oracle(mesh, bc, mach, alpha, cfl)
    s = mfs.Solver(g, p)
    for k, a in st.items():
        o.set(k, a)
        s.upload(k, a)
    o.run(1, 0)
    s.step(1)
    for nm in FIELDS:
        np.testing.assert_array_equal(s.field(nm), o.get(nm), err_msg=nm)
    s.close()
    o.close()
    g.close()


@pytest.mark.parametrize("precision", [mfs.MFS_FP64, mfs.MFS_MIXED])
@pytest.mark.parametrize("cells,sizes", [("tet", (2, 8, 16)), ("hex", (5, 27, 3))])
def test_batch_time_step_clamp_equals_standalone(precision, cells, sizes):
    """The ratio_dtmax clamp of a batch walks each solve's cells on a fixed
    number of workgroups (64 of 256 cells: the middle and last tetrahedral
    meshes and the middle hexahedral one need a second turn or part of one);
    one solve has it off.  Every member equals the same solve alone."""
    print(f"[layout] batch clamp precision={precision} {cells} {sizes}", flush=True)
    cases = []
    for k, n in enumerate(sizes):
        p = mfs.make_params(mach=0.8, alpha=1.25, cfl=10.0, ratio_dtmax=1e80 if k == 0 else 1.2)
        cases.append((mfs.Grid.box_bump(n, seed=k + 1, cells=cells).decouple().preprocess(p), p))
    b = mfs.Batch(precision)
    members = [b.add(g, p) for g, p in cases]
    b.step(3)
    for m, (g, p) in zip(members, cases):
        s = mfs.Solver(g, p, precision=precision)
        s.step(3)
        for nm in FIELDS:
            np.testing.assert_array_equal(m.field(nm), s.field(nm), err_msg=nm)
        np.testing.assert_array_equal(m.history(), s.history())
        s.close()
    b.close()


@pytest.mark.parametrize("precision", [mfs.MFS_FP64, mfs.MFS_MIXED])
@pytest.mark.parametrize("cells,dims,tree", [("tet", (40, 40, 40), (2, 64)), ("tet", (40, 40, 40), (4, 512)),
                                             ("hex", (72, 70, 71), (2, 32)), ("hex", (31, 30, 32), (4, 512))])
def test_gradient_inside_the_tails_equals_the_solver_stream(precision, cells, dims, tree):
    """The gradient as side work of the thin launches, on few or more
    workgroups per CU (many cells per thin level: the shallow orders; few: the
    deep ones), equals the gradient on the solver stream."""
    print(f"[layout] gradient inside {cells} {dims} {tree} precision={precision}", flush=True)
    p = mfs.make_params(mach=0.8, alpha=1.25, cfl=10.0)
    g = mfs.Grid.box_bump(*dims, seed=4, cells=cells).decouple(*tree).preprocess(p)
    out = []
    for stream in (5, 1):
        s = mfs.Solver(g, p, precision=precision, gradient_stream=stream)
        s.step(3)
        out.append([s.field(nm) for nm in ("rho", "dqdx", "dqdy", "dqdz")])
        s.close()
    g.close()
    for a, b in zip(*out):
        np.testing.assert_array_equal(a, b)


@pytest.mark.parametrize("cells,dims", [("hex", (25, 25, 26)), ("hex", (26, 26, 26)), ("prism", (20, 20, 20)),
                                        ("prism", (21, 19, 23))])
def test_thin_line_of_six_face_meshes(cells, dims):
    """On both sides of the mesh size from which levels of up to 128 groups
    are thin, the thin tails' launches give the tile schedule's bits."""
    p = mfs.make_params(mach=0.8, alpha=1.25, cfl=10.0)
    g = mfs.Grid.box_bump(*dims, cells=cells).decouple().preprocess(p)
    a, b = mfs.Solver(g, p), mfs.Solver(g, p, sweep_by_tiles=1)
    for s in (a, b):
        s.step(6)
    for nm in ("rho", "u", "v", "w", "p", "dqdx", "dqdy", "dqdz"):
        np.testing.assert_array_equal(a.field(nm), b.field(nm), err_msg=nm)
    a.close()
    b.close()
