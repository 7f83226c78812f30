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
