"""GPU tests of what a context's steps launch (mfs_ctx_get_launches), and of
the gradient on each path that those launches take."""
import numpy as np
import pytest

import minifs_amd as mfs
from minifs_amd._lib import MFS_GRADIENT_INSIDE

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
