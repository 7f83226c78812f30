"""Cases that time the solver path through the package's public entry points.

A case is one block of a steady solve as a driver, the reference-side
binding or the serving loop runs it: `iters` iterations of one or several
solves, then the flow state and the gradients (or, for several solves, the
states) copied out in the reference's layout.  `prepare` builds the device
contexts and uploads a flow state in the middle of a solve: freestream with
smooth disturbances of a few per cent, drawn from the seed together with
the Mach number and the angle of attack.  The mesh belongs to the case, so
a seed is another flow over the same mesh, as in a sweep of flow conditions.

Fields of a case: `mode` is "step" (Solver.step), "entry" (the loop of the
individual kernel entry points), "noalloc" (mfs_step_noalloc into a device
buffer of the caller) or "batch" (Batch.step); `cells` the cell kind;
`nx, ny, nz` the boxes' hexes per axis (a batch draws its members' sizes
between `lo` and `hi` from `mesh_seed`); `tree`, `leaf` the TDTree
parameters of the cell order; `mixed` the precision; `ghosts` the refresh of
the ghost states after each update; `iters` the iterations of a pass.
"""
from __future__ import annotations

import ctypes
import math

import numpy as np
import torch

import minifs_amd as mfs

STATE = ("rho", "u", "v", "w", "p")
GRADS = ("dqdx", "dqdy", "dqdz")
CFL = 10.0
BUMP_SEED = 20260101
PER_HEX = {"tet": 6, "hex": 1, "prism": 2}
MOST_CELLS = 6_000_000   # the largest mesh: 100^3 hexes of 6 tetrahedra
EXACT_CELL_ITERS = 4.0e6  # above this the numpy path takes too long


def _case(name, mode, nx, ny, nz, iters, cells="tet", tree=4, leaf=512, mixed=False, ghosts=False):
    return {"name": name, "mode": mode, "cells": cells, "nx": nx, "ny": ny, "nz": nz, "tree": tree, "leaf": leaf,
            "mixed": mixed, "ghosts": ghosts, "iters": iters}


def listed():
    return [
        # a mesh of a test or a first try-out (1,296 cells): every level of the sweeps is a few chunks, so launches
        # and dependency latency are all there is
        _case("tet_1k_fp64", "step", 6, 6, 6, 200),
        # the smallest requests of the serving workload (20k cells), solved alone in the default precision
        _case("tet_20k_fp64", "step", 15, 15, 15, 60),
        # a medium request in mixed precision on a box with unequal sides, with the ghost refresh that an unsteady
        # far field needs
        _case("tet_94k_mixed_ghosts", "step", 23, 27, 25, 40, mixed=True, ghosts=True),
        # the reference's driver loop on the individual entry points, as the C++ binding calls them
        _case("tet_384k_entry", "entry", 40, 40, 40, 100),
        # a hexahedral mesh (6 faces per cell, quadrilateral faces)
        _case("hex_262k_fp64", "step", 64, 64, 64, 200, cells="hex"),
        # a prism mesh with odd sides (5 faces per cell) in mixed precision
        _case("prism_195k_mixed", "step", 47, 43, 48, 200, cells="prism", mixed=True),
        # a mesh of 1.3M cells stepped by a caller that must not allocate (its own history buffer on the device)
        _case("tet_1m3_noalloc", "noalloc", 60, 60, 60, 200),
        # a large request (2.9M cells, unequal sides) on the shallower cell order, mixed precision
        _case("tet_2m9_shallow_mixed", "step", 77, 83, 76, 150, tree=2, leaf=128, mixed=True),
        # the benchmark mesh: 6.0M cells in the reference's cell order, FP64
        _case("tet_6m_fp64", "step", 100, 100, 100, 150),
        # the batch that the serving loop steps: 12 requests of 20k to 0.4M cells in one launch per kernel
        {"name": "batch12_mixed", "mode": "batch", "cells": "tet", "members": 12, "lo": 15, "hi": 41, "mesh_seed": 4,
         "tree": 4, "leaf": 512, "mixed": True, "iters": 60},
    ]


def draw(rng):
    """One more case: sizes log-uniform from 1k to 6.0M cells of a box with unequal sides, iterations so that a pass
    stays below the largest listed one's."""
    mode = rng.choice(("step", "step", "step", "entry", "noalloc", "batch"))
    cells = "tet" if mode == "batch" else rng.choice(("tet", "tet", "tet", "hex", "prism"))
    tree, leaf = rng.choice(((4, 512), (4, 512), (4, 512), (2, 128)))
    mixed = rng.random() < 0.5
    if mode == "batch":
        lo = rng.randint(9, 18)
        return {"mode": mode, "cells": cells, "members": rng.randint(2, 12), "lo": lo, "hi": lo + rng.randint(6, 24),
                "mesh_seed": rng.randrange(1 << 20), "tree": tree, "leaf": leaf, "mixed": mixed, "iters": 60}
    n = math.exp(rng.uniform(math.log(1000.0), math.log(0.9 * MOST_CELLS)))
    if cells != "tet":
        n = min(n, 1.0e6)
    side = (n / PER_HEX[cells]) ** (1.0 / 3.0)
    nx = max(3, round(side * rng.uniform(0.85, 1.1)))
    ny = max(3, round(side * rng.uniform(0.85, 1.1)))
    nz = max(3, round(n / PER_HEX[cells] / (nx * ny)))
    ghosts = mode == "step" and rng.random() < 0.25
    iters = 150 if n > 1.0e6 else 100
    case = _case("", mode, nx, ny, nz, iters, cells, tree, leaf, mixed, ghosts)
    del case["name"]
    return case


# ---------------------------------------------------------------- meshes
_MESHES: dict = {}  # the meshes of the case in hand


def _boxes(case):
    if case["mode"] != "batch":
        return [(case["nx"], case["ny"], case["nz"], BUMP_SEED)]
    r = np.random.default_rng(case["mesh_seed"])
    return [tuple(int(r.integers(case["lo"], case["hi"] + 1)) for _ in range(3)) + (int(r.integers(1, 2**31)),)
            for _ in range(case["members"])]


def _meshes(case):
    """The case's preprocessed meshes, kept until another case asks for its own."""
    key = (case["cells"], case["tree"], case["leaf"], tuple(_boxes(case)))
    if key not in _MESHES:
        for grids in _MESHES.values():
            for g in grids:
                g.close()
        _MESHES.clear()
        p = mfs.make_params(mach=0.5, alpha=0.0, cfl=CFL)
        _MESHES[key] = [mfs.Grid.box_bump(nx, ny, nz, seed=s, cells=case["cells"])
                        .decouple(case["tree"], case["leaf"]).preprocess(p) for nx, ny, nz, s in _boxes(case)]
    return _MESHES[key]


def _flow(grid, rng):
    """Flow parameters, and a state in the middle of a solve for every cell and ghost of the mesh."""
    p = mfs.make_params(mach=float(rng.uniform(0.3, 0.85)), alpha=float(rng.uniform(-3.0, 5.0)), cfl=CFL)
    x = [grid.array(nm) for nm in ("xcc", "ycc", "zcc")]

    def mode():
        k, ph = rng.uniform(2.0, 7.0, 3), rng.uniform(0.0, 2.0 * math.pi)
        return np.sin(k[0] * x[0] + k[1] * x[1] + k[2] * x[2] + ph)

    a = math.sqrt(p.gam * p.p_bar / p.rho_s)
    q = [p.rho_s * (1.0 + 0.03 * mode()), p.u_s + 0.03 * a * mode(), p.v_s + 0.03 * a * mode(),
         p.w_s + 0.03 * a * mode(), 0.03 * p.p_bar * mode()]
    # ghosts: the mirrored velocity behind a wall, the freestream behind the far field
    i = grid.info
    nC, nB = i["nTCell"], i["nBFace"]
    c1 = grid.array("f2c").reshape(-1, 2)[:nB, 0]
    n = [grid.array(nm)[:nB] for nm in ("xfn", "yfn", "zfn")]
    wall = grid.array("bctype") == mfs.BC_WALL
    inner = [f[c1] for f in q]
    vn = 2.0 * (n[0] * inner[1] + n[1] * inner[2] + n[2] * inner[3])
    free = (p.rho_s, p.u_s, p.v_s, p.w_s, p.p_s)
    for j in range(5):
        mirrored = inner[j] - vn * n[j - 1] if 1 <= j <= 3 else inner[j]
        q[j][nC:] = np.where(wall, mirrored, free[j])
    return p, q


def _inputs(case, seed):
    rng = np.random.default_rng(seed)
    return [(g,) + _flow(g, rng) for g in _meshes(case)]


# ---------------------------------------------------------------- a case on the GPU
def prepare(case, seed):
    precision = mfs.MFS_MIXED if case["mixed"] else mfs.MFS_FP64
    solvers = []
    for g, p, q in _inputs(case, seed):
        s = mfs.Solver(g, p, precision=precision)
        for nm, f in zip(STATE, q):
            s.upload(nm, f)
        if case.get("ghosts"):
            s.ghost_refresh(True)
        solvers.append(s)
    state = {"case": case, "solvers": solvers}
    if case["mode"] == "batch":
        state["batch"] = mfs.Batch(precision)
        state["solvers"] = [state["batch"].attach(s) for s in solvers]
    elif case["mode"] == "noalloc":
        state["hist"] = torch.zeros(7 * case["iters"], dtype=torch.float64, device="cuda")
        torch.cuda.synchronize()  # the buffer is ready before the solver's own stream writes it
    return state


def run(state):
    case, s = state["case"], state["solvers"][0]
    n = case["iters"]
    if case["mode"] == "batch":
        state["batch"].step(n)
        state["batch"].sync()
        return [[m.field(nm) for nm in STATE] for m in state["solvers"]]
    if case["mode"] == "entry":
        s.iterate_reference_order(n)
    elif case["mode"] == "noalloc":
        lib = mfs.lib()
        if lib.mfs_step_noalloc(s._h, n, ctypes.c_void_p(state["hist"].data_ptr())) != 0:
            raise RuntimeError(lib.mfs_last_error().decode())
    else:
        s.step(n)
    # the state first, then the gradients: what the reference's driver holds after its loop
    return {nm: s.field(nm) for nm in STATE + GRADS}


def work(case):
    """Bytes and operations of one pass.  Per iteration, each array of the path read or written once: per face its
    cells, normal and area and the rest of its geometry in each of the five kernels that walk the faces, per cell the
    state, residual, Diag, DQ and gradients, per boundary face its ghost, per node its weights and values; FP32 halves
    the operator's and the gradients' share.  Then the copied fields, once."""
    by, fl = 0.0, 0.0
    for nx, ny, nz, _ in _boxes(case):
        hexes = nx * ny * nz
        quads = 2 * (nx * ny + ny * nz + nx * nz)
        nN = (nx + 1) * (ny + 1) * (nz + 1)
        if case["cells"] == "tet":
            nC, nB = 6 * hexes, 2 * quads
            nF = (4 * nC + nB) // 2
        elif case["cells"] == "hex":
            nC, nB = hexes, quads
            nF = (6 * nC + nB) // 2
        else:
            nC, nB = 2 * hexes, quads + 2 * nx * ny
            nF = (5 * nC + nB) // 2
        it = 56 * nF + 104 * nC + 40 * nB  # residual, time step, Diag
        op = 2 * (36 * nF + 100 * nC) + 80 * nB + 120 * nC  # both sweeps: operator inputs and DQ; then the update
        gr = 52 * nF + 216 * nC + 156 * nB + 92 * nN  # node values and gradients
        it += (op + gr) * (0.55 if case["mixed"] else 1.0) + (80 * nC if case["mixed"] else 0)
        by += case["iters"] * it + 8.0 * (5 if case["mode"] == "batch" else 20) * (nC + nB)
        fl += case["iters"] * (430.0 * nF + 260.0 * nC)
    return {"bytes": by, "flops": fl}


# ---------------------------------------------------------------- the same in numpy
def exact(case, seed):
    cells = sum(PER_HEX[case["cells"]] * b[0] * b[1] * b[2] for b in _boxes(case))
    if case["mode"] == "batch" or cells * case["iters"] > EXACT_CELL_ITERS:
        return None
    g, p, q = _inputs(case, seed)[0]
    return _Numpy(g, p, np.array(q)).solve(case["iters"], bool(case["ghosts"]))


class _Numpy:
    """The solver iteration on the mesh arrays, in double precision: Roe flux, local time step, LU-SGS over the cell
    order, update, node-based Green-Gauss gradients."""

    def __init__(self, g, p, q):
        a = g.array
        self.p, self.q = p, q
        i = g.info
        self.nC, self.nB, self.nF, self.nN = i["nTCell"], i["nBFace"], i["nTFace"], i["nTNode"]
        nC, nB = self.nC, self.nB
        f2c = a("f2c").reshape(-1, 2)
        self.c1, self.c2 = f2c[:, 0].copy(), f2c[:, 1].copy()
        self.n = np.array([a("xfn"), a("yfn"), a("zfn")])
        self.A, self.vol = a("area"), a("vol")[:nC]
        fc = np.array([a("xfc"), a("yfc"), a("zfc")])
        cc = np.array([a("xcc"), a("ycc"), a("zcc")])
        x = np.array([a("x"), a("y"), a("z")])
        self.wall = a("bctype") == mfs.BC_WALL
        # (cell, face) pairs of the interior cells: first sides, then second sides
        inner = np.arange(nB, self.nF)
        self.pc = np.concatenate([self.c1, self.c2[inner]])
        self.pf = np.concatenate([np.arange(self.nF), inner])
        self.psign = np.concatenate([np.ones(self.nF), -np.ones(len(inner))])
        pnb = np.concatenate([self.c2, self.c1[inner]])
        self.pdn = np.abs(np.sum((fc[:, self.pf] - cc[:, self.pc]) * self.n[:, self.pf], axis=0))
        # sweep levels: a cell follows its lower-numbered neighbours
        low = pnb < self.pc
        level = np.zeros(nC, dtype=np.int64)
        left = np.bincount(self.pc[low], minlength=nC)
        order = np.argsort(pnb[low], kind="stable")
        up, to = pnb[low][order], self.pc[low][order]
        start = np.searchsorted(up, np.arange(nC + 1))
        front, lev = np.flatnonzero(left == 0), 0
        while len(front):
            level[front] = lev
            take = np.concatenate([np.arange(start[c], start[c + 1]) for c in front]) if len(front) else front
            np.subtract.at(left, to[take], 1)
            nxt = np.unique(to[take])
            front, lev = nxt[left[nxt] == 0], lev + 1
        self.fwd = self._schedule(level, low, pnb, range(lev))
        self.bwd = self._schedule(level, pnb > self.pc, pnb, range(lev - 1, -1, -1))
        # node weights: inverse distances; wall nodes from wall faces, far-field nodes from far-field faces, the
        # others from their cells
        nNPF, f2n = a("nNPF"), a("f2n")
        face_of = np.repeat(np.arange(self.nF), nNPF)
        mark = np.zeros(self.nN, dtype=np.int64)
        b = face_of < nB
        bn, bf = f2n[b], face_of[b]
        mark[bn[~self.wall[bf]]] = 2
        mark[bn[self.wall[bf]]] = 1
        use = np.where(self.wall[bf], True, mark[bn] == 2)
        bn, bf = bn[use], bf[use]
        pair = np.unique(np.concatenate([self.c1[face_of].astype(np.int64) * self.nN + f2n,
                                         self.c2[face_of[~b]].astype(np.int64) * self.nN + f2n[~b]]))
        cn, nn = pair // self.nN, pair % self.nN
        keep = mark[nn] == 0
        cn, nn = cn[keep], nn[keep]
        self.eb = (bn, bf, 1.0 / np.sqrt(np.sum((x[:, bn] - fc[:, bf]) ** 2, axis=0)))
        self.ec = (nn, cn, 1.0 / np.sqrt(np.sum((x[:, nn] - cc[:, cn]) ** 2, axis=0)))
        self.den = np.bincount(bn, self.eb[2], self.nN) + np.bincount(nn, self.ec[2], self.nN)
        inside = ~b
        self.fn = (face_of[inside], f2n[inside], nNPF)

    def _schedule(self, level, use, pnb, levels):
        k = np.flatnonzero(use)
        k = k[np.argsort(level[self.pc[k]], kind="stable")]
        lk = level[self.pc[k]]
        cells = np.argsort(level, kind="stable")
        lc = level[cells]
        place = np.empty(self.nC, dtype=np.int64)
        out = []
        for lev in levels:
            c = cells[np.searchsorted(lc, lev):np.searchsorted(lc, lev + 1)]
            place[c] = np.arange(len(c))
            d = k[np.searchsorted(lk, lev):np.searchsorted(lk, lev + 1)]
            out.append((c, place[self.pc[d]], pnb[d], self.psign[d] * self.n[:, self.pf[d]], self.A[self.pf[d]]))
        return out

    def _cells(self, values):
        """Sums per cell of values given per (cell, face) pair."""
        return np.bincount(self.pc, values, self.nC)

    def _energy(self, q):
        return q[4] / self.p.gamm1 + 0.5 * q[0] * (q[1] ** 2 + q[2] ** 2 + q[3] ** 2)

    def _roe(self):
        P, n = self.p, self.n
        L, R = self.q[:, self.c1], self.q[:, self.c2]

        def side(s):
            h = self._energy(s) + P.p_bar / P.gamm1 + s[4] + P.p_bar
            vn = n[0] * s[1] + n[1] * s[2] + n[2] * s[3]
            m = s[0] * vn
            return h, vn, np.array([m, m * s[1] + n[0] * s[4], m * s[2] + n[1] * s[4], m * s[3] + n[2] * s[4], h * vn])

        hl, vl, fl = side(L)
        hr, vr, fr = side(R)
        w = np.sqrt(R[0] / L[0])
        ua = [(L[j] + R[j] * w) / (1.0 + w) for j in (1, 2, 3)]
        ha = (hl / L[0] + hr / R[0] * w) / (1.0 + w)
        ra = np.sqrt(L[0] * R[0])
        va = ua[0] * n[0] + ua[1] * n[1] + ua[2] * n[2]
        q2 = 0.5 * (ua[0] ** 2 + ua[1] ** 2 + ua[2] ** 2)
        c2 = np.abs(P.gamm1 * (ha - q2))
        c = np.sqrt(c2)
        eps = P.alf_l * (np.abs(ua[0]) + np.abs(ua[1]) + np.abs(ua[2]) + c)
        e1, e2, e3 = (np.where(e < 2.0 * eps, e * e * 0.25 / eps + eps, e)
                      for e in (np.abs(va), np.abs(va + c), np.abs(va - c)))
        d, dvn = R - L, vr - vl
        a1 = (d[0] - d[4] / c2) * e1
        a2 = 0.5 * (d[4] / c2 + ra * dvn / c) * e2
        a3 = 0.5 * (d[4] / c2 - ra * dvn / c) * e3
        s, t = a1 + a2 + a3, e1 * ra
        z = -t * dvn + (a2 - a3) * c
        dis = [s] + [s * ua[j] + t * d[j + 1] + z * n[j] for j in range(3)]
        dis.append(a1 * q2 + (a2 + a3) * ha + t * (ua[0] * d[1] + ua[1] * d[2] + ua[2] * d[3]) + z * va)
        return 0.5 * self.A * (fl + fr - np.array(dis))

    def _time_step(self):
        P, q, pc, pf = self.p, self.q, self.pc, self.pf
        a = np.sqrt(P.gam * (q[4] + P.p_bar) / q[0])
        eig = np.abs(q[1][pc] * self.n[0][pf] + q[2][pc] * self.n[1][pf] + q[3][pc] * self.n[2][pf]) + a[pc]
        dt = np.full(self.nC, np.inf)
        np.minimum.at(dt, pc, self.pdn / eig)
        pl, pr = q[4][self.c1], q[4][self.c2]
        jump = np.abs(pr - pl) / (pr + pl + 2.0 * P.p_bar) > 0.1
        rough = np.zeros(self.nC, dtype=bool)
        rough[pc[jump[pf]]] = True
        p, low = q[4][:self.nC], 0.5 * CFL
        cfl = np.where(p > P.p_break, CFL, np.where(p < P.p_min, low,
                       (p - P.p_min) / (P.p_break - P.p_min) * (CFL - low) + low))
        dt *= np.where(rough, low, cfl)
        return dt, self.vol / dt + self._cells(0.5 * self.A[pf] * eig * P.lhs_omga)

    def _term(self, q, dq, n):
        """Change of the normal flux by dq, less the spectral radius times dq."""
        P = self.p

        def flux(Q):
            p = P.gamm1 * (Q[4] - 0.5 * (Q[1] ** 2 + Q[2] ** 2 + Q[3] ** 2) / Q[0])
            vn = (Q[1] * n[0] + Q[2] * n[1] + Q[3] * n[2]) / Q[0]
            return np.array([Q[0] * vn, Q[1] * vn + p * n[0], Q[2] * vn + p * n[1], Q[3] * vn + p * n[2],
                             (Q[4] + p + P.gam * P.p_bar / P.gamm1) * vn])

        Q = np.array([q[0], q[0] * q[1], q[0] * q[2], q[0] * q[3], self._energy(q)])
        vn = q[1] * n[0] + q[2] * n[1] + q[3] * n[2]
        eig = (np.abs(vn) + np.sqrt(P.gam * (q[4] + P.p_bar) / q[0])) * P.lhs_omga
        return flux(Q + dq) - flux(Q) - eig * dq

    def _limit(self, q, d):
        P = self.p
        vv = q[1] ** 2 + q[2] ** 2 + q[3] ** 2
        for factor in (0.1, 0.1, 0.0):
            dp = P.gamm1 * (d[4] + 0.5 * d[0] * vv - (d[1] * q[1] + d[2] * q[2] + d[3] * q[3]))
            bad = ((q[0] + d[0] < P.rho_min) | (q[0] + d[0] > P.rho_max) | (q[4] + dp < P.p_min)
                   | (q[4] + dp > P.p_max))
            d = np.where(bad, d * factor, d)
        return d

    def _lusgs(self, res, diag):
        q, dq = self.q, np.zeros_like(self.q)
        for c, owner, nb, n, A in self.fwd:
            t = 0.5 * A * self._term(q[:, nb], dq[:, nb], n)
            d = (res[:, c] - np.array([np.bincount(owner, tj, len(c)) for tj in t])) / diag[c]
            first = c == 0
            dq[:, c] = np.where(first, d, self._limit(q[:, c], d))
        out = np.zeros_like(dq)
        for c, owner, nb, n, A in self.bwd:
            t = A * self._term(q[:, nb], out[:, nb], n)
            d = dq[:, c] - np.array([np.bincount(owner, tj, len(c)) for tj in t]) / (2.0 * diag[c])
            out[:, c] = self._limit(q[:, c], d)
        return out

    def _update(self, dq):
        P, q = self.p, self.q[:, :self.nC]
        Q = np.array([q[0], q[0] * q[1], q[0] * q[2], q[0] * q[3], self._energy(q)]) + dq[:, :self.nC]
        vel = Q[1:4] / Q[0]

        def relaxed(delta, ratio):
            return np.where(ratio < -0.2, delta / (0.6 + 2.0 * np.abs(ratio)), delta)

        rho = np.clip(q[0] + relaxed(dq[0][:self.nC], dq[0][:self.nC] / q[0]), P.rho_min, P.rho_max)
        dp = P.gamm1 * (Q[4] - 0.5 * np.sum(vel ** 2, axis=0) * rho) - q[4]
        p = np.clip(q[4] + relaxed(dp, dp / (q[4] + P.p_bar)), P.p_min, P.p_max)
        self.q = np.concatenate([np.array([rho, vel[0], vel[1], vel[2], p]), self.q[:, self.nC:]], axis=1)

    def _refresh_ghosts(self):
        P, n = self.p, self.n[:, :self.nB]
        s = self.q[:, self.c1[:self.nB]]
        vn = n[0] * s[1] + n[1] * s[2] + n[2] * s[3]
        mirrored = np.array([s[0]] + [s[j + 1] - 2.0 * vn * n[j] for j in range(3)] + [s[4]])
        # Riemann state of the far field, extrapolated to the ghost
        one = np.ones(self.nB)
        m = np.array([P.rho_s * one, P.u_s * one, P.v_s * one, P.w_s * one, (P.p_s + P.p_bar) * one])
        i = s.copy()
        i[4] = s[4] + P.p_bar
        g1 = P.gam - 1.0
        vm = n[0] * m[1] + n[1] * m[2] + n[2] * m[3]
        out_, in_ = vn + 2.0 * np.sqrt(P.gam * i[4] / i[0]) / g1, vm - 2.0 * np.sqrt(P.gam * m[4] / m[0]) / g1
        vb, cb = 0.5 * (out_ + in_), 0.25 * (out_ - in_) * g1
        enters = vb <= 0.0
        b, bvn = np.where(enters, m, i), np.where(enters, vm, vn)
        rho = (cb * cb / (P.gam * b[4] / b[0] ** P.gam)) ** (1.0 / g1)
        sub = np.array([rho] + [b[j + 1] + (vb - bvn) * n[j] for j in range(3)] + [cb * cb * rho / P.gam])
        far = 2.0 * np.where(np.abs(vb / cb) > 1.0, b, sub) - i
        far[4] -= P.p_bar
        gh = np.where(self.wall, mirrored, far)
        gh[0], gh[4] = np.clip(gh[0], P.rho_min, P.rho_max), np.clip(gh[4], P.p_min, P.p_max)
        self.q[:, self.nC:] = gh

    def _gradients(self):
        q, nB = self.q, self.nB
        face_b = 0.5 * (q[:, self.c1[:nB]] + q[:, self.c2[:nB]])
        bn, bf, bw = self.eb
        nn, cn, cw = self.ec
        node = np.array([(np.bincount(bn, fb[bf] * bw, self.nN) + np.bincount(nn, qj[cn] * cw, self.nN)) / self.den
                         for fb, qj in zip(face_b, q)])
        face, fnode, cnt = self.fn
        out = np.zeros((3, 5, self.nC + nB))
        for j in range(5):
            val = np.bincount(face, node[j][fnode], self.nF) / cnt
            val[:nB] = face_b[j]
            for k in range(3):
                out[k, j, :self.nC] = self._cells(self.psign * (val * self.A * self.n[k])[self.pf]) / self.vol
        return out

    def solve(self, iters, ghosts):
        for _ in range(iters):
            F = self._roe()[:, self.pf] * self.psign
            res = -np.array([self._cells(f) for f in F])
            _, diag = self._time_step()
            self._update(self._lusgs(res, diag))
            if ghosts:
                self._refresh_ghosts()
        g = self._gradients()
        return {**dict(zip(STATE, self.q)), **{nm: g[k].reshape(-1) for k, nm in enumerate(GRADS)}}
