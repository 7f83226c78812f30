// Device-layout construction (see mfs_prep.hpp).
#include "mfs_prep.hpp"

#include <algorithm>
#include <atomic>
#include <cmath>
#include <numeric>
#include <sstream>
#include <thread>

#include "mfs_mesh.hpp"

namespace mfs {


namespace {
constexpr double kTINY_ = 1.e-40;

// Runs fn(begin, end, t) over T contiguous ranges of [0, n) on T threads
// (the calling thread takes the last range).  Every result below is written
// by exactly one range and does not depend on T.
int layout_threads(size_t n) {
    const unsigned hw = std::thread::hardware_concurrency();
    const size_t want = n / 65536 + 1;
    return (int)std::max<size_t>(1, std::min<size_t>({want, hw ? hw : 1, 16}));
}
template <typename F>
void parallel_ranges(size_t n, int T, F&& fn) {
    std::vector<std::thread> th;
    th.reserve(T > 0 ? T - 1 : 0);
    for (int t = 0; t + 1 < T; ++t) th.emplace_back([&, t] { fn(n * t / T, n * (t + 1) / T, t); });
    fn(n * (T - 1) / T, n, T - 1);
    for (auto& x : th) x.join();
}
template <typename F>
void parallel_for(size_t n, F&& fn) {
    parallel_ranges(n, layout_threads(n), [&](size_t b, size_t e, int) {
        for (size_t i = b; i < e; ++i) fn(i);
    });
}
}  // namespace

std::string check_sweep_order(const HostLayout& L, int dir, const lvec<LatestDep>& latest) {
    const SweepLayout& S = L.sweep[dir];
    const int n = S.nchunk;
    auto first = [&](int u) { return S.crec[4 * (size_t)u]; };
    auto cells = [&](int u) { return S.crec[4 * (size_t)u + 1] & 0xff; };
    auto depth = [&](int d) {
        const int l = L.flevel[L.cell_of_dev[d]];
        return dir == 0 ? l : L.nlev - l;
    };
    // the chunks of all tiles, forward or backward in each, cover the cells
    bool ok = true;
    int next = 0;
    for (size_t t = 0; t + 1 < S.tile_chunk.size() && ok; ++t) {
        const int b = S.tile_chunk[t], e = S.tile_chunk[t + 1];
        for (int k = 0; k < e - b && ok; ++k) {
            const int i = dir == 0 ? b + k : e - 1 - k, u = S.pos[i];
            ok = u >= 0 && u < n && first(u) == next && cells(u) > 0 && (i == b || S.pos[i - 1] < u);
            if (ok) next += cells(u);
        }
    }
    ok = ok && S.tile_chunk.back() == n && next == L.nC;
    // each has cells of one depth, none less deep than the chunk before, and
    // every cell's latest dependency is less deep
    std::atomic<bool> ordered{true};
    if (ok)
        parallel_for(n, [&](size_t uu) {
            const int u = (int)uu, l = depth(first(u));
            bool good = u == 0 || depth(first(u - 1)) <= l;
            for (int d = first(u); d < first(u) + cells(u); ++d) good = good && depth(d) == l && latest[d].rank < 2 * l;
            if (!good) ordered = false;
        });
    return ok && ordered ? "" : std::string(dir == 0 ? "forward" : "backward") + " sweep chunks are not topological";
}

std::string build_layout(const mfs_mesh_view& v, HostLayout& L, int kTileCells) {
    if (kTileCells < 64) return "tile size must be at least 64 cells";
    if (v.nTCell <= 0 || v.nTFace <= 0 || v.nTNode <= 0 || v.nBFace < 0 || v.nBFace > v.nTFace)
        return "mesh view has invalid sizes";
    if (!v.x || !v.y || !v.z || !v.nNPF || !v.f2n || !v.f2c || !v.xfn || !v.yfn || !v.zfn || !v.area || !v.xfc ||
        !v.yfc || !v.zfc || !v.xcc || !v.ycc || !v.zcc || !v.vol || !v.rho || !v.u || !v.v || !v.w || !v.p ||
        (v.nBFace > 0 && !v.bc_type))
        return "mesh view has a null array";
    const int nC = v.nTCell, nF = v.nTFace, nB = v.nBFace, nN = v.nTNode, n = nC + nB;
    L.nC = nC;
    L.nF = nF;
    L.nB = nB;
    L.nN = nN;

    // ---- mesh-order face tables and validation
    std::vector<int> mfo(nF + 1);
    mfo[0] = 0;
    for (int i = 0; i < nF; ++i) {
        if (v.nNPF[i] < 3) return "face with fewer than 3 nodes";
        mfo[i + 1] = mfo[i] + v.nNPF[i];
    }
    for (int k = 0; k < mfo[nF]; ++k)
        if (v.f2n[k] < 0 || v.f2n[k] >= nN) return "f2n has an invalid node";
    for (int i = 0; i < nF; ++i) {
        const int a = v.f2c[2 * i], b = v.f2c[2 * i + 1];
        if (a < 0 || a >= nC) return "f2c has an invalid first cell";
        if (i < nB) {
            if (b != nC + i) return "boundary face k must have ghost cell nTCell+k (SpecifyBC)";
        } else if (b < 0 || b >= nC || b == a) {
            return "interior face has an invalid second cell";
        }
    }
    L.btype.assign(v.bc_type, v.bc_type + nB);

    // ---- mesh cell -> faces in ascending mesh face id (CalnFPC/CalC2F)
    std::vector<int> mcfo(nC + 1, 0), mcf;
    for (int i = 0; i < nF; ++i) {
        mcfo[v.f2c[2 * i] + 1]++;
        if (i >= nB) mcfo[v.f2c[2 * i + 1] + 1]++;
    }
    for (int c = 0; c < nC; ++c) mcfo[c + 1] += mcfo[c];
    mcf.resize(mcfo[nC]);
    {
        std::vector<int> fill(mcfo.begin(), mcfo.end() - 1);
        for (int i = 0; i < nF; ++i) {
            mcf[fill[v.f2c[2 * i]]++] = i;
            if (i >= nB) mcf[fill[v.f2c[2 * i + 1]]++] = i;
        }
    }
    L.max_faces = 0;
    for (int c = 0; c < nC; ++c) {
        const int k = mcfo[c + 1] - mcfo[c];
        if (k == 0) return "cell without faces";
        L.max_faces = std::max(L.max_faces, k);
    }
    if (L.max_faces > 8) return "cells with more than 8 faces are not supported";
    auto other = [&](int c, int f) { return v.f2c[2 * f] == c ? v.f2c[2 * f + 1] : v.f2c[2 * f]; };

    // ---- LU-SGS levels on mesh ids.  With LUSGSLayer[i] = i
    // (ReorderCellforLUSGS_0, grid_polyhedra.cpp:1127-1142) the forward sweep
    // of cell c reads the final DQ of every face neighbour with a smaller id
    // and the backward sweep that of every neighbour with a larger id.
    L.flevel.assign(nC, 0);
    int mf = 0;
    for (int c = 0; c < nC; ++c) {
        int l = 0;
        for (int k = mcfo[c]; k < mcfo[c + 1]; ++k) {
            const int f = mcf[k];
            if (f < nB) continue;
            const int nb = other(c, f);
            if (nb < c) l = std::max(l, L.flevel[nb] + 1);
        }
        L.flevel[c] = l;
        mf = std::max(mf, l);
    }
    L.nlev = mf + 1;

    // ---- device cell order: tile (kTileCells consecutive mesh ids, a
    // compact region in TDTree numbering), then forward level, then mesh id.
    // The cells of one level inside a tile are contiguous (sweep chunks),
    // and a cell's face neighbours are mostly in its own tile (gathers of
    // the face kernels stay in a small window of memory).
    std::vector<int> dcell(nC);
    std::vector<int> gfirst, glevel, gtile;  // (tile, level) groups: first device cell (and nC), level, tile
    {
        const int ntile = (nC + kTileCells - 1) / kTileCells;
        const size_t nkey = (size_t)ntile * L.nlev;
        std::vector<int> cnt(nkey + 1, 0);
        auto key = [&](int c) { return (size_t)(c / kTileCells) * L.nlev + L.flevel[c]; };
        for (int c = 0; c < nC; ++c) cnt[key(c) + 1]++;
        for (size_t k = 0; k < nkey; ++k) {
            if (cnt[k + 1] > 0) {
                gfirst.push_back(cnt[k]);
                glevel.push_back((int)(k % L.nlev));
                gtile.push_back((int)(k / L.nlev));
            }
            cnt[k + 1] += cnt[k];
        }
        gfirst.push_back(nC);
        L.cell_of_dev.resize(nC);
        for (int c = 0; c < nC; ++c) {
            const int d = cnt[key(c)]++;
            dcell[c] = d;
            L.cell_of_dev[d] = c;
        }
    }
    L.dev_cell0 = dcell[0];
    auto dmap = [&](int c) { return c < nC ? dcell[c] : c; };  // ghosts keep nC+k

    // ---- device face order: first touch in the device cell traversal
    std::vector<int> dface(nF, -1);
    L.face_of_dev.resize(nF);
    {
        int next = 0;
        for (int d = 0; d < nC; ++d) {
            const int c = L.cell_of_dev[d];
            for (int k = mcfo[c]; k < mcfo[c + 1]; ++k) {
                const int f = mcf[k];
                if (dface[f] < 0) {
                    dface[f] = next;
                    L.face_of_dev[next] = f;
                    ++next;
                }
            }
        }
        if (next != nF) return "face not attached to any cell";
    }
    // per device cell: device face ids, still in ascending mesh face id, the
    // sweep dependency masks and, per direction, the cell's latest dependency
    lvec<LatestDep> latest[2];
    for (auto& l : latest) l.resize(nC);
    L.cfo.assign(nC + 1, 0);
    L.cf.resize(mcf.size());
    L.depmask.assign(nC, 0);
    for (int d = 0; d < nC; ++d) L.cfo[d + 1] = L.cfo[d] + (mcfo[L.cell_of_dev[d] + 1] - mcfo[L.cell_of_dev[d]]);
    parallel_for(nC, [&](size_t dd) {
        {
            const int d = (int)dd;
            int pos = L.cfo[d];
            const int c = L.cell_of_dev[d];
            int s = 0;
            unsigned mask = 0;
            LatestDep late[2] = {{-1, -1}, {-1, -1}};
            for (int k = mcfo[c]; k < mcfo[c + 1]; ++k, ++s) {
                const int f = mcf[k];
                L.cf[pos++] = dface[f];
                const int nb = other(c, f);
                if (nb < c) mask |= 1u << s;  // ghosts have nb >= nC > c
                if (nb > c) {
                    mask |= 1u << (8 + s);
                    if (nb < nC) mask |= 1u << (16 + s);
                }
                if (nb < nC) {
                    const int dir = nb < c ? 0 : 1, l = L.flevel[nb];
                    const int rank = 2 * (dir == 0 ? l : L.nlev - l) + (nb / kTileCells != c / kTileCells ? 1 : 0);
                    if (rank > late[dir].rank) late[dir] = {rank, dcell[nb]};
                }
                // gradient: boundary faces other than SYMM and INTERFACE take
                // the face-centre average of cell and ghost instead of the
                // node mean (cal_gradient.cpp:1740-1795)
                if (nb >= nC) {
                    const int t = L.btype[nb - nC];
                    if (t != BC_SYMM && t != BC_INTERFACE) mask |= 1u << (24 + s);
                }
            }
            L.depmask[d] = (int)mask;
            for (int dir = 0; dir < 2; ++dir) latest[dir][d] = late[dir];
        }
    });

    // ---- device node order: first touch over the device faces
    std::vector<int> dnode(nN, -1);
    L.node_of_dev.assign(nN, -1);
    {
        int next = 0;
        for (int d = 0; d < nF; ++d) {
            const int f = L.face_of_dev[d];
            for (int j = mfo[f]; j < mfo[f + 1]; ++j) {
                const int p = v.f2n[j];
                if (dnode[p] < 0) {
                    dnode[p] = next;
                    L.node_of_dev[next] = p;
                    ++next;
                }
            }
        }
        for (int p = 0; p < nN; ++p)  // nodes used by no face keep their relative order at the end
            if (dnode[p] < 0) {
                dnode[p] = next;
                L.node_of_dev[next] = p;
                ++next;
            }
    }

    // ---- faces in device order
    L.c1.resize(nF);
    L.c2.resize(nF);
    L.fgeo.resize(4 * (size_t)nF);
    L.dn1.resize(nF);
    L.dn2.assign(nF, 0.0);
    L.fno.resize(nF + 1);
    L.fno[0] = 0;
    for (int d = 0; d < nF; ++d) L.fno[d + 1] = L.fno[d] + v.nNPF[L.face_of_dev[d]];
    L.fn.resize(mfo[nF]);
    parallel_for(nF, [&](size_t dd) {
        const int d = (int)dd;
        const int i = L.face_of_dev[d];
        const int a = v.f2c[2 * i], b = v.f2c[2 * i + 1];
        L.c1[d] = dmap(a);
        L.c2[d] = dmap(b);
        L.fgeo[4 * (size_t)d + 0] = v.xfn[i];
        L.fgeo[4 * (size_t)d + 1] = v.yfn[i];
        L.fgeo[4 * (size_t)d + 2] = v.zfn[i];
        L.fgeo[4 * (size_t)d + 3] = v.area[i];
        // TimeStepNormal_new (compute_timestep.cpp:758-823): the same
        // expression in every iteration, so it is evaluated once here.
        L.dn1[d] = fabs((v.xfc[i] - v.xcc[a]) * v.xfn[i] + (v.yfc[i] - v.ycc[a]) * v.yfn[i] +
                        (v.zfc[i] - v.zcc[a]) * v.zfn[i]);
        if (i >= nB)
            L.dn2[d] = fabs((v.xfc[i] - v.xcc[b]) * v.xfn[i] + (v.yfc[i] - v.ycc[b]) * v.yfn[i] +
                            (v.zfc[i] - v.zcc[b]) * v.zfn[i]);
        for (int j = mfo[i], o = L.fno[d]; j < mfo[i + 1]; ++j, ++o) L.fn[o] = dnode[v.f2n[j]];
    });
    L.vol.resize(nC);
    parallel_for(nC, [&](size_t d) { L.vol[d] = v.vol[L.cell_of_dev[d]]; });

    // ---- node weights (ComputeWeight3D_Node, grid_polyhedra_auxiliary_functions.cpp:831-1049)
    // and the accumulation order of CompNodeVar3D_dist (cal_gradient.cpp:1922-2372),
    // computed on mesh ids.
    std::vector<double> wnode(nN, 0.0);
    std::vector<int> Nmark(nN, 0);
    std::vector<double> wbf(mfo[nB] + 1, 0.0);  // WeightNodeBFace2C
    auto bf_weight = [&](int i, int j, int p1) {
        const double dx = v.x[p1] - v.xfc[i], dy = v.y[p1] - v.yfc[i], dz = v.z[p1] - v.zfc[i];
        double wr = dx * dx + dy * dy + dz * dz;
        wr = sqrt(wr);
        wr = 1. / wr;
        wbf[mfo[i] + j] = wr;
        wnode[p1] += wr;
    };
    for (int i = 0; i < nB; i++) {
        if (L.btype[i] != BC_WALL) continue;
        for (int j = 0; j < v.nNPF[i]; j++) {
            const int p1 = v.f2n[mfo[i] + j];
            bf_weight(i, j, p1);
            Nmark[p1] = BC_WALL;
        }
    }
    for (int i = 0; i < nB; i++) {
        if (L.btype[i] != BC_FAR_FIELD && L.btype[i] != BC_FAR_FIELD_MOD) continue;
        for (int j = 0; j < v.nNPF[i]; j++) {
            const int p1 = v.f2n[mfo[i] + j];
            if (Nmark[p1] == BC_WALL) continue;
            bf_weight(i, j, p1);
            Nmark[p1] = BC_FAR_FIELD;
        }
    }
    for (int i = 0; i < nB; i++) {
        const int t = L.btype[i];
        if (t == BC_WALL || t == BC_SYMM || t == BC_FAR_FIELD || t == BC_FAR_FIELD_MOD || t == BC_INTERFACE) continue;
        for (int j = 0; j < v.nNPF[i]; j++) {
            const int p1 = v.f2n[mfo[i] + j];
            if (Nmark[p1] == BC_WALL || Nmark[p1] == BC_FAR_FIELD) continue;
            bf_weight(i, j, p1);
            Nmark[p1] = 101;
        }
    }
    // Face loops of CompNodeVar3D_dist: WALL faces, FAR_FIELD faces (not on
    // WALL nodes), other types (not on WALL or FAR_FIELD nodes); then the
    // cell loop, whose per-node order is ascending mesh cell id because
    // each (cell,node) pair is visited once.
    auto loop_of = [&](int i) {
        const int t = L.btype[i];
        if (t == BC_WALL) return 1;
        if (t == BC_FAR_FIELD) return 2;
        if (t == BC_SYMM || t == BC_INTERFACE) return 0;
        return 3;
    };
    auto face_entry_ok = [&](int p1, int loop) {
        if (loop == 1) return true;
        if (loop == 2) return Nmark[p1] != BC_WALL;
        return Nmark[p1] != BC_WALL && Nmark[p1] != BC_FAR_FIELD;
    };
    std::vector<int> ecount(nN, 0);
    for (int loop = 1; loop <= 3; ++loop)
        for (int i = 0; i < nB; i++) {
            if (loop_of(i) != loop) continue;
            for (int j = mfo[i]; j < mfo[i + 1]; j++)
                if (face_entry_ok(v.f2n[j], loop)) ecount[v.f2n[j]]++;
        }
    // The cell loop on threads, each over a contiguous range of cells: a
    // node's entries come in ascending cell id, so thread t's entries of
    // node p follow those of threads < t (a counting sort per node).
    auto cell_nodes = [&](int c, std::vector<int>& nodes) {  // the cell's distinct nodes, first-visit order
        nodes.clear();
        for (int k = mcfo[c]; k < mcfo[c + 1]; ++k) {
            const int f = mcf[k];
            for (int j = mfo[f]; j < mfo[f + 1]; ++j) {
                const int p1 = v.f2n[j];
                if (std::find(nodes.begin(), nodes.end(), p1) == nodes.end()) nodes.push_back(p1);
            }
        }
    };
    const int TC = layout_threads(nC);
    std::vector<std::vector<int>> tcount(TC);  // per thread: interior-node entries per node, then fill offsets
    parallel_ranges(nC, TC, [&](size_t b, size_t e, int t) {
        std::vector<int>& cnt = tcount[t];
        cnt.assign(nN, 0);
        std::vector<int> nodes;
        for (int c = (int)b; c < (int)e; ++c) {
            cell_nodes(c, nodes);
            for (int p1 : nodes)
                if (Nmark[p1] == 0) cnt[p1]++;
        }
    });
    for (int t = 0; t < TC; ++t)
        for (int p1 = 0; p1 < nN; ++p1) ecount[p1] += tcount[t][p1];
    L.nlo.assign(nN + 1, 0);
    for (int d = 0; d < nN; ++d) L.nlo[d + 1] = L.nlo[d] + ecount[L.node_of_dev[d]];
    L.nla.resize(L.nlo[nN]);
    L.nlb.resize(L.nlo[nN]);
    L.nlw.resize(L.nlo[nN]);
    std::vector<int> efill(nN);
    for (int d = 0; d < nN; ++d) efill[L.node_of_dev[d]] = L.nlo[d];
    for (int loop = 1; loop <= 3; ++loop)
        for (int i = 0; i < nB; i++) {
            if (loop_of(i) != loop) continue;
            for (int j = 0; j < v.nNPF[i]; j++) {
                const int p1 = v.f2n[mfo[i] + j];
                if (!face_entry_ok(p1, loop)) continue;
                const int e = efill[p1]++;
                L.nla[e] = dmap(v.f2c[2 * i]);
                L.nlb[e] = v.f2c[2 * i + 1];  // ghost
                L.nlw[e] = wbf[mfo[i] + j];
            }
        }
    // each thread's first entry of every interior node
    parallel_for(nN, [&](size_t pp) {
        int o = efill[pp];
        for (int t = 0; t < TC; ++t) {
            const int k = tcount[t][pp];
            tcount[t][pp] = o;
            o += k;
        }
    });
    parallel_ranges(nC, TC, [&](size_t b, size_t e, int t) {
        std::vector<int>& off = tcount[t];
        std::vector<int> nodes;
        for (int c = (int)b; c < (int)e; ++c) {
            cell_nodes(c, nodes);
            for (int p1 : nodes) {
                if (Nmark[p1] != 0) continue;
                const double dx = v.x[p1] - v.xcc[c], dy = v.y[p1] - v.ycc[c], dz = v.z[p1] - v.zcc[c];
                double wr = dx * dx + dy * dy + dz * dz;
                wr = sqrt(wr);
                wr = 1. / wr;
                const int en = off[p1]++;
                L.nla[en] = dcell[c];
                L.nlb[en] = -1;
                L.nlw[en] = wr;
            }
        }
    });
    tcount.clear();
    // WeightNode of an interior node: its cell weights summed in ascending
    // cell id, the order of the reference's loop (:1007-1044)
    L.nden.resize(nN);
    parallel_for(nN, [&](size_t dd) {
        const int pp = L.node_of_dev[dd];
        if (Nmark[pp] == 0) {
            double w = 0.0;
            for (int en = L.nlo[dd]; en < L.nlo[dd + 1]; ++en) w += L.nlw[en];
            wnode[pp] = w;
        }
        L.nden[dd] = wnode[pp] + kTINY_;
    });

    // FindNodeSYMM (grid_polyhedra_auxiliary_functions.cpp:2060-2140)
    {
        std::vector<int> nodesymm(nN, 2);
        std::vector<double> xs(nN, 0.0), ys(nN, 0.0), zs(nN, 0.0), nface(nN, 0.0);
        for (int i = 0; i < nB; i++) {
            if (L.btype[i] != BC_SYMM) continue;
            for (int j = mfo[i]; j < mfo[i + 1]; j++) {
                const int p1 = v.f2n[j];
                nodesymm[p1] = 1;
                xs[p1] += v.xfn[i];
                ys[p1] += v.yfn[i];
                zs[p1] += v.zfn[i];
                nface[p1] += 1.0;
            }
        }
        L.sym_node.clear();
        L.sym_n.clear();
        for (int d = 0; d < nN; ++d) {
            const int p = L.node_of_dev[d];
            if (nodesymm[p] == 1) {
                L.sym_node.push_back(d);
                L.sym_n.push_back(xs[p] / nface[p]);
                L.sym_n.push_back(ys[p] / nface[p]);
                L.sym_n.push_back(zs[p] / nface[p]);
            }
        }
    }

    // ---- sweep chunks, per direction (mfs_prep.hpp).  A lower neighbour has
    // a smaller mesh id (same or earlier tile) and a lower level, so every
    // forward dependency lies in an earlier level and tile order and every
    // backward dependency in a later one.
    L.lpc = L.max_faces <= 4 ? 4 : 8;
    {
        // the levels' widths in 64/lpc-cell units
        const int unit = 64 / L.lpc;
        const int ng = (int)glevel.size();
        std::vector<int> width(L.nlev, 0);
        for (int g = 0; g < ng; ++g) width[glevel[g]] += (gfirst[g + 1] - gfirst[g] + unit - 1) / unit;
        // The run of levels of at most `line` groups that ends the order: its
        // first level (nlev without one, or where it is shorter than
        // kMinTailChunks or the whole order), groups and cells.
        auto tail_of = [&](int line, int& levels, int& groups, int& cells) {
            int first = L.nlev;
            groups = cells = 0;
            while (first > 0 && width[first - 1] <= line) groups += width[--first];
            levels = L.nlev - first;
            if (first == 0 || groups < kMinTailChunks) {
                first = L.nlev;
                groups = 0;
            }
            for (int g = 0; g < ng; ++g)
                if (glevel[g] >= first) cells += gfirst[g + 1] - gfirst[g];
            return first;
        };
        const int line = L.lpc == 8 ? kWideThinLevelChunks : kThinLevelChunks;
        const int tail_level = tail_of(line, L.thin_levels, L.tail_chunks, L.tail_cells);
        L.all_thin = L.thin_levels == L.nlev;
        int levels = 0;
        tail_of(kThinLevelChunks, levels, L.narrow_chunks, L.narrow_cells);
        std::vector<char> thin(L.nlev);
        for (int l = 0; l < L.nlev; ++l) thin[l] = width[l] <= line;
        L.cdep.resize(2 * (size_t)nC);
        std::vector<int> gchunk(ng + 1);
        for (int dir = 0; dir < 2; ++dir) {
            SweepLayout& S = L.sweep[dir];
            // The chunks of group g in device order: fn(first cell, cells,
            // dependencies) for each, cell(d, dependencies before it in its
            // chunk, its own) for each cell.
            auto cut = [&](int g, auto&& fn, auto&& cell) {
                const int most = thin[glevel[g]] ? kThinCells : 64;
                for (int d = gfirst[g]; d < gfirst[g + 1];) {
                    const int first = d;
                    int deps = 0;
                    while (d < gfirst[g + 1] && d - first < most) {
                        const int n = __builtin_popcount(((unsigned)L.depmask[d] >> (8 * dir)) & 0xffu);
                        if (deps + n > 64) break;
                        cell(d, deps, n);
                        deps += n;
                        ++d;
                    }
                    fn(first, d - first, deps);
                }
            };
            parallel_ranges(ng, layout_threads(nC), [&](size_t b, size_t e, int) {
                for (int g = (int)b; g < (int)e; ++g) {
                    int k = 0;
                    cut(g, [&](int, int, int) { ++k; },
                        [&](int d, int start, int n) { L.cdep[2 * (size_t)d + dir] = (unsigned short)(start | (n << 8)); });
                    gchunk[g + 1] = k;
                }
            });
            gchunk[0] = 0;
            for (int g = 0; g < ng; ++g) gchunk[g + 1] += gchunk[g];
            const int nchunk = gchunk[ng];
            S.nchunk = nchunk;
            S.tile_chunk.clear();
            for (int g = 0; g < ng; ++g)
                if (g == 0 || gtile[g] != gtile[g - 1]) S.tile_chunk.push_back(gchunk[g]);
            S.tile_chunk.push_back(nchunk);
            // flat order: forward by level, then device order (a stable
            // counting sort over the groups); backward exactly from the end
            std::vector<int> at(L.nlev + 1, 0);
            for (int g = 0; g < ng; ++g) at[glevel[g] + 1] += gchunk[g + 1] - gchunk[g];
            for (int l = 0; l < L.nlev; ++l) at[l + 1] += at[l];
            S.tail = nchunk - at[tail_level];
            S.pos.resize(nchunk);
            S.crec.resize(4 * (size_t)nchunk);
            S.batch_wait.resize(nchunk);
            std::vector<int> gat(ng);  // forward position of the group's first chunk
            for (int g = 0; g < ng; ++g) {
                gat[g] = at[glevel[g]];
                at[glevel[g]] += gchunk[g + 1] - gchunk[g];
            }
            parallel_ranges(ng, layout_threads(nC), [&](size_t b, size_t e, int) {
                for (int g = (int)b; g < (int)e; ++g) {
                    int k = 0;
                    cut(g,
                        [&](int first, int cells, int deps) {
                            const int u = dir == 0 ? gat[g] + k : nchunk - 1 - (gat[g] + k);
                            S.pos[gchunk[g] + k] = u;
                            S.crec[4 * (size_t)u] = first;
                            S.crec[4 * (size_t)u + 1] = cells | (deps << 8) | (thin[glevel[g]] ? kThinChunkFlag : 0);
                            ++k;
                        },
                        [](int, int, int) {});
                }
            });
            size_t nd = 0;
            for (int u = 0; u < nchunk; ++u) {
                S.crec[4 * (size_t)u + 2] = (int)nd;
                nd += (S.crec[4 * (size_t)u + 1] >> 8) & 0xff;
            }
            S.ndep = nd;
            if (nd > 0x7fffffffu - 64) return "mesh too large for the sweep tables";
            // the tile schedule walks a tile's chunks in the sweep's order
            if (dir == 1)
                for (size_t t = 0; t + 1 < S.tile_chunk.size(); ++t)
                    std::reverse(S.pos.begin() + S.tile_chunk[t], S.pos.begin() + S.tile_chunk[t + 1]);
            // per chunk the dependency of the latest level, another tile's
            // first, the first of equal rank in the chunk's cell and face
            // order; narrow levels wait on that dependency's own latest
            parallel_for(nchunk, [&](size_t u) {
                const int d0 = S.crec[4 * u], cells = S.crec[4 * u + 1] & 0xff;
                LatestDep rep = latest[dir][d0];
                for (int d = d0 + 1; d < d0 + cells; ++d)
                    if (latest[dir][d].rank > rep.rank) rep = latest[dir][d];
                const int further = rep.cell >= 0 ? latest[dir][rep.cell].cell : -1;
                const int groups = width[L.flevel[L.cell_of_dev[d0]]];
                S.batch_wait[u] = groups <= kBatchDirectLevelChunks ? further : rep.cell;
                S.crec[4 * u + 3] = groups <= kDirectLevelChunks ? further : rep.cell;
            });
            const std::string e = check_sweep_order(L, dir, latest[dir]);
            if (!e.empty()) return e;
        }
        // face slots per device cell (device face ids, ascending mesh face id, -1 = none)
        L.cfs.assign((size_t)nC * L.lpc, -1);
        parallel_for(nC, [&](size_t d) {
            for (int k = L.cfo[d]; k < L.cfo[d + 1]; ++k) L.cfs[d * L.lpc + (k - L.cfo[d])] = L.cf[k];
        });
        // tetrahedral meshes whose slots are all triangles take the
        // gradient's slot-node path (the device builds the slot tables from
        // cfs and the face arrays)
        L.tri_slots = false;
        if (L.max_faces == 4) {
            bool tri = true;
            for (size_t i = 0; i < L.cfs.size() && tri; ++i) {
                const int f = L.cfs[i];
                tri = f >= 0 && L.fno[f + 1] - L.fno[f] == 3;
            }
            L.tri_slots = tri;
        }
    }

    // ---- state, device order (ghosts unchanged)
    L.q.resize(5 * (size_t)n);
    const double* src[5] = {v.rho, v.u, v.v, v.w, v.p};
    parallel_for(nC, [&](size_t d) {
        for (int j = 0; j < 5; ++j) L.q[(size_t)j * n + d] = src[j][L.cell_of_dev[d]];
    });
    for (int j = 0; j < 5; ++j)
        for (int k = nC; k < n; ++k) L.q[(size_t)j * n + k] = src[j][k];
    L.dev_of_cell = std::move(dcell);
    L.dev_of_node = std::move(dnode);
    return "";
}

}  // namespace mfs
