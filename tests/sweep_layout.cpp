// Checks of the sweeps' tables (SweepLayout, minifs_amd/csrc/mfs_prep.hpp)
// against the mesh, from their definitions.  Built and run by
// test_sweep_layout.py; one argument list per mesh:
//   sweep_layout cells nx ny nz nb_parts part_size tile_cells [spoil direction]
// prints "ok", or what is wrong.  With `spoil` the order is made wrong in one
// place and the library's own check of it is printed.
#include <cstdio>
#include <cstdlib>
#include <string>
#include <vector>

#include "mfs_prep.hpp"

namespace {

struct Mesh {
    mfs_grid* g = nullptr;
    mfs_mesh_view v{};
    mfs::HostLayout L;
    std::string error;
    Mesh(char** a) {
        mfs_params p;
        mfs_params_default(&p);
        p.mach = 0.8;
        if (mfs_params_derive(&p) || mfs_grid_generate_box(atoi(a[1]), atoi(a[2]), atoi(a[3]), atoi(a[0]), 0.1, 0.1, 0.15, 7, &g) ||
            mfs_grid_decouple_ex(g, atoi(a[4]), atoi(a[5])) || mfs_grid_preprocess(g, &p) || mfs_grid_view(g, &v))
            error = mfs_last_error();
        else
            error = mfs::build_layout(v, L, atoi(a[6]));
    }
    ~Mesh() { mfs_grid_destroy(g); }
};

#define NEED(x)                                                                                     \
    do {                                                                                            \
        if (!(x)) return std::string("direction ") + (dir ? "backward" : "forward") + ": " + #x;    \
    } while (0)

// Everything that the tables of one direction promise.
std::string check(const mfs::HostLayout& L, int dir, int tile_cells) {
    const mfs::SweepLayout& S = L.sweep[dir];
    const int nC = L.nC;
    auto other = [&](int d, int f) { return L.c1[f] == d ? L.c2[f] : L.c1[f]; };
    auto tile = [&](int d) { return L.cell_of_dev[d] / tile_cells; };
    auto level = [&](int d) { return L.flevel[L.cell_of_dev[d]]; };
    // a cell's dependencies in its face order (ghosts too in the backward sweep)
    auto deps = [&](int d) {
        std::vector<int> out;
        for (int k = L.cfo[d]; k < L.cfo[d + 1]; ++k) {
            const int nb = other(d, L.cf[k]);
            const bool lower = nb < nC && L.cell_of_dev[nb] < L.cell_of_dev[d];
            if (dir == 0 ? lower : !lower) out.push_back(nb);
        }
        return out;
    };
    NEED((int)S.pos.size() == S.nchunk && (int)S.crec.size() == 4 * S.nchunk && (int)S.batch_wait.size() == S.nchunk);
    const int unit = 64 / L.lpc;
    std::vector<int> width(L.nlev, 0), at(nC, -1);
    for (int d = 0, first = 0; d <= nC; ++d)
        if (d == nC || (d > first && (level(d) != level(first) || tile(d) != tile(first)))) {
            if (d > first) width[level(first)] += (d - first + unit - 1) / unit;
            first = d;
        }
    size_t nd = 0;
    int before = dir == 0 ? -1 : L.nlev;
    for (int u = 0; u < S.nchunk; ++u) {
        const int d0 = S.crec[4 * u], cells = S.crec[4 * u + 1] & 0xff, nk = (S.crec[4 * u + 1] >> 8) & 0xff;
        NEED(cells >= 1 && cells <= 64 && nk <= 64 && d0 >= 0 && d0 + cells <= nC);
        const bool thin = width[level(d0)] <= (L.lpc == 8 ? mfs::kWideThinLevelChunks : mfs::kThinLevelChunks);
        NEED(thin == ((S.crec[4 * u + 1] & mfs::kThinChunkFlag) != 0) && (!thin || cells <= mfs::kThinCells));
        NEED((size_t)S.crec[4 * u + 2] == nd);
        NEED(dir == 0 ? level(d0) >= before : level(d0) <= before);
        before = level(d0);
        int start = 0;
        for (int d = d0; d < d0 + cells; ++d) {
            NEED(at[d] < 0);
            at[d] = u;
            NEED(level(d) == level(d0) && tile(d) == tile(d0));
            const int n = (int)deps(d).size();
            NEED(L.cdep[2 * (size_t)d + dir] == (unsigned short)(start | (n << 8)));
            start += n;
        }
        NEED(start == nk);
        nd += nk;
    }
    NEED(nd == S.ndep);
    // the dependency of the latest level, another tile's first, the first of
    // equal rank
    auto latest = [&](int d0, int cells) {
        long long best = -1;
        int rep = -1;
        for (int d = d0; d < d0 + cells; ++d)
            for (int nb : deps(d)) {
                if (nb >= nC) continue;
                const long long r = 2LL * (dir == 0 ? level(nb) : L.nlev - level(nb)) + (tile(nb) != tile(d));
                if (r > best) {
                    best = r;
                    rep = nb;
                }
            }
        return rep;
    };
    for (int u = 0; u < S.nchunk; ++u) {
        const int d0 = S.crec[4 * u], cells = S.crec[4 * u + 1] & 0xff;
        for (int d = d0; d < d0 + cells; ++d)
            for (int nb : deps(d)) NEED(nb >= nC || at[nb] < u);
        const int rep = latest(d0, cells), further = rep < 0 ? -1 : latest(rep, 1);
        NEED(S.crec[4 * u + 3] == (width[level(d0)] <= mfs::kDirectLevelChunks ? further : rep));
        NEED(S.batch_wait[u] == (width[level(d0)] <= mfs::kBatchDirectLevelChunks ? further : rep));
    }
    // the tile schedule: each tile's chunks in the sweep's order, every
    // dependency in an earlier tile (in the sweep's order) or before it
    NEED(S.tile_chunk.front() == 0 && S.tile_chunk.back() == S.nchunk);
    for (size_t t = 0; t + 1 < S.tile_chunk.size(); ++t)
        for (int i = S.tile_chunk[t]; i < S.tile_chunk[t + 1]; ++i) {
            NEED(tile(S.crec[4 * (size_t)S.pos[i]]) == (int)t);
            NEED(i == S.tile_chunk[t] || S.pos[i] > S.pos[i - 1]);
        }
    for (int d = 0; d < nC; ++d) {
        NEED(at[d] >= 0);
        for (int nb : deps(d)) NEED(nb >= nC || (dir == 0 ? tile(nb) <= tile(d) : tile(nb) >= tile(d)));
    }
    return "";
}

// The latest dependencies of every cell, as check_sweep_order takes them.
mfs::lvec<mfs::LatestDep> latest_of(const mfs::HostLayout& L, int dir, int tile_cells) {
    mfs::lvec<mfs::LatestDep> out(L.nC);
    for (int d = 0; d < L.nC; ++d) {
        out[d] = {-1, -1};
        const int c = L.cell_of_dev[d];
        for (int k = L.cfo[d]; k < L.cfo[d + 1]; ++k) {
            const int f = L.cf[k], nb = L.c1[f] == d ? L.c2[f] : L.c1[f];
            if (nb >= L.nC) continue;
            const int m = L.cell_of_dev[nb], l = L.flevel[m];
            const int r = 2 * (dir == 0 ? l : L.nlev - l) + (m / tile_cells != c / tile_cells ? 1 : 0);
            if ((dir == 0 ? m < c : m > c) && r > out[d].rank) out[d] = {r, nb};
        }
    }
    return out;
}

std::string spoiled(mfs::HostLayout& L, const std::string& how, int dir, int tile_cells) {
    mfs::SweepLayout& S = L.sweep[dir];
    mfs::lvec<mfs::LatestDep> latest = latest_of(L, dir, tile_cells);
    const std::string before = mfs::check_sweep_order(L, dir, latest);
    if (!before.empty()) return "wrong before: " + before;
    const int mid = S.nchunk / 2;
    if (how == "dependency")  // a cell that waits for one of its own level
        latest[S.crec[4 * mid]].rank = 2 * (dir == 0 ? L.flevel[L.cell_of_dev[S.crec[4 * mid]]]
                                                     : L.nlev - L.flevel[L.cell_of_dev[S.crec[4 * mid]]]);
    if (how == "level")  // a cell of another level among a chunk's
        L.flevel[L.cell_of_dev[S.crec[4 * mid]]] += 1;
    if (how == "order") {  // the first and the last chunk change places
        for (int k = 0; k < 4; ++k) std::swap(S.crec[k], S.crec[4 * (S.nchunk - 1) + k]);
        for (int& u : S.pos) u = u == 0 ? S.nchunk - 1 : u == S.nchunk - 1 ? 0 : u;
    }
    if (how == "cells") S.crec[4 * mid + 1] += 1;  // a cell in two chunks
    if (how == "position") S.pos[mid] = S.pos[mid - 1];  // a chunk twice, another never
    return mfs::check_sweep_order(L, dir, latest);
}

}  // namespace

int main(int argc, char** argv) {
    if (argc != 8 && argc != 10) return 2;
    Mesh m(argv + 1);
    std::string e = m.error;
    if (argc == 10 && e.empty()) e = spoiled(m.L, argv[8], atoi(argv[9]), atoi(argv[7]));
    if (argc == 10) {
        puts(e.c_str());
        return 0;
    }
    for (int dir = 0; dir < 2 && e.empty(); ++dir) e = check(m.L, dir, atoi(argv[7]));
    puts(e.empty() ? "ok" : e.c_str());
    return e.empty() ? 0 : 1;
}
