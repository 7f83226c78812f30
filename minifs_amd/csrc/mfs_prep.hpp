// Host-side construction of the device layout from a preprocessed mesh view.
//
// Every per-cell or per-node sum of the reference is a face-ordered (or
// cell-ordered) serial accumulation.  The device kernels gather instead of
// scatter, so this layout stores, for each cell and each node, its
// contributions in exactly the order the reference's serial loops add them;
// a gather that walks these lists in order performs the same floating-point
// additions in the same order as the reference's scatter.
//
// Storage order on the device is free as long as that order of operations
// is kept.  Cells are stored in the order of the forward LU-SGS schedule
// (DAG level, then mesh id), so the cells of a sweep chunk are contiguous;
// faces and nodes are stored in first-touch order of that cell traversal.  Everything that depends on mesh numbering (per-cell face
// order, the sweep direction test "neighbour id < cell id", the per-node
// summation order) is evaluated here on mesh ids and stored as lists or
// masks.
#pragma once
#include <cstdint>
#include <string>
#include <memory>
#include <type_traits>
#include <utility>
#include <vector>

#include "../../include/mfs.h"

namespace mfs {

// Allocator whose resize() leaves new elements default-initialised (no
// zero fill): the layout's large arrays are then first touched by the
// threads that fill them, not by one thread's memset.
template <typename T>
struct NoFillAlloc : std::allocator<T> {
    template <typename U>
    struct rebind {
        using other = NoFillAlloc<U>;
    };
    NoFillAlloc() = default;
    template <typename U>
    NoFillAlloc(const NoFillAlloc<U>&) noexcept {}
    template <typename U>
    void construct(U* p) noexcept(std::is_nothrow_default_constructible<U>::value) {
        ::new (static_cast<void*>(p)) U;
    }
    template <typename U, typename... Args>
    void construct(U* p, Args&&... args) {
        ::new (static_cast<void*>(p)) U(std::forward<Args>(args)...);
    }
};
template <typename T>
using lvec = std::vector<T, NoFillAlloc<T>>;

// One direction's sweep schedule.  A chunk is the cells one wave takes at a
// time: consecutive device cells of one (tile, level) group with at most 64
// dependencies among them, at most 64 cells (kThinCells on a thin level).
// A dependency is a face whose neighbour this direction reads: forward the
// interior neighbours with a smaller mesh id, backward those with a larger
// one and the ghosts.  The dependencies of a chunk are stored together,
// cell by cell in the cell's ascending face order, so each lane of the wave
// takes one; 64/2 cells per wave on average, where one lane per face slot
// held 16 cells and left half the lanes idle (8 and two thirds on meshes
// with up to 6 faces per cell).
struct SweepLayout {
    int nchunk = 0;
    size_t ndep = 0;
    int tail = 0;                       // chunks of the thin tail (forward: the last, backward: the first)
    // per position of the sweep's order {first device cell, cells |
    // dependencies << 8 | kThinChunkFlag, first dependency, the dependency
    // expected to be published last (device cell, -1: none; on levels of at
    // most kDirectLevelChunks the one that this dependency itself waits for
    // last)}
    lvec<int> crec;
    lvec<int> batch_wait;               // the last of these for a batch (kBatchDirectLevelChunks)
    lvec<int> tile_chunk;               // ntile+1: first entry of each tile in pos
    lvec<int> pos;                      // positions by tile, in the sweep's level order within the tile
};

struct HostLayout {
    int nC = 0, nF = 0, nB = 0, nN = 0;
    // cells in device order; cell_of_dev[d] = mesh cell id (ghost k stays at nC+k)
    lvec<int> cell_of_dev;
    std::vector<int> dev_of_cell, dev_of_node;  // the inverse maps
    int dev_cell0 = 0;                         // device id of mesh cell 0
    // per device cell: bits 0-7 forward dependency slots (interior neighbour
    // with a smaller mesh id), bits 8-15 backward slots (neighbour with a
    // larger mesh id, ghosts included), bits 16-23 backward slots whose
    // neighbour is an interior cell, bits 24-31 boundary slots whose face
    // value in the gradient is the cell/ghost average (not SYMM/INTERFACE)
    lvec<int> depmask;
    // faces, in device order; face_of_dev[d] = mesh face id
    lvec<int> face_of_dev;
    lvec<int> c1, c2;                   // nF, device cell ids (c2 = nC+k for boundary face k)
    lvec<double> fgeo;                  // 4*nF: xfn, yfn, zfn, area
    lvec<double> dn1, dn2;              // nF: |(x_fc - x_cc) . n| for each side
    lvec<int> fno, fn;                  // face->node CSR in device node ids
    lvec<int> btype;                    // nB, by boundary face (ghost) index k
    // cells: device face ids in ascending mesh face id (CalC2F,
    // grid_polyhedra_auxiliary_functions.cpp:1345-1399)
    lvec<int> cfo, cf;                  // nC+1, sum nFPC
    lvec<double> vol;                   // nC
    int max_faces = 0;
    // nodes, in device order; node_of_dev[d] = mesh node id
    lvec<int> node_of_dev;
    // node values (CompNodeVar3D_dist): per device node, ordered entries
    // value = q[a] (b < 0) or 0.5*(q[a]+q[b]) (b >= 0, boundary face average)
    lvec<int> nlo;                      // nN+1
    lvec<int> nla, nlb;                 // entries
    lvec<double> nlw;                   // entry weights
    lvec<double> nden;                  // nN: WeightNode + TINY
    lvec<int> sym_node;                 // device nodes with nodesymm == 1
    lvec<double> sym_n;                 // 3 per symmetry node (xfn_n_symm, ...)
    // LU-SGS sweeps: forward DAG level of each mesh cell, the number of
    // levels, and each direction's chunks
    lvec<int> flevel;                   // nC, by mesh id
    int nlev = 0;
    int lpc = 4;                        // slots per cell of the slot tables (4 for tetrahedra, otherwise 8)
    lvec<int> cfs;                      // lpc slots per device cell: device face id or -1
    SweepLayout sweep[2];               // forward, backward
    // per device cell, forward then backward: its first dependency within its
    // chunk's (bits 0-7) and its dependency count (bits 8-15)
    lvec<unsigned short> cdep;          // 2*nC
    // the thin tail of the sweep order: the run of thin levels that ends it,
    // counted in the level-width unit below, and its cells
    int tail_chunks = 0, tail_cells = 0, thin_levels = 0;  // thin_levels: also where every level is thin
    bool all_thin = false;              // every level is thin
    int narrow_chunks = 0, narrow_cells = 0;  // the same tail with levels of at most kThinLevelChunks groups
    bool tri_slots = false;                    // tetrahedra with triangular slots only
    // initial state, 5 blocks of nC+nB, device cell order
    lvec<double> q;
};

// Cells per storage tile of the device order (the sweeps' workgroup unit).
constexpr int kDefaultTileCells = 4096;
// Thin levels.  A level's width is counted in groups of 64/lpc cells per
// tile; levels of at most kThinLevelChunks groups are thin (on meshes of 8
// slots per cell kWideThinLevelChunks, below).  A thin chunk
// holds at most kThinCells cells, so that each of its 5-value results has a
// lane of its own.
constexpr int kThinLevelChunks = 64;
constexpr int kThinCells = 12;
// With 8 slots per cell a group has 8 cells, half of a tetrahedral mesh's, so
// the same 1,024 cells of a level are 128 groups: 86 thin chunks, one for
// each of the 128 waves that sweep the tail.  ms per iteration with 64 and
// with 128 groups, FP64: 8k hexahedra 0.163 -> 0.142 (every level is thin
// then), 10.6k 0.183 -> 0.159, 16k 0.200 -> 0.196, 33k 0.260 -> 0.248, 262k
// 0.593 -> 0.583, 1M 1.206 -> 1.179; prisms 8.2k on a shallow order 0.148 ->
// 0.128, 11k 0.174 -> 0.150, 16k 0.195 -> 0.191; mixed 195k 0.432 -> 0.418.
// Smaller meshes have only thin levels with either.  Batches, whose waits do
// not use the line, change by less than 1% (8 solves of hexahedra 0.924 ->
// 0.921, of prisms 1.205 -> 1.212).  Tetrahedra gained nothing from 128: 20k,
// 94k and 384k cells all within 0.2%.
constexpr int kWideThinLevelChunks = 128;
// On levels of at most this many groups a wave waits on a dependency one
// level further back and then polls its own at once (SweepLayout::crec); on
// wider ones it waits on its latest dependency with one load, since there the
// waves that poll are many.  Measured, ms per iteration for 64 / 256 / 1024 /
// 2048: 262k hexahedra FP64 0.653 / 0.640 / 0.630 / 0.630, 195k prisms mixed
// 0.456 / 0.445 / 0.440 / 0.437, 1.3M tetrahedra FP64 0.963 / 0.955 / 0.947 /
// 0.951, 6.0M 2.90 / 2.88 / 2.86 / 2.87.  A batch interleaves its solves'
// levels, so more waves poll at once there and the line lies lower (12 mixed
// solves of 2.3M cells: 1.236 with 0, then 1.167 / 1.175 / 1.190 / 1.198).
constexpr int kDirectLevelChunks = 1024, kBatchDirectLevelChunks = 64;
constexpr int kMinTailChunks = 256;  // shorter tails stay with the wide levels
constexpr int kThinChunkFlag = 0x10000;

// A device cell's latest dependency in one direction: its device cell and its
// rank, 2 * its depth (the levels before its own in the sweep's order, plus
// one in the backward sweep) + 1 for another tile's; the first of equal rank
// in the cell's face order, -1 without one.
struct LatestDep {
    int rank, cell;
};
// What the sweeps' progress rests on: each direction's chunks cover the cells
// once, in the order of their depth, in the tile schedule too, and every
// dependency is less deep than its cell.  Returns "" where that holds.
std::string check_sweep_order(const HostLayout& L, int dir, const lvec<LatestDep>& latest);

// Returns "" on success.
std::string build_layout(const mfs_mesh_view& v, HostLayout& L, int tile_cells = kDefaultTileCells);

}  // namespace mfs
