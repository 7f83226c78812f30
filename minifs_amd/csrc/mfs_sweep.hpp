// LU-SGS sweeps (SolveLUSGS3D, src/Kernels/forward_lusgs.cpp:803-1249) on
// the GPU, included by mfs_device.hip inside namespace mfs::dev.
//
// With LUSGSLayer[i] = i (ReorderCellforLUSGS_0, grid_polyhedra.cpp:1127-1142)
// the forward sweep of cell c reads the final DQ of its lower-numbered face
// neighbours and the backward sweep that of its higher-numbered neighbours
// and of its ghost cells (DQ = 0).
//
// Work decomposition: a wave handles one chunk of cells of the same forward
// DAG level (contiguous in device order) with at most 64 dependencies, one
// lane per dependency: a face whose neighbour this sweep reads.  Each lane
// evaluates FluxLUSGS3D for its own face and leaves the product in LDS; then
// each cell has one lane, which adds its cell's products in the cell's face
// order, exactly as the serial sweep forms the sum, and runs the limiter and
// the update.  A cell has two dependencies per sweep on average, so a chunk
// holds about 30 cells.
// Bound: the wide levels by the latency of a chunk's rounds of loads and by
// the memory system's gathers, so what counts is cells per round.  With one
// lane per face slot (16 cells per wave, 8 on meshes with up to 6 faces per
// cell) half the lanes had no dependency and every cell's lanes ran the
// limiter and the update.  Wide-level launches, forward / backward, with one
// lane per face slot and now: 6.0M tetrahedra FP64 808 / 938 -> 650 / 745 us,
// 262k hexahedra FP64 190 / 203 -> 111 / 112 us (fewer levels are wide), a
// mixed batch of 2.3M cells, whose sweeps are one launch each, 603 / 686 ->
// 384 / 487 us.
//
// Schedule: cells are stored by tile (4096 consecutive mesh ids, a compact
// region in TDTree numbering), then forward level; a chunk is as many cells
// of one (tile, level) group as have 64 dependencies together, so its cells
// never depend on one another.  Two schedules, both on a grid sized to be resident at once:
//   flat (default): the chunks in forward level order, the backward sweep's
//     by level from the end; the steps go to the ticket groups in
//     runs of 2^run_shift consecutive steps, run k to group k mod ngroups,
//     and a free wave of the group takes the group's next step from the
//     group's counter, so waves that finish early take more chunks and no
//     wave's delay holds back the chunks after it.  A group's workgroups
//     share an XCD, so a run's chunks (neighbours in one tile and level,
//     whose rows share cache lines) meet in one L2.
//   tiles: a workgroup of W waves owns a tile, wave w taking the tile's
//     chunks w, w+W, ... in level order; tiles go to workgroups
//     round-robin, each workgroup walking its tiles in sweep order.
// In both, every dependency of a chunk comes earlier in the sweep order and
// each wave takes its chunks in that order, so the first unfinished chunk
// is always being worked on with its dependencies finished, or is the next
// ticket of a group whose waves are all free: the sweep cannot deadlock
// while every wave of the grid is resident.  (On 6M cells the flat
// schedule measured 2x faster: dependencies inside a tile cost the same
// device-coherent hop as across tiles, and a workgroup held by one tile
// delays its next.)
//
// Publication: before a sweep every DQ slot it writes holds a NaN payload
// (the sentinel) that arithmetic never produces.  A cell writes its 5 final
// DQ values with device-coherent stores; a dependent cell reads them with
// device-coherent loads and retries while any is the sentinel (each store
// is single-copy atomic, so a non-sentinel value is final).  One lane per
// wave first waits on the chunk's latest dependency (rep), which keeps the
// polling traffic to one load per wave; on narrow levels it waits on that
// dependency's own latest one, so that the wave's lanes are polling when
// their dependencies come, which saves a round trip on the level's critical
// path.  The forward sweep re-arms the
// backward array and the backward sweep the forward one.
//
// Precision: R is the type of the implicit operator (state snapshot,
// geometry, Diag, DQ).  With R = double the sweeps are the reference's
// arithmetic bit for bit.  With R = float (mixed precision) the operator
// runs in FP32 while the right-hand side (the FP64 residual) and the state
// update stay FP64, so the iteration is a defect correction whose fixed
// point is the FP64 solution.

constexpr int kMaxFaces = 6;  // tetrahedra, pyramids, prisms, hexahedra

constexpr unsigned long long kSentinel = Real<double>::kSent;

template <typename R>
__device__ __forceinline__ typename Real<R>::bits ld_dev(const R* p) {
    using B = typename Real<R>::bits;
    return __hip_atomic_load(reinterpret_cast<B*>(const_cast<R*>(p)), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
template <typename R>
__device__ __forceinline__ void st_dev(R* p, R v) {
    using B = typename Real<R>::bits;
    __hip_atomic_store(reinterpret_cast<B*>(p), __builtin_bit_cast(B, v), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
// The same for readers on this XCD only: the store stops at the XCD's L2,
// where the device-scope loads of its other CUs find it.
// This is an assumption about gfx950 and not the language's memory model, in
// which a workgroup-scope store and another workgroup's device-scope load are
// a race: (1) a CU's vector cache writes every store through to its XCD's L2,
// (2) a device-scope load misses the CU's cache and goes to that L2, which
// cannot pass over a line that it holds modified, (3) XCC_ID names the L2.
// Where it did not hold, a reader would go on seeing the sentinel: a word is 8
// or 4 aligned bytes, written once between two launches, and whatever an
// earlier launch left is the sentinel.  So the bounded wait would end with the
// error of a sweep that cannot go on, never with another value.  Readers in
// later launches see the stores as they see any other kernel's.
#if defined(__HIP_DEVICE_COMPILE__) && !defined(__gfx950__)
#error "st_xcd relies on the caches of gfx950"
#endif
template <typename R>
__device__ __forceinline__ void st_xcd(R* p, R v) {
    using B = typename Real<R>::bits;
    __hip_atomic_store(reinterpret_cast<B*>(p), __builtin_bit_cast(B, v), __ATOMIC_RELAXED,
                       __HIP_MEMORY_SCOPE_WORKGROUP);
}
__device__ __forceinline__ int xcd_id() {  // HW_REG_XCC_ID, bits 0-3
    return (int)__builtin_amdgcn_s_getreg(20 | (0 << 6) | ((4 - 1) << 11));
}

// The next ticket of a counter, taken by lane 0 (0 in the others).  The
// address is kept in vector registers: for an address that the compiler
// knows to be uniform it combines the wave's atomics and broadcasts the
// result at once, which waits for the atomic's round trip.  A wave's loads
// and atomics return in the order of issue, so a chunk takes its wave's next
// ticket after its last load of the first rounds: nothing that it waits for
// then queues behind the atomic except a late dependency.
__device__ __forceinline__ int take_ticket(int* ctr) {
    auto p = (__attribute__((address_space(1))) int*)ctr;
    asm volatile("" : "+v"(p));
    int t = 0;
    if ((threadIdx.x & 63) == 0) t = __hip_atomic_fetch_add(p, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    return t;
}

// 5-value records read with 128-bit buffer loads: 3 loads for a 40-byte
// record, 2 for a 20-byte one, where per-value loads take 5.  The sweeps
// read their dependencies' published DQ this way: those loads bypass the
// CU's cache, so each of them is a request to the memory system (the
// plain loads of a chunk's own and its neighbours' records hit the CU's
// cache after the first and gain nothing from it).  Buffer offsets are
// 32-bit, so the sweeps take this path only while the state arrays are
// below 2 GiB (wide_records).
constexpr int kBufferDword3 = 0x00020000;  // raw buffer resource: byte-addressed, no format
constexpr int kLoadDevice = 16;            // the cache policy of ld_dev (device-coherent, sc1)
__device__ __forceinline__ bool wide_records(int nq) { return (size_t)nq * 5 * sizeof(double) <= 0x7fffffffu; }

template <int AUX, typename T>
__device__ __forceinline__ void ld5w(const T* base, int nrec, int i, T (&v)[5]) {
    const __amdgpu_buffer_rsrc_t r =
        __builtin_amdgcn_make_buffer_rsrc(const_cast<T*>(base), 0, nrec * 5 * (int)sizeof(T), kBufferDword3);
    const int off = i * 5 * (int)sizeof(T);
    if constexpr (sizeof(T) == 8) {
        const auto a = __builtin_amdgcn_raw_buffer_load_b128(r, off, 0, AUX);
        const auto b = __builtin_amdgcn_raw_buffer_load_b128(r, off + 16, 0, AUX);
        const auto c = __builtin_amdgcn_raw_buffer_load_b64(r, off + 32, 0, AUX);
        const unsigned w[10] = {a[0], a[1], a[2], a[3], b[0], b[1], b[2], b[3], c[0], c[1]};
#pragma unroll
        for (int j = 0; j < 5; ++j)
            v[j] = __builtin_bit_cast(T, ((unsigned long long)w[2 * j + 1] << 32) | w[2 * j]);
    } else {
        // the words go through plain integers: a bit_cast straight from an
        // element of the returned vector compiled to element 0 repeated
        const auto a = __builtin_amdgcn_raw_buffer_load_b128(r, off, 0, AUX);
        const unsigned b = __builtin_amdgcn_raw_buffer_load_b32(r, off + 16, 0, AUX);
        const unsigned w[5] = {a[0], a[1], a[2], a[3], b};
#pragma unroll
        for (int j = 0; j < 5; ++j) v[j] = __builtin_bit_cast(T, w[j]);
    }
}
// Record i of `base` (nrec records) as published by another wave.  Each of
// its values is read whole (8 or 4 aligned bytes), so a value other than the
// sentinel is final.  The wide path is not an atomic to the compiler: a wait
// loop puts a memory barrier for the compiler between its turns.
template <typename T>
__device__ __forceinline__ void read_published(bool wide, const T* base, int nrec, int i, T (&v)[5]) {
    if (wide) {
        ld5w<kLoadDevice>(base, nrec, i, v);
    } else {
#pragma unroll
        for (int j = 0; j < 5; ++j) v[j] = __builtin_bit_cast(T, ld_dev<T>(base + (size_t)i * 5 + j));
    }
}

// True when another wave has already given up (checked every 4096 spins),
// so that one expired wait ends the whole sweep quickly.
__device__ __forceinline__ bool wait_failed(int* err, unsigned spins) {
    if ((spins & 4095u) != 0) return false;
    return __shfl(__hip_atomic_load(err, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT), 0, 64) != 0;
}

// One direction's schedule and tables (SweepLayout in mfs_prep.hpp).
template <typename R>
struct SweepDir {
    const int4* crec;                       // per position: first cell, cells | deps << 8 | flag, first dep, wait
    const int* batch_wait;                  // per position: the dependency a batch waits on
    const int* dnb;                         // per dependency: the neighbour
    const typename Real<R>::vec4* dgeo;     // per dependency: normal away from the cell + area
    const int* tile_chunk;                  // tiles schedule: first entry of each tile in pos
    const int* pos;                         // tiles schedule: positions, tile by tile
};

template <typename R>
struct SweepArgs {
    int nC;
    int nq;                                 // records of the state arrays: interior and ghost cells
    int ntiles;
    SweepDir<R> dir[2];                     // forward, backward
    const unsigned short* cdep;             // per cell and direction: first dependency in the chunk, count
    const R* q;                             // operator state (cell-major, 5 per cell)
    const double* q64;                      // FP64 state the backward sweep updates
    const double* res;                      // forward: initial DQ (FP64 residual)
    const R* diag;
    R* dqf;                                 // forward DQ, 5 per cell
    R* dqb;                                 // backward (final) DQ, 5 per cell incl. ghosts (0)
    double* qout;                           // backward: updated state
    int cell0;                              // cell with mesh id 0 (forward: divide only)
    int* err;
    int* tickets;                           // this sweep's ticket counters (flat schedule)
    int* tickets_next;                      // the other direction's, zeroed here for its next sweep
    int ngroups;                            // ticket groups in use (<= kTicketGroups and <= workgroups)
    // flat schedule: this launch walks positions [ubeg, uend) of the sweep's
    // order; a sweep split in two launches runs its wide levels and its thin
    // tail apart, each launch ending when all its chunks are done
    int ubeg, uend;
    // flat schedule: the positions go to the ticket groups in runs of
    // 2^run_shift consecutive ones (run k to group k mod ngroups)
    int run_shift;
};

// This wave's words of LDS: the dependencies' products (5 x 64 values), then
// the chunk's records (64 cells of 5 values).  A wave's LDS accesses complete
// in order; lds_order keeps the compiler from moving them across each other.
// A launch gives every wave of a workgroup kStageWords doubles.
constexpr int kStageWords = 5 * 64;
inline size_t stage_bytes(int waves) { return (size_t)waves * kStageWords * sizeof(double); }
__device__ __forceinline__ double* stage_words() {
    extern __shared__ double mfs_stage[];
    return mfs_stage + (threadIdx.x / 64) * kStageWords;
}
__device__ __forceinline__ void lds_order() {
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
}

// The part of the face term that does not depend on the neighbour's DQ:
// the reference's FluxLUSGS3D split in two (FP64), or its increment form
// (FP32 operator of mixed precision).
template <typename R>
using FacePre = std::conditional_t<sizeof(R) == sizeof(double), FluxPre<R>, FluxDeltaPre<R>>;

// v[j] by selects (an array indexed at run time would go to scratch memory).
template <typename R>
__device__ __forceinline__ R pick5(R v0, R v1, R v2, R v3, R v4, int j) {
    const R a = j == 1 ? v1 : v0, b = j == 3 ? v3 : v2;
    const R x = j < 2 ? a : b;
    return j == 4 ? v4 : x;
}

// The room that value v has inside (lo, hi), and zero where it has none
// beyond the rounding of sums of its size.
template <typename R>
__device__ __forceinline__ R min_room(R v, R lo, R hi) {
    const R a = v - lo, b = hi - v;
    const R m = a < b ? a : b;
    const R size = __builtin_fabs(v) + __builtin_fabs(lo) + __builtin_fabs(hi);
    return m > size * (sizeof(R) == 8 ? R(1e-9) : R(1e-3)) ? m : R(0);
}

// The limiter's three stages for the wave's cells; `x` is scaled with DQ.  A
// cell outside the limits is rare, and where the first stage scales no cell
// of the wave the others see the same values again, so they are left out.
template <typename R>
__device__ __forceinline__ void limit_dq(bool skip, const R (&q)[5], R (&DQ)[5], R& x, R gamm1, R rho_min, R rho_max,
                                         R p_min, R p_max) {
    const R vv = q[1] * q[1] + q[2] * q[2] + q[3] * q[3];
#pragma unroll 1
    for (int stage = 0; stage < 3; ++stage) {
        const bool bad = !skip & dq_outside(q, DQ, vv, gamm1, rho_min, rho_max, p_min, p_max);
        if (__builtin_amdgcn_ballot_w64(bad) == 0) return;
        if (bad) {
#pragma unroll
            for (int j = 0; j < 5; ++j) DQ[j] = stage < 2 ? DQ[j] * R(0.1) : R(0.0);
            x = stage < 2 ? x * R(0.1) : R(0.0);
        }
    }
}

// What a launch's chunks are: all treated as wide, all thin (the thin tail),
// each by its flag, or a batch's (wide, with waits of their own).
constexpr int kWideChunks = 0, kThinChunks = 1, kAnyChunks = 2, kBatchChunks = 3;

// A record that no kernel writes, at an index that every lane shares: read
// through the scalar cache.
__device__ __forceinline__ int load_record(const int* p, int u) {
    return ((const __attribute__((address_space(4))) int*)p)[u];
}
__device__ __forceinline__ int4 load_record(const int4* p, int u) {
    typedef int v4i __attribute__((ext_vector_type(4)));
    const v4i r = ((const __attribute__((address_space(4))) v4i*)p)[u];
    return make_int4(r[0], r[1], r[2], r[3]);
}

// The chunk at position u (the same in every lane) of a sweep's order.
// Returns false when a wait expired (the error word is set).
//
// Latency: a chunk's operands come in three rounds of loads: its record;
// then the latest dependency's first value (lane 0, requested first), the
// dependencies' neighbours and geometry, the cells' state, Diag and
// right-hand side; then the neighbours' states together with their DQ when
// the latest dependency was already published.  The DQ-independent half of
// every face term is evaluated before waiting, so only the DQ-dependent
// half, the sum, the limiter and the stores follow the dependency's arrival.
// With a ticket counter, `next` receives the wave's next ticket.
//
// On a thin level the chunk has at most 12 cells and its 5-value
// results one lane each: lane 5k + j sums, divides and stores value j of
// cell k, so that one subtraction chain, one division and one store stand
// where a lane per cell would run five of each on the level's critical path.
template <bool FWD, int MAXD, typename R, int KIND>
__device__ __forceinline__ bool sweep_chunk(const SweepArgs<R>& A, const FlowConst& K, int u, int* ctr, int& next) {
    using B = typename Real<R>::bits;
    constexpr B kSent = Real<R>::kSent;
    const SweepDir<R>& S = A.dir[FWD ? 0 : 1];
    const int lane = (int)threadIdx.x & 63;
    R* const poll = FWD ? A.dqf : A.dqb;
    const int4 rec = load_record(S.crec, u);
    const int c0 = rec.x, nc = rec.y & 0xff, nd = (rec.y >> 8) & 0xff;
    const int rep = KIND == kBatchChunks ? load_record(S.batch_wait, u) : rec.w;
    // a thin level: every lane polls its own dependency (a batch interleaves
    // many solves, so no level of one solve is thin there)
    const bool thin = KIND == kThinChunks || (KIND == kAnyChunks && (rec.y & kThinChunkFlag) != 0);
    B rv = 0;
    if (lane == 0 && rep >= 0) rv = ld_dev<R>(poll + (size_t)rep * 5);
    // this lane's dependency
    const bool mine = lane < nd;
    const size_t kd = (size_t)rec.z + (mine ? lane : 0);
    const int nb = S.dnb[kd];
    const typename Real<R>::vec4 g = S.dgeo[kd];
    bool pend = mine && (FWD || nb < A.nC);  // ghosts have DQ = 0
    // this lane's cell (thin: and value); lanes past the chunk's cells read
    // the first cell and store nothing
    const int k5 = thin ? lane / 5 : lane;
    const int j5 = lane - 5 * (lane / 5);
    const bool active = k5 < nc;
    const int c = c0 + (active ? k5 : 0);
    const unsigned cd = A.cdep[2 * (size_t)c + (FWD ? 0 : 1)];
    const int dep0 = (int)(cd & 0xffu), ndep = (int)(cd >> 8);
    R qc[5], D[5];
    load5r(A.q + (size_t)c * 5, qc);
    const R dg = A.diag[c];
    if (thin) {
        const size_t w = (size_t)c * 5 + j5;
        D[0] = FWD ? (R)A.res[w] : A.dqf[w];
    } else if (FWD) {
#pragma unroll
        for (int j = 0; j < 5; ++j) D[j] = (R)A.res[(size_t)c * 5 + j];
    } else {
        load5r(A.dqf + (size_t)c * 5, D);
    }
    // the FP64 state the backward sweep updates (mixed precision), fetched
    // before the wait so that no memory round trip follows the dependencies
    double q64c[5];
    if constexpr (!FWD && sizeof(R) != sizeof(double)) load5(A.q64 + (size_t)c * 5, q64c);
    bool rep_seen = (rep < 0) || (__shfl(rv, 0, 64) != kSent);
    R qnb[5] = {R(0), R(0), R(0), R(0), R(0)};
    R dv[5] = {R(0), R(0), R(0), R(0), R(0)};  // the neighbour's DQ (a ghost's stays 0)
    if (mine) load5r(A.q + (size_t)nb * 5, qnb);
    const bool wide = wide_records(A.nq);  // the same for every wave
    // one read of every pending dependency (they are interior cells); a
    // value still the sentinel leaves the lane pending
    auto settle = [&] {
        bool missing = false;
#pragma unroll
        for (int j = 0; j < 5; ++j) missing |= __builtin_bit_cast(B, dv[j]) == kSent;
        pend = missing;
    };
    // where the latest dependency is out, the others most likely are too:
    // their reads go out with the neighbours' states
    const bool early = rep_seen && pend;
    if (early) read_published(wide, static_cast<const R*>(poll), A.nC, nb, dv);
    if (ctr) next = take_ticket(ctr);
    FacePre<R> pre;
    if (mine) {
        if constexpr (sizeof(R) == sizeof(double))
            flux_lusgs_pre<R>(pre, qnb, g.x, g.y, g.z, (R)K.gam, (R)K.p_bar, (R)K.lhs_omga);
        else
            flux_lusgs_delta_pre<R>(pre, qnb, g.x, g.y, g.z, (R)K.gam, (R)K.p_bar, (R)K.lhs_omga);
    }

    if (early) settle();
    // Thin levels: bounds under which this lane's value cannot take its cell
    // near the limiter's limits.  With |DQ_0| at most half the room that rho
    // has, and each of the five terms of dp at most a 16th of the room that p
    // has, rho and p stay well inside; where there is no room beyond rounding
    // (a clamped state) no value counts as safe.
    R safe_r = R(-1), safe_p = R(-1), safe_w = R(0);
    if (thin) {
        const R mr = min_room(qc[0], (R)K.rho_min, (R)K.rho_max), mp = min_room(qc[4], (R)K.p_min, (R)K.p_max);
        const R vv = qc[1] * qc[1] + qc[2] * qc[2] + qc[3] * qc[3];
        const R w = pick5(R(0.5) * vv, qc[1], qc[2], qc[3], R(1), j5);
        safe_w = (R)K.gamm1 * __builtin_fabs(w);
        safe_r = j5 == 0 ? R(0.5) * mr : Real<R>::kMost;
        safe_p = R(0.0625) * mp;
        if (!((mr > R(0)) & (mp > R(0)))) safe_r = R(-1);
    }
    unsigned spins = 0;
    if (!rep_seen) {  // one lane waits for the chunk's latest dependency (narrow levels: for that one's own)
        while (true) {
            B v = 0;
            if (lane == 0) v = ld_dev<R>(poll + (size_t)rep * 5);
            v = __shfl(v, 0, 64);
            if (v != kSent) break;
            if (++spins > kSpinLimit || wait_failed(A.err, spins)) {
                if (lane == 0) atomicExch(A.err, 1);
                return false;
            }
            __builtin_amdgcn_s_sleep(2);
        }
    }
    // every lane reads its face's dependency and retries an unpublished one
    while (__ballot(pend) != 0) {
        if (pend) {
            asm volatile("" ::: "memory");  // the reads of this turn are not those of the last
            read_published(wide, static_cast<const R*>(poll), A.nC, nb, dv);
            settle();
        }
        if (__ballot(pend) == 0) break;
        if (++spins > kSpinLimit || wait_failed(A.err, spins)) {
            if (lane == 0) atomicExch(A.err, 1);
            return false;
        }
        if (KIND != kThinChunks) __builtin_amdgcn_s_sleep(1);
    }
    // this lane's face term: forward 0.5*A*F (DQ -= term), backward A*F (summed)
    R* const st = reinterpret_cast<R*>(stage_words());
    if (mine) {
        R fl[5];
        if constexpr (sizeof(R) == sizeof(double))  // the reference's expression, bit for bit
            flux_lusgs_post<R>(pre, dv, g.x, g.y, g.z, fl);
        else  // FP32 operator: the same function in increment form (no cancellation floor)
            flux_lusgs_delta_post<R>(pre, dv, g.x, g.y, g.z, fl);
        const R tmp = FWD ? R(0.5) * g.w : g.w;
#pragma unroll
        for (int j = 0; j < 5; ++j) st[j * 64 + lane] = tmp * fl[j];
    }
    lds_order();
    R* const own = FWD ? A.dqf : A.dqb;    // published
    R* const other = FWD ? A.dqb : A.dqf;  // re-armed for the next sweep
    const R sent = __builtin_bit_cast(R, kSent);
    const int nw = 5 * nc;  // words of the chunk's records
    const size_t w0 = (size_t)c0 * 5;
    if (thin) {
        R t[MAXD];
#pragma unroll
        for (int m = 0; m < MAXD; ++m) t[m] = st[j5 * 64 + ((dep0 + m) & 63)];
        R x = D[0], acc = R(0);
#pragma unroll
        for (int m = 0; m < MAXD; ++m)
            if (m < ndep) {
                if (FWD)
                    x -= t[m];
                else
                    acc += t[m];
            }
        if (FWD) {
            x /= dg;
        } else {
            const R tmp = R(2.0) * dg;
            x -= acc / tmp;
        }
        // The limiter needs the cell's five values, an exchange through LDS on
        // the level's critical path.  A value so small that no cell's limits
        // can be reached is known by its own lane (safe_r, safe_p below), so
        // the exchange is left to the rare chunk with a larger one; the
        // backward sweep's update makes it after publishing.
        const bool near = !((__builtin_fabs(x) <= safe_r) & (__builtin_fabs(x) * safe_w <= safe_p));
        bool have = false;
        auto exchange = [&] {
            lds_order();
            st[lane] = x;
            lds_order();
#pragma unroll
            for (int j = 0; j < 5; ++j) D[j] = st[5 * (lane / 5) + j];
            lds_order();
            have = true;
        };
        if (__builtin_amdgcn_ballot_w64(near) != 0) {
            exchange();
            limit_dq<R>(FWD && c == A.cell0, qc, D, x, (R)K.gamm1, (R)K.rho_min, (R)K.rho_max, (R)K.p_min,
                        (R)K.p_max);
        }
        if (lane < nw) {
            if (KIND == kThinChunks)
                st_xcd<R>(own + w0 + lane, x);
            else
                st_dev<R>(own + w0 + lane, x);
            other[w0 + lane] = sent;
        }
        if (!FWD && !have) exchange();
    } else {
        R acc[5] = {R(0), R(0), R(0), R(0), R(0)};
#pragma unroll
        for (int m = 0; m < MAXD; ++m) {
            R t[5];
#pragma unroll
            for (int j = 0; j < 5; ++j) t[j] = st[j * 64 + ((dep0 + m) & 63)];
            if (m < ndep) {
#pragma unroll
                for (int j = 0; j < 5; ++j) {
                    if (FWD)
                        D[j] -= t[j];
                    else
                        acc[j] += t[j];
                }
            }
        }
        if (FWD) {
#pragma unroll
            for (int j = 0; j < 5; ++j) D[j] /= dg;
        } else {
            const R tmp = R(2.0) * dg;
#pragma unroll
            for (int j = 0; j < 5; ++j) D[j] -= acc[j] / tmp;
        }
        R none = R(0);
        limit_dq<R>(FWD && c == A.cell0, qc, D, none, (R)K.gamm1, (R)K.rho_min, (R)K.rho_max, (R)K.p_min, (R)K.p_max);
        // Stores.  The chunk's cells are contiguous, so its 5-value records
        // form one run of words: lane w stores words w, w + 64, ..., and
        // every store instruction writes whole, consecutive words.  Stored
        // value by value from the cell's lane, a record's words would go out
        // as pieces of lines, and the wide levels are bound by memory traffic.
        lds_order();
        if (active) {
#pragma unroll
            for (int j = 0; j < 5; ++j) st[lane * 5 + j] = D[j];
        }
        lds_order();
        for (int w = lane; w < nw; w += 64) st_dev<R>(own + w0 + w, st[w]);
        for (int w = lane; w < nw; w += 64) other[w0 + w] = sent;
        lds_order();
    }
    if (!FWD) {
        double qnew[5], dd[5];
#pragma unroll
        for (int j = 0; j < 5; ++j) {
            if constexpr (sizeof(R) == sizeof(double))
                qnew[j] = qc[j];
            else
                qnew[j] = q64c[j];
            dd[j] = (double)D[j];
        }
        update_cell(qnew, dd, K);
        if (thin) {
            if (lane < nw) A.qout[w0 + lane] = pick5(qnew[0], qnew[1], qnew[2], qnew[3], qnew[4], j5);
        } else {
            double* const sd = stage_words();
            if (active) {
#pragma unroll
                for (int j = 0; j < 5; ++j) sd[lane * 5 + j] = qnew[j];
            }
            lds_order();
            for (int w = lane; w < nw; w += 64) A.qout[w0 + w] = sd[w];
            lds_order();
        }
    }
    return true;
}

// Ticket counters of a launch: one int per group, kTicketStride apart; the
// ints after the first counter are the words of an XCD-local launch: the
// XCD it runs on plus one, and the workgroups that joined it.
constexpr int kElectWord = 1, kJoinWord = 2;
__device__ __forceinline__ void clear_tickets(int* tickets) {
    if (blockIdx.x != 0) return;
    if (threadIdx.x < kTicketGroups) tickets[threadIdx.x * kTicketStride] = 0;
    if (threadIdx.x >= 64 && threadIdx.x < 66) tickets[kElectWord + (threadIdx.x - 64)] = 0;
}

// A launch of wide levels, or of a whole sweep, on the resident grid.
template <bool FWD, int MAXD, typename R, int KIND>
__global__ __launch_bounds__(kSweepBlock) void k_sweep(SweepArgs<R> A, FlowConst K) {
    // a sweep that follows a failed one in the same stream does not start
    if (__hip_atomic_load(A.err, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != 0) return;
    clear_tickets(A.tickets_next);  // the other set of counters is idle during this launch
    const int ng = A.ngroups;
    const int grp = (int)blockIdx.x % ng;
    int* const ctr = A.tickets + grp * kTicketStride;
    int tk = __builtin_amdgcn_readfirstlane(take_ticket(ctr));
    while (true) {
        const int sh = A.run_shift;
        const int u = A.ubeg + ((((tk >> sh) * ng + grp) << sh) | (tk & ((1 << sh) - 1)));
        if (u >= A.uend) return;
        int next = 0;
        if (!sweep_chunk<FWD, MAXD, R, KIND>(A, K, u, ctr, next)) return;
        tk = __builtin_amdgcn_readfirstlane(next);
    }
}

// The gradient of the previous iteration beside a sweep's thin levels: its
// node values (a forward launch) or its Green-Gauss pass (a backward one), in
// blocks of kBlock nodes or cells.
template <typename R>
struct SideWork {
    int nblk;             // blocks, a multiple of 8 (0: none)
    int* counters;        // one per XCD's span of blocks, kTicketStride apart, zero at the launch
    int* clear;           // the counters of the other direction's launch, zeroed here
    // node values
    int nN;
    const int *nlo, *ell_off;
    const int2* ell_ab;
    const R* ell_w;
    const double *nden, *q;
    R* qn;
    // gradient: tetrahedra by cnode, other cells by their face lists
    int nC, n;
    const int* snb;
    const typename Real<R>::vec4 *sgeo, *fgeo;
    const int4* cnode;
    const unsigned short* gsel;
    const double* vol;
    const int *cfo, *cf, *fno, *fn, *btype;
    const int2* fcell;
    R *gx, *gy, *gz;
};

template <bool FWD, int MAXF, typename R>
__device__ __forceinline__ void side_block(const SideWork<R>& W, int b) {
    const int i = b * kBlock + (int)threadIdx.x;
    if constexpr (FWD)
        node_body<R>(i, b * (kBlock / 64) + (int)threadIdx.x / 64, W.nN, W.nlo, W.ell_off, W.ell_ab, W.ell_w, W.nden,
                     W.q, W.qn);
    else if (MAXF == 4 && W.cnode)
        grad_tet_body<R>(i, W.nC, W.n, W.snb, W.sgeo, W.cnode, W.gsel, W.q, W.qn, W.vol, W.gx, W.gy, W.gz);
    else
        grad_body<MAXF, R>(i, W.nC, W.n, W.cfo, W.cf, W.fcell, W.fgeo, W.fno, W.fn, W.btype, W.q, W.qn, W.vol, W.gx,
                           W.gy, W.gz);
}

// Claims and works blocks until none are left: those of this XCD's span
// first (blocks x*span .. (x+1)*span-1, whose gathers then share one L2),
// then the other XCDs'.  The next block is claimed while the current one is
// worked on.
template <bool FWD, int MAXF, typename R>
__device__ __forceinline__ void side_blocks(const SideWork<R>& W, int home) {
    __shared__ int claimed;
    const int span = W.nblk / kXcd;
    for (int t = 0; t < kXcd; ++t) {
        const int x = (home + t) % kXcd;
        int* const ctr = W.counters + x * kTicketStride;
        __syncthreads();
        if (threadIdx.x == 0)
            claimed = t > 0 && __hip_atomic_load(ctr, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) >= span
                          ? span
                          : atomicAdd(ctr, 1);
        __syncthreads();
        int k = claimed;
        while (k < span) {
            __syncthreads();  // every thread has read `claimed`
            int next = 0;
            if (threadIdx.x == 0) next = atomicAdd(ctr, 1);
            side_block<FWD, MAXF, R>(W, x * span + k);
            if (threadIdx.x == 0) claimed = next;
            __syncthreads();
            k = claimed;
        }
    }
}

template <typename R>
struct XcdArgs {
    SweepArgs<R> A;
    FlowConst K;
    SideWork<R> W;
    int join;
};

// A launch of thin levels on one XCD, with the previous iteration's gradient
// on the others.  The first workgroup to start elects its XCD, and up to
// `join` workgroups of that XCD take the chunks from one counter; its other
// workgroups leave at once (workgroups are dealt to the XCDs in turn, so the
// grid holds at least 8 times `join`).  Whichever XCD it is, the workgroup
// that elected it runs, and a chunk is only ever held by a running wave, so
// the launch ends however its workgroups are placed.  The workgroups of the
// other XCDs work the side blocks, and so do the sweeping ones once their
// chunks are done.
//
// Measured between two waves, an 8-byte word takes 0.39 us to another XCD,
// 0.36 us to this one with a device-scope store, and 0.22 us with a store
// that stops in this XCD's L2: a device-scope load is served from the L2 of
// its own XCD as long as no other XCD has written the line.  With the chunk's
// results one lane each and the next ticket taken behind the first loads, a
// level of the 6.0M-cell mesh's tail (234 levels, FP64) took 1.88 us before
// and 1.20 us now (tails alone, forward and backward, 438 / 442 -> 279 / 288
// us; 262k hexahedra 252 -> 131 us; all 27 levels of a 1,296-cell mesh 53 ->
// 32 us).  Of it the store and the polls take 0.5 to 0.65 us, the face terms 0.2,
// the sum and the division 0.25.  One wave per SIMD of the XCD is
// fastest (128 waves; 256: 2% slower iterations, 512: 7%): more waves only
// add polls.
//
// The side blocks fill the CUs that the sweep leaves idle without sharing its
// XCD's issue slots and L2: on a second stream their workgroups landed there
// too, and a tail of 303 us took 605 us beside the node values and 436 beside
// the gradient (6.0M cells, FP64); inside, the two launches take 325 us with
// the node values (292 us alone) and 450 with the gradient (397 alone).
template <bool FWD, int MAXF, typename R>
__global__ __launch_bounds__(kBlock) void k_sweep_xcd(XcdArgs<R> P) {
    const SweepArgs<R>& A = P.A;
    __shared__ int role;  // 1: sweeps, 0: side blocks only, -1: leaves
    const int me = xcd_id();
    if (threadIdx.x == 0) {
        int* const elect = A.tickets + kElectWord;
        int won = __hip_atomic_load(elect, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        if (won == 0) {
            won = atomicCAS(elect, 0, me + 1);
            if (won == 0) won = me + 1;
        }
        role = won != me + 1 ? 0 : atomicAdd(A.tickets + kJoinWord, 1) < P.join ? 1 : -1;
    }
    clear_tickets(A.tickets_next);
    if (blockIdx.x == 0 && threadIdx.x < kXcd) P.W.clear[threadIdx.x * kTicketStride] = 0;
    __syncthreads();
    const int r = role;
    if (r < 0) return;
    if (r == 1 && __hip_atomic_load(A.err, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == 0) {
        int tk = __builtin_amdgcn_readfirstlane(take_ticket(A.tickets));
        while (true) {
            const int u = A.ubeg + tk;
            if (u >= A.uend) break;
            int next = 0;
            if (!sweep_chunk<FWD, MAXF, R, kThinChunks>(A, P.K, u, A.tickets, next)) break;
            tk = __builtin_amdgcn_readfirstlane(next);
        }
    }
    // The side work's arguments are read from the kernel's argument memory
    // from here on: read at the start they would take the scalar registers
    // that the sweep's loop needs.
    typedef const __attribute__((address_space(4))) unsigned* Words;
    Words w = (Words)__builtin_amdgcn_kernarg_segment_ptr() + offsetof(XcdArgs<R>, W) / 4;
    asm volatile("" : "+s"(w));
    struct Copy {
        unsigned v[sizeof(SideWork<R>) / 4];
    } copy;
#pragma unroll
    for (unsigned i = 0; i < sizeof(copy) / 4; ++i) copy.v[i] = w[i];
    const SideWork<R> W = __builtin_bit_cast(SideWork<R>, copy);
    if (W.nblk > 0) side_blocks<FWD, MAXF, R>(W, me % kXcd);
}

// The tile schedule: one workgroup per tile.
template <bool FWD, int MAXD, typename R>
__global__ __launch_bounds__(kSweepBlock) void k_sweep_tiles(SweepArgs<R> A, FlowConst K) {
    if (__hip_atomic_load(A.err, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != 0) return;
    const SweepDir<R>& S = A.dir[FWD ? 0 : 1];
    const int W = (int)blockDim.x / 64;
    const int w = (int)threadIdx.x / 64;
    int none = 0;
    for (int kk = blockIdx.x; kk < A.ntiles; kk += gridDim.x) {
        const int k = FWD ? kk : A.ntiles - 1 - kk;
        const int t0 = S.tile_chunk[k], t1 = S.tile_chunk[k + 1];
        for (int t = t0 + w; t < t1; t += W)
            if (!sweep_chunk<FWD, MAXD, R, kAnyChunks>(A, K, __builtin_amdgcn_readfirstlane(S.pos[t]), nullptr, none))
                return;
    }
}
