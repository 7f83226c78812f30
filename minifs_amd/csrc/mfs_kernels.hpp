// Per-cell and per-node gather kernels of the solver path, included by
// mfs_device.hip inside namespace mfs::dev.
//
// Device layout: state q, residual and node values are stored cell-major
// (5 consecutive doubles per cell or node) so that a gather of one
// neighbour touches one or two cache lines; faces and nodes are stored in
// first-touch order of the cell traversal.  Each kernel visits a cell's
// faces in ascending mesh face id (the per-cell list order), which is the
// order in which the reference's face loops add into that cell.
//
// The MAXF template bounds the faces per cell (4 for tetrahedral meshes, 6
// otherwise).  Slots beyond a cell's face count are loaded from the cell's
// first face, so every load of a cell can be issued at once, and their
// contributions are skipped.

// Real types of the kernels: FP64 (the reference's arithmetic) and FP32
// (the mixed-precision operator).  kSent is a NaN payload that arithmetic
// never produces, used by the sweeps to mark unpublished values.
template <typename R>
struct Real;
template <>
struct Real<double> {
    using bits = unsigned long long;
    using vec4 = double4;
    static constexpr bits kSent = 0x7FF4D51F5EED0000ULL;
    static constexpr double kMost = 1.7976931348623157e308;  // largest finite value
};
template <>
struct Real<float> {
    using bits = unsigned int;
    using vec4 = float4;
    static constexpr bits kSent = 0x7FA5D51Fu;
    static constexpr float kMost = 3.4028235e38f;
};

// A value that the last block of the same launch reads (write-through, where
// a plain store may stay in the XCD's L2).
__device__ __forceinline__ void st_part(double* p, double v) {
    __hip_atomic_store(reinterpret_cast<unsigned long long*>(p), __builtin_bit_cast(unsigned long long, v),
                       __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

template <int NV, int NW = kBlock / 64>
__device__ __forceinline__ void block_sum(double (&v)[NV], double* out, int stride = 1) {
    __shared__ double s[NW][NV];
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1)
#pragma unroll
        for (int j = 0; j < NV; ++j) v[j] += __shfl_down(v[j], off, 64);
    const int w = threadIdx.x >> 6;
    if ((threadIdx.x & 63) == 0)
#pragma unroll
        for (int j = 0; j < NV; ++j) s[w][j] = v[j];
    __syncthreads();
    if (threadIdx.x == 0) {
#pragma unroll
        for (int j = 0; j < NV; ++j) {
            double a = s[0][j];
            for (int k = 1; k < (int)(blockDim.x >> 6); ++k) a += s[k][j];
            out[(size_t)j * stride] = a;
        }
    }
}

template <int NW = kBlock / 64>
__device__ __forceinline__ void block_minmax(double vmin, double vmax, double* out_min, double* out_max) {
    __shared__ double smin_[NW], smax_[NW];
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1) {
        vmin = smin(vmin, __shfl_down(vmin, off, 64));
        vmax = smax(vmax, __shfl_down(vmax, off, 64));
    }
    const int w = threadIdx.x >> 6;
    if ((threadIdx.x & 63) == 0) {
        smin_[w] = vmin;
        smax_[w] = vmax;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        double a = smin_[0], b = smax_[0];
        for (int k = 1; k < (int)(blockDim.x >> 6); ++k) {
            a = smin(a, smin_[k]);
            b = smax(b, smax_[k]);
        }
        *out_min = a;
        *out_max = b;
    }
}

// Logical index of this workgroup.  Workgroups are dispatched round-robin
// over the 8 XCDs, each with its own L2; mapping consecutive logical blocks
// to one XCD gives each L2 a contiguous range of cells, whose neighbours
// (and their faces and nodes) are mostly in the same range.  The grid is a
// multiple of kXcd blocks.
__device__ __forceinline__ int xcd_block() {
    const int b = (int)blockIdx.x;
    return (b % kXcd) * ((int)gridDim.x / kXcd) + b / kXcd;
}

__device__ __forceinline__ void load5(const double* __restrict__ p, double v[5]) {
#pragma unroll
    for (int j = 0; j < 5; ++j) v[j] = p[j];
}
template <typename R>
__device__ __forceinline__ void load5r(const R* __restrict__ p, R v[5]) {
#pragma unroll
    for (int j = 0; j < 5; ++j) v[j] = p[j];
}

__global__ void k_fill(double* p, size_t n, double v) {
    size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) p[i] = v;
}
__global__ void k_fill_f(float* p, size_t n, float v) {
    size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) p[i] = v;
}
__global__ void k_fill_i(int* p, size_t n, int v) {
    size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) p[i] = v;
}

// A field between its device array and the reference layout.  Value t of the
// layout is row t % rows of block t / rows; a row below nmap is stored at
// device row map[row], and the value of block j at row d at
// [d * row_stride + j * block_stride + offset].
struct FieldMap {
    size_t rows, nmap;
    const int* map;
    size_t row_stride, block_stride, offset;
};
__device__ __forceinline__ size_t field_index(const FieldMap& M, size_t t) {
    const size_t j = t / M.rows, row = t - j * M.rows;
    const size_t d = row < M.nmap ? (size_t)M.map[row] : row;
    return d * M.row_stride + j * M.block_stride + M.offset;
}
// Values [t0, t0 + cnt) of the layout to out, as doubles (src32: an FP32 field).
__global__ __launch_bounds__(kBlock) void k_field_out(FieldMap M, size_t t0, size_t cnt, const double* __restrict__ src,
                                                      const float* __restrict__ src32, double* __restrict__ out) {
    const size_t i = (size_t)blockIdx.x * kBlock + threadIdx.x;
    if (i >= cnt) return;
    const size_t k = field_index(M, t0 + i);
    out[i] = src32 ? (double)src32[k] : src[k];
}
// The other way, into one array or two.
__global__ __launch_bounds__(kBlock) void k_field_in(FieldMap M, size_t t0, size_t cnt, const double* __restrict__ in,
                                                     double* __restrict__ dst, double* __restrict__ dst2) {
    const size_t i = (size_t)blockIdx.x * kBlock + threadIdx.x;
    if (i >= cnt) return;
    const size_t k = field_index(M, t0 + i);
    const double v = in[i];
    dst[k] = v;
    if (dst2) dst2[k] = v;
}
__global__ __launch_bounds__(kBlock) void k_narrow(size_t n, const double* __restrict__ src, float* __restrict__ dst) {
    const size_t i = (size_t)blockIdx.x * kBlock + threadIdx.x;
    if (i < n) dst[i] = (float)src[i];
}

// SetGhostVariables (src/Kernels/load_grid.cpp:953-1212), inviscid branch:
// the ghost state behind each boundary face from the state of the cell in
// front of it.  One thread per boundary face k; the ghost is cell nC+k and
// gface[k] the device id of its face.  WALL and SYMM mirror the velocity
// in the face plane; FAR_FIELD takes the Riemann-invariant state
// (supersonic in/outflow, subsonic in/outflow with the entropy of the
// upwind side) and extrapolates it to the ghost.  Expressions and their
// order follow the reference; the FAR_FIELD subsonic branch calls pow,
// whose GPU result may differ from the host's in the last bit.
struct GhostConst {
    double rho_s, u_s, v_s, w_s, p_s;  // freestream (p gauge)
};

__global__ __launch_bounds__(kBlock) void k_ghost(int nB, int nC, const int* __restrict__ gface,
                                                  const int2* __restrict__ fcell, const double4* __restrict__ fgeo,
                                                  const int* __restrict__ btype, FlowConst K, GhostConst G,
                                                  double* __restrict__ q, float* __restrict__ q32) {
    const int k = (int)(blockIdx.x * blockDim.x + threadIdx.x);
    if (k >= nB) return;
    const int type = btype[k];
    if (type == BC_INTERFACE) return;
    const int f = gface[k];
    const int c1 = fcell[f].x;
    const size_t o1 = (size_t)c1 * 5, o2 = (size_t)(nC + k) * 5;
    const double4 g = fgeo[f];
    const double xfn = g.x, yfn = g.y, zfn = g.z;
    const double gam = K.gam, p_bar = K.p_bar;
    const double r1 = q[o1], u1 = q[o1 + 1], v1 = q[o1 + 2], w1 = q[o1 + 3], p1 = q[o1 + 4];
    double rho2 = q[o2], u2 = q[o2 + 1], v2 = q[o2 + 2], w2 = q[o2 + 3], p2 = q[o2 + 4];
    if (type == BC_WALL || type == BC_SYMM) {
        p2 = p1;
        rho2 = r1;
        const double vn = 2. * (xfn * u1 + yfn * v1 + zfn * w1);
        u2 = u1 - vn * xfn;
        v2 = v1 - vn * yfn;
        w2 = w1 - vn * zfn;
    } else if (type == BC_FAR_FIELD) {
        const double um = G.u_s, vm = G.v_s, wm = G.w_s;
        const double up = u1, vp = v1, wp = w1;
        const double rhom = G.rho_s, pm = G.p_s + p_bar;
        const double rhop = r1, pp = p1 + p_bar;
        const double norm_of_uvw = sqrt(um * um + vm * vm + wm * wm);
        const double vnm = xfn * um + yfn * vm + zfn * wm;
        const double vnp = xfn * up + yfn * vp + zfn * wp;
        const double cm = sqrt(gam * pm / rhom);
        const double cp = sqrt(gam * pp / rhop);
        const double riemm = vnm - 2. * cm / (gam - 1.);
        const double riemp = vnp + 2. * cp / (gam - 1.);
        const double vnb = 0.5 * (riemp + riemm);
        const double cb = 0.25 * (riemp - riemm) * (gam - 1.);
        if (fabs(vnb / cb) > 1.) {
            if (vnb <= 0.0) {
                rho2 = rhom;
                u2 = um;
                v2 = vm;
                w2 = wm;
                p2 = pm;
            } else {
                rho2 = rhop;
                u2 = up;
                v2 = vp;
                w2 = wp;
                p2 = pp;
            }
        } else {
            const double rela_vnb = vnb / norm_of_uvw;
            if (rela_vnb <= -0.0 || rela_vnb > 0.0) {
                const bool in = rela_vnb <= -0.0;
                const double bu = in ? um : up, bv = in ? vm : vp, bw = in ? wm : wp, bvn = in ? vnm : vnp;
                const double bp = in ? pm : pp, brho = in ? rhom : rhop;
                const double vtx = bu - bvn * xfn, vty = bv - bvn * yfn, vtz = bw - bvn * zfn;
                const double entr = bp / pow(brho, gam);
                rho2 = pow((cb * cb / (entr * gam)), double(1. / (gam - 1.)));
                u2 = vtx + vnb * xfn;
                v2 = vty + vnb * yfn;
                w2 = vtz + vnb * zfn;
                p2 = cb * cb * rho2 / gam;
            } else {
                rho2 = 0.5 * (rhop + rhom);
                u2 = 0.5 * (up + um);
                v2 = 0.5 * (vp + vm);
                w2 = 0.5 * (wp + wm);
                p2 = 0.5 * (pp + pm);
            }
        }
        rho2 = 2 * rho2 - rhop;
        u2 = 2 * u2 - up;
        v2 = 2 * v2 - vp;
        w2 = 2 * w2 - wp;
        p2 = 2 * p2 - pp;
        p2 -= p_bar;
    }  // other types: the reference reports an error, keeps the ghost state and clamps it below
    rho2 = smax(rho2, K.rho_min);
    rho2 = smin(rho2, K.rho_max);
    p2 = smax(p2, K.p_min);
    p2 = smin(p2, K.p_max);
    const double out[5] = {rho2, u2, v2, w2, p2};
#pragma unroll
    for (int j = 0; j < 5; ++j) q[o2 + j] = out[j];
    if (q32) {
#pragma unroll
        for (int j = 0; j < 5; ++j) q32[o2 + j] = (float)out[j];
    }
}

// Cell-face slots of one cell: device face ids, padded with the first face.
template <int MAXF>
__device__ __forceinline__ int cell_faces(const int* __restrict__ cfo, const int* __restrict__ cf, int c,
                                          int (&fs)[MAXF]) {
    const int k0 = cfo[c];
    const int nf = cfo[c + 1] - k0;
#pragma unroll
    for (int s = 0; s < MAXF; ++s) fs[s] = cf[k0 + (s < nf ? s : 0)];
    return nf;
}

// Slots of a cell that can hold a face, of the LPC its neighbour and face
// rows have room for, and the place of slot s of cell c in the slot geometry
// and distances: slot by slot, so that a wave's load of one slot's 32 bytes a
// cell spans 16 lines.  Stored cell by cell, every lane's load was in a line
// of its own, and the CU's cache takes a cycle or more per line.
// Before and after (residual pass, gradient): 6.0M tetrahedra FP64 565 -> 513
// and 440 -> 397 us, 1.3M 128 -> 117 and 2.9M mixed 297 -> 276 us (residual);
// 262k hexahedra, whose pass also took the two empty slots along, 47 -> 39 us.
// The separate entry points' passes read these tables too, where each face's
// cells, normal and distances were a gather of their own (384k cells: residual
// 36 -> 31, time step 24.5 -> 17.4, diagonal 12.8 -> 11.4 us).
template <int LPC>
constexpr int kSlots = LPC == 4 ? 4 : 6;
__device__ __forceinline__ size_t slot_at(int s, int c, int nC) { return (size_t)s * nC + c; }

// A cell's slots: neighbour, the face's stored normal and area, this side's
// distance, and whether the cell is the face's first (the slot normal points
// away from the cell; negated back where the cell is second, exactly).
template <int NS>
struct CellSlots {
    int nf, oth[NS];
    double4 g[NS];
    double dn[NS];
    bool first[NS];
};
template <int LPC, bool DN>
__device__ __forceinline__ void load_slots(int c, int nC, const int* __restrict__ snb,
                                           const double4* __restrict__ sgeo, const double* __restrict__ sdn,
                                           const int* __restrict__ sflip, CellSlots<kSlots<LPC>>& L) {
#pragma unroll
    for (int s = 0; s < kSlots<LPC>; ++s) L.oth[s] = snb[(size_t)c * LPC + s];
    const unsigned sf = (unsigned)sflip[c];
    L.nf = (int)((sf >> 8) & 15u);
#pragma unroll
    for (int s = 0; s < kSlots<LPC>; ++s) {
        const size_t i = slot_at(s, c, nC);
        const double4 v = sgeo[i];
        L.first[s] = ((sf >> s) & 1u) == 0;
        L.g[s] = L.first[s] ? v : make_double4(-v.x, -v.y, -v.z, v.w);
        if (DN) L.dn[s] = sdn[i];
    }
}

// The cell's flux across one slot, added with the face's sign.  hc = the
// cell's total enthalpy, hqc = that by its density, qo = the other state.
__device__ __forceinline__ void add_face_flux(const double (&qc)[5], double hc, double hqc, const double (&qo)[5],
                                              bool first, const double4& g, bool used, const FlowConst& K,
                                              double (&r)[5]) {
    double ql[5], qr[5], F[5];
#pragma unroll
    for (int j = 0; j < 5; ++j) {
        ql[j] = first ? qc[j] : qo[j];
        qr[j] = first ? qo[j] : qc[j];
    }
    const double ho = total_enthalpy(qo, K.gamm1, K.p_bar), hqo = ho / qo[0];
    roe_flux<double>(ql, qr, first ? hc : ho, first ? ho : hc, first ? hqc : hqo, first ? hqo : hqc, g.x, g.y, g.z,
                     g.w, K.gamm1, K.alf_l, kTINYd, F);
    if (used) {
        if (first) {
#pragma unroll
            for (int j = 0; j < 5; ++j) r[j] -= F[j];
        } else {
#pragma unroll
            for (int j = 0; j < 5; ++j) r[j] += F[j];
        }
    }
}

// CellIsMG's test of one face: |dp| / (sum of both total pressures) > 0.1,
// without the division where no lane of the wave is near the limit (at most
// 0.0999 of a positive sum, the rounded quotient is below 0.1).
__device__ __forceinline__ bool pressure_jump(double pl, double pr, double p_bar) {
    const double pd = fabs(pr - pl), ps = pr + pl + p_bar + p_bar;
    bool jump = !((pd <= 0.0999 * ps) & (ps > 1e-280));
    if (__builtin_amdgcn_ballot_w64(jump) != 0) jump = pd / ps > 0.1;
    return jump;
}

// ---------------------------------------------------------------------------
// Residual: InviscidFlux + RoeFlux_noprec + LoadFlux (cal_flux.cpp:84-192,
// 682-833, 1219-1254).  res[c] starts at its current value and receives -F for
// faces where c is c1 and +F where c is c2, in ascending face order.  Block partial sums of res^2 feed the
// residual norm of main.cpp:294-317.
template <int LPC>
__global__ __launch_bounds__(kBlock) void k_flux(int nC, const int* __restrict__ snb,
                                                 const double4* __restrict__ sgeo, const int* __restrict__ sflip,
                                                 const double* __restrict__ q, double* __restrict__ res,
                                                 double* __restrict__ part, FlowConst K) {
    constexpr int NS = kSlots<LPC>;
    const int c = xcd_block() * kBlock + (int)threadIdx.x;
    double r[5] = {0.0, 0.0, 0.0, 0.0, 0.0};
    if (c < nC) {
        load5(res + (size_t)c * 5, r);
        double qc[5];
        load5(q + (size_t)c * 5, qc);
        CellSlots<NS> L;
        load_slots<LPC, false>(c, nC, snb, sgeo, nullptr, sflip, L);
        const double hc = total_enthalpy(qc, K.gamm1, K.p_bar), hqc = hc / qc[0];
#pragma unroll
        for (int s = 0; s < NS; ++s) {
            double qo[5];
            load5(q + (size_t)L.oth[s] * 5, qo);
            add_face_flux(qc, hc, hqc, qo, L.first[s], L.g[s], s < L.nf, K, r);
        }
#pragma unroll
        for (int j = 0; j < 5; ++j) res[(size_t)c * 5 + j] = r[j];
    }
    double s2[5];
#pragma unroll
    for (int j = 0; j < 5; ++j) s2[j] = r[j] * r[j];
    block_sum<5>(s2, part + blockIdx.x, (int)gridDim.x);
}

// ---------------------------------------------------------------------------
// Local time step: TimeStepNormal_new + CellIsMG + LimitTimeStep
// (compute_timestep.cpp:758-823, 1315-1338, 836-918), with the cell's own
// |u.n| + a on every face.
template <int LPC>
__global__ __launch_bounds__(kBlock) void k_timestep(int nC, const int* __restrict__ snb,
                                                     const double4* __restrict__ sgeo, const double* __restrict__ sdn,
                                                     const int* __restrict__ sflip, const double* __restrict__ q,
                                                     double* __restrict__ dt, double* __restrict__ part, FlowConst K,
                                                     double cfl, double cfl_min) {
    constexpr int NS = kSlots<LPC>;
    const int c = xcd_block() * kBlock + (int)threadIdx.x;
    double vmin = kBIGd, vmax = 0.0;
    if (c < nC) {
        double qc[5];
        load5(q + (size_t)c * 5, qc);
        const double rho = qc[0], u = qc[1], v = qc[2], w = qc[3], p = qc[4];
        CellSlots<NS> L;
        load_slots<LPC, true>(c, nC, snb, sgeo, sdn, sflip, L);
        double po[NS];
#pragma unroll
        for (int s = 0; s < NS; ++s) po[s] = q[(size_t)L.oth[s] * 5 + 4];
        const double c2tmp = K.gam * (p + K.p_bar) / rho;
        const double a = sqrt(c2tmp);
        double dtc = kBIGd;
        int det = 1;
        double eig[NS];
#pragma unroll
        for (int s = 0; s < NS; ++s) {
            double vn = u * L.g[s].x + v * L.g[s].y + w * L.g[s].z;
            vn = fabs(vn);
            eig[s] = vn + a;
            const bool jump = pressure_jump(p, po[s], K.p_bar);
            if (s < L.nf) {
                dtc = smin(dtc, L.dn[s] / eig[s]);
                if (jump) det = 0;
            }
        }
        double cfl_tmp;
        if (p > K.p_break)
            cfl_tmp = cfl;
        else if (p < K.p_min)
            cfl_tmp = cfl_min;
        else
            cfl_tmp = (p - K.p_min) / (K.p_break - K.p_min) * (cfl - cfl_min) + cfl_min;
        if (!det) cfl_tmp = cfl_min;
        dtc *= cfl_tmp;
        dt[c] = dtc;
        vmin = dtc;
        vmax = dtc;
    }
    block_minmax(vmin, vmax, part + (size_t)5 * gridDim.x + blockIdx.x, part + (size_t)6 * gridDim.x + blockIdx.x);
}

// Residual, local time step and LU-SGS diagonal in one pass over a cell's
// faces, for the fused iteration: the arithmetic of k_flux (from zero),
// k_timestep and k_diag, which all read the state at the start of the
// iteration.  The cell's own state is loaded once and only the neighbour's
// is gathered per face.  With MIXED the FP32 inputs of the implicit
// operator (state snapshot, Diag) are written as well.
// The pass is near its bytes (6.0M cells FP64: 1.84 GB, 367 us at the rate of
// a copy, 513 us taken) with 316 us of FP64 arithmetic beside them, so the
// cell's own enthalpy and its quotient are formed once instead of at every
// face and the pressure jump is decided without a division where it can be:
// 10% fewer instructions, 6.0M 513 -> 491 us, 2.9M mixed 276 -> 265 us.  (Four
// waves a SIMD instead of three: spills, 6.0M 5% slower iterations.  One lane
// per face instead of per cell: 6.0M 538 -> 567, 262k hexahedra 47 -> 75 us.)
// Per cell: the faces' fluxes added in slot order (the cell's ascending
// face order), the time step from the smallest dn/eig, the CFL choice and
// the diagonal.  NS slots, the first nf used; oth = the face's other cell,
// g = the face's stored normal and area (c1 -> c2), first = this cell is c1.
template <int NS, bool MIXED>
__device__ __forceinline__ void flux_ts_cell(int c, const double (&qc)[5], const CellSlots<NS>& L,
                                             const double* __restrict__ q, const double* __restrict__ vol,
                                             double* __restrict__ res, double* __restrict__ dt,
                                             double* __restrict__ diag, const FlowConst& K, double cfl, double cfl_min,
                                             float* __restrict__ q32, float* __restrict__ diag32, double (&r)[5],
                                             double& dtc) {
    const double c2tmp = K.gam * (qc[4] + K.p_bar) / qc[0];
    const double a = sqrt(c2tmp);
    const double hc = total_enthalpy(qc, K.gamm1, K.p_bar), hqc = hc / qc[0];
    dtc = kBIGd;
    int det = 1;
    double eig[NS];
#pragma unroll
    for (int s = 0; s < NS; ++s) {
        double qo[5];
        load5(q + (size_t)L.oth[s] * 5, qo);
        add_face_flux(qc, hc, hqc, qo, L.first[s], L.g[s], s < L.nf, K, r);
        double vn = qc[1] * L.g[s].x + qc[2] * L.g[s].y + qc[3] * L.g[s].z;
        vn = fabs(vn);
        eig[s] = vn + a;
        const bool jump = pressure_jump(qc[4], qo[4], K.p_bar);
        if (s < L.nf) {
            dtc = smin(dtc, L.dn[s] / eig[s]);
            if (jump) det = 0;
        }
    }
#pragma unroll
    for (int j = 0; j < 5; ++j) res[(size_t)c * 5 + j] = r[j];
    const double p = qc[4];
    double cfl_tmp;
    if (p > K.p_break)
        cfl_tmp = cfl;
    else if (p < K.p_min)
        cfl_tmp = cfl_min;
    else
        cfl_tmp = (p - K.p_min) / (K.p_break - K.p_min) * (cfl - cfl_min) + cfl_min;
    if (!det) cfl_tmp = cfl_min;
    dtc *= cfl_tmp;
    dt[c] = dtc;
    double dg = vol[c] / dtc;
#pragma unroll
    for (int s = 0; s < NS; ++s)
        if (s < L.nf) dg += 0.5 * L.g[s].w * eig[s] * K.lhs_omga;
    diag[c] = dg;
    if (MIXED) {
        diag32[c] = (float)dg;
#pragma unroll
        for (int j = 0; j < 5; ++j) q32[(size_t)c * 5 + j] = (float)qc[j];
    }
}

// The pass from the per-slot tables laid out by cell (neighbour, normal
// pointing away from the cell with its area, this side's distance, and the
// slots whose face has this cell second): contiguous reads, then the
// neighbours' states.  The stored normal is the slot normal negated back
// where the cell is the face's second cell, exactly.
template <int LPC, bool MIXED>
__device__ __forceinline__ void flux_ts_slot_body(int c, int nC, const int* __restrict__ snb,
                                                  const double4* __restrict__ sgeo, const double* __restrict__ sdn,
                                                  const int* __restrict__ sflip, const double* __restrict__ q,
                                                  const double* __restrict__ vol, double* __restrict__ res,
                                                  double* __restrict__ dt, double* __restrict__ diag,
                                                  double* __restrict__ pblk, int pstride, const FlowConst& K, double cfl,
                                                  double cfl_min, float* __restrict__ q32,
                                                  float* __restrict__ diag32) {
    constexpr int NS = kSlots<LPC>;
    double r[5] = {0.0, 0.0, 0.0, 0.0, 0.0};
    double vmin = kBIGd, vmax = 0.0;
    if (c < nC) {
        double qc[5];
        load5(q + (size_t)c * 5, qc);
        CellSlots<NS> L;
        load_slots<LPC, true>(c, nC, snb, sgeo, sdn, sflip, L);
        double dtc;
        flux_ts_cell<NS, MIXED>(c, qc, L, q, vol, res, dt, diag, K, cfl, cfl_min, q32, diag32,
                                 r, dtc);
        vmin = dtc;
        vmax = dtc;
    }
    double s2[5];
#pragma unroll
    for (int j = 0; j < 5; ++j) s2[j] = r[j] * r[j];
    __shared__ double tot[7];
    block_sum<5>(s2, tot);
    block_minmax(vmin, vmax, tot + 5, tot + 6);
    if (threadIdx.x == 0) {
#pragma unroll
        for (int j = 0; j < 7; ++j) st_part(pblk + (size_t)j * pstride, tot[j]);
    }
}

// Diag alone (forward_lusgs.cpp:94-99 + CalDiagLUSGS :554-595), from dt.
// With `run`, only cells whose dt exceeds ratio_dtmax*dt_min are clamped
// and recomputed (compute_timestep.cpp:929-945), and only when the
// reduction found the ratio exceeded.
template <int LPC>
__device__ __forceinline__ void diag_body(int c, int nC, const double4* __restrict__ sgeo, const int* __restrict__ sflip,
                                          const double* __restrict__ q, const double* __restrict__ vol,
                                          double* __restrict__ dt, double* __restrict__ diag,
                                          const double* __restrict__ run, double ratio_dtmax, const FlowConst& K,
                                          float* __restrict__ diag32) {
    if (c >= nC) return;
    double dtc = dt[c];
    if (run) {
        if (run[2] == 0.0) return;
        const double lim = ratio_dtmax * run[1];
        if (!(dtc > lim)) return;
        dtc = lim;
        dt[c] = dtc;
    }
    double qc[5];
    load5(q + (size_t)c * 5, qc);
    const int nf = (sflip[c] >> 8) & 15;
    const double a = sqrt(K.gam * (qc[4] + K.p_bar) / qc[0]);
    double dg = vol[c] / dtc;
#pragma unroll
    for (int s = 0; s < kSlots<LPC>; ++s) {
        const double4 g = sgeo[slot_at(s, c, nC)];  // either side's normal: |u.n| is the same
        double vn = qc[1] * g.x + qc[2] * g.y + qc[3] * g.z;
        vn = fabs(vn);
        if (s < nf) dg += 0.5 * g.w * (vn + a) * K.lhs_omga;
    }
    diag[c] = dg;
    if (diag32) diag32[c] = (float)dg;
}
template <int LPC>
__global__ __launch_bounds__(kBlock) void k_diag(int nC, const double4* __restrict__ sgeo,
                                                 const int* __restrict__ sflip, const double* __restrict__ q,
                                                 const double* __restrict__ vol, double* __restrict__ dt,
                                                 double* __restrict__ diag, const double* __restrict__ run,
                                                 double ratio_dtmax, FlowConst K, float* __restrict__ diag32) {
    diag_body<LPC>(xcd_block() * kBlock + (int)threadIdx.x, nC, sgeo, sflip, q, vol, dt, diag, run, ratio_dtmax, K,
                   diag32);
}

// The ratio_dtmax clamp alone (compute_timestep.cpp:929-945) over a small
// grid: every workgroup reads the reduction's flag first and returns when
// the clamp is off, which is the rule at the reference's ratio_dtmax.
template <int LPC>
__global__ __launch_bounds__(kBlock) void k_clamp(int nC, const double4* __restrict__ sgeo,
                                                  const int* __restrict__ sflip, const double* __restrict__ q,
                                                  const double* __restrict__ vol, double* __restrict__ dt,
                                                  double* __restrict__ diag, const double* __restrict__ run,
                                                  double ratio_dtmax, FlowConst K, float* __restrict__ diag32) {
    if (run[2] == 0.0) return;
    for (int c = (int)(blockIdx.x * kBlock + threadIdx.x); c < nC; c += (int)(gridDim.x * kBlock))
        diag_body<LPC>(c, nC, sgeo, sflip, q, vol, dt, diag, run, ratio_dtmax, K, diag32);
}

// FP32 operator inputs of a mixed-precision context from the FP64 state and
// Diag (interior cells; the ghost part of the snapshot never changes).
__global__ __launch_bounds__(kBlock) void k_mixed_inputs(int nC, const double* __restrict__ q,
                                                         const double* __restrict__ diag, float* __restrict__ q32,
                                                         float* __restrict__ diag32) {
    const int c = blockIdx.x * kBlock + (int)threadIdx.x;
    if (c >= nC) return;
#pragma unroll
    for (int j = 0; j < 5; ++j) q32[(size_t)c * 5 + j] = (float)q[(size_t)c * 5 + j];
    diag32[c] = (float)diag[c];
}

// ---------------------------------------------------------------------------
// Reductions.  mode bits: 1 = residual norms -> run[3..7], 2 = dt extrema
// (running max/min of compute_timestep.cpp:914-918, clamp flag), 4 = write
// history record `slot` from run[].
// One workgroup of kReduceBlock threads reads each block's partials once
// (norms and extrema together) and sums them in a fixed tree.  The partials
// are stored value-major, part[j * nblk + block] for the five squared
// norms (j = 0..4), dt min (5) and dt max (6), so that every load of a wave
// reads 64 consecutive doubles: with one 64-byte record per block, a wave's
// load touched 32 cache lines, and a 6.0M-cell reduction took 57 us in the
// single workgroup's load unit.
constexpr int kReduceBlock = 1024;

// The second half of a reduction: the block tree over the threads' folds
// (s: squared-norm sums, a: dt min, b: dt max), the running extrema, the
// clamp flag and the history record.
__device__ __forceinline__ void reduce_finish(double (&s)[5], double a, double b, double* __restrict__ run,
                                              double* __restrict__ hist, int slot, int mode, double ratio_dtmax) {
    constexpr int NW = kReduceBlock / 64;
    if (mode & 1) {
        __shared__ double tot[5];
        block_sum<5, NW>(s, tot);
        __syncthreads();
        if (threadIdx.x == 0)
            for (int j = 0; j < 5; ++j) run[3 + j] = sqrt(tot[j]);
    }
    if (mode & 2) {
        __shared__ double mn, mx;
        block_minmax<NW>(a, b, &mn, &mx);
        __syncthreads();
        if (threadIdx.x == 0) {
            const double dmax = smax(run[0], mx);
            const double dmin = smin(run[1], mn);
            run[0] = dmax;
            run[1] = dmin;
            run[2] = (dmax / dmin > ratio_dtmax) ? 1.0 : 0.0;
        }
    }
    __syncthreads();
    if (threadIdx.x == 0 && (mode & 4)) {
        double* h = hist + (size_t)slot * 7;
        for (int j = 0; j < 5; ++j) h[j] = run[3 + j];
        h[5] = run[0];
        h[6] = run[1];
    }
}

__device__ __forceinline__ void reduce_body(int nblk, const double* __restrict__ part, double* __restrict__ run,
                                            double* __restrict__ hist, int slot, int mode, double ratio_dtmax) {
    double s[5] = {0.0, 0.0, 0.0, 0.0, 0.0};
    double a = kBIGd, b = 0.0;
    // each thread folds records k, k+1024, ... in that order; the records
    // of a group of kReduceBatch are loaded together before they are added
    // (a group past the end loads a valid record in place of the missing
    // ones and skips them), so the thread waits for one round trip per
    // group, not per record
    constexpr int kReduceBatch = 7;  // 8 spills registers
    for (int k = threadIdx.x; k < nblk; k += kReduceBatch * kReduceBlock) {
        double r[kReduceBatch][7];
#pragma unroll
        for (int i = 0; i < kReduceBatch; ++i) {
            const int e = min(k + i * kReduceBlock, nblk - 1);
#pragma unroll
            for (int j = 0; j < 7; ++j) r[i][j] = part[(size_t)j * nblk + e];
        }
#pragma unroll
        for (int i = 0; i < kReduceBatch; ++i) {
            if (k + i * kReduceBlock >= nblk) break;
            if (mode & 1) {
#pragma unroll
                for (int j = 0; j < 5; ++j) s[j] += r[i][j];
            }
            if (mode & 2) {
                a = smin(a, r[i][5]);
                b = smax(b, r[i][6]);
            }
        }
    }
    reduce_finish(s, a, b, run, hist, slot, mode, ratio_dtmax);
}
__global__ __launch_bounds__(kReduceBlock) void k_reduce(int nblk, const double* __restrict__ part, double* __restrict__ run,
                                                   double* __restrict__ hist, int slot, int mode, double ratio_dtmax) {
    reduce_body(nblk, part, run, hist, slot, mode, ratio_dtmax);
}

// The same reduction by the last block of the pass that writes the partials,
// for up to kInlineReduceBlocks of them: no launch of its own (k_reduce takes
// 8 us on a mesh of a few blocks, most of it start and a serial tree of 16
// waves' sums).  Thread t stands for threads t, t + 256, ... of k_reduce, so
// the sums are k_reduce's.  Each block counts itself in `counter` after its
// partials are written through; the last one sets it back to zero.
// ms per iteration, launch of its own -> here: 1k cells 0.0885 -> 0.083, 20k
// 0.198 -> 0.192, 94k (368 blocks) 0.309 -> 0.306; with 768 and 1024 blocks,
// whose partials the one block of 256 threads reads in eight round trips,
// both take the same (0.443 | 0.442 and 0.634 | 0.632), hence the line.
constexpr int kInlineReduceBlocks = 512;
struct InlineReduce {
    int* counter;  // null: no reduction here
    double *run, *hist;
    int slot;
    double ratio_dtmax;
};
__device__ __forceinline__ double ld_part(const double* p) {
    return __builtin_bit_cast(double, __hip_atomic_load(reinterpret_cast<const unsigned long long*>(p),
                                                        __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT));
}
__device__ __forceinline__ void reduce_last_block(int nblk, const double* part, const InlineReduce& I) {
    __shared__ int last;
    if (threadIdx.x == 0) {
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // this thread's partials are written
        last = __hip_atomic_fetch_add(I.counter, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == nblk - 1;
    }
    __syncthreads();
    if (!last) return;
    constexpr int NW = kReduceBlock / 64, P = kReduceBlock / kBlock;
    __shared__ double wave[NW][7];
    const int lane = (int)threadIdx.x & 63, w = (int)threadIdx.x / 64;
    if (threadIdx.x == 0) __hip_atomic_store(I.counter, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    const int groups = min(P, (nblk + kBlock - 1) / kBlock);  // of 256 threads of k_reduce with records
    for (int g = 0; g < groups; ++g) {
        double v[5] = {0.0, 0.0, 0.0, 0.0, 0.0};
        double a = kBIGd, b = 0.0;
        for (int k = g * kBlock + (int)threadIdx.x; k < nblk; k += kReduceBlock) {
            double r[7];
#pragma unroll
            for (int j = 0; j < 7; ++j) r[j] = ld_part(part + (size_t)j * nblk + k);
#pragma unroll
            for (int j = 0; j < 5; ++j) v[j] += r[j];
            a = smin(a, r[5]);
            b = smax(b, r[6]);
        }
#pragma unroll
        for (int off = 32; off >= 1; off >>= 1) {
#pragma unroll
            for (int j = 0; j < 5; ++j) v[j] += __shfl_down(v[j], off, 64);
            a = smin(a, __shfl_down(a, off, 64));
            b = smax(b, __shfl_down(b, off, 64));
        }
        if (lane == 0) {
            double* const o = wave[g * (kBlock / 64) + w];
#pragma unroll
            for (int j = 0; j < 5; ++j) o[j] = v[j];
            o[5] = a;
            o[6] = b;
        }
    }
    __syncthreads();
    if (threadIdx.x < 7) {  // one value each, over the waves that had records
        const int j = (int)threadIdx.x, waves = groups * (kBlock / 64);
        double x = wave[0][j];
        for (int k = 1; k < waves; ++k) {
            const double y = wave[k][j];
            x = j < 5 ? x + y : j == 5 ? smin(x, y) : smax(x, y);
        }
        double out = x;
        if (j < 5) out = I.run[3 + j] = sqrt(x);
        if (j == 5) out = I.run[1] = smin(I.run[1], x);
        if (j == 6) out = I.run[0] = smax(I.run[0], x);
        wave[0][j] = out;  // the wave's lanes run together: every read of this word is done
        I.hist[(size_t)I.slot * 7 + (j < 5 ? j : j == 5 ? 6 : 5)] = out;
    }
    __syncthreads();
    if (threadIdx.x == 0) I.run[2] = (wave[0][6] / wave[0][5] > I.ratio_dtmax) ? 1.0 : 0.0;
}

template <int LPC, bool MIXED>
__global__ __launch_bounds__(kBlock) void k_flux_ts_slot(int nC, const int* __restrict__ snb,
                                                         const double4* __restrict__ sgeo,
                                                         const double* __restrict__ sdn, const int* __restrict__ sflip,
                                                         const double* __restrict__ q, const double* __restrict__ vol,
                                                         double* __restrict__ res, double* __restrict__ dt,
                                                         double* __restrict__ diag, double* part, FlowConst K,
                                                         double cfl, double cfl_min, float* __restrict__ q32,
                                                         float* __restrict__ diag32, InlineReduce I) {
    flux_ts_slot_body<LPC, MIXED>(xcd_block() * kBlock + (int)threadIdx.x, nC, snb, sgeo, sdn, sflip, q, vol, res,
                                  dt, diag, part + blockIdx.x, (int)gridDim.x, K, cfl, cfl_min, q32, diag32);
    if (I.counter) reduce_last_block((int)gridDim.x, part, I);
}

// The same reduction in two launches, for many blocks.  One workgroup
// reading all the records is bound by the misses one CU keeps in flight
// (42 us for the 23,438 records of 6.0M cells, whatever the batching).
// k_reduce_fold does the threads' folds on many CUs: the fold of thread t
// of k_reduce (records t, t+1024, ... in that order) is shared by
// kFoldLanes consecutive lanes, each loading up to kFoldRecs of its
// records at once; the running values pass from lane to lane in record
// order, so every addition is k_reduce's, in k_reduce's order.  The folds
// go to fold[j * 1024 + t] (j: 5 sums, dt min, dt max) and k_reduce_tree
// finishes them exactly as k_reduce does, so both give the same bits.
constexpr int kFoldLanes = 8, kFoldRecs = 4;
constexpr int kFoldThreads = 256;
__global__ __launch_bounds__(kFoldThreads) void k_reduce_fold(int nblk, const double* __restrict__ part,
                                                              double* __restrict__ fold) {
    const int g = (int)(blockIdx.x * blockDim.x + threadIdx.x);
    const int t = g / kFoldLanes;  // thread of k_reduce whose fold this is
    const int sub = g % kFoldLanes;
    const int lane = (int)threadIdx.x & 63;
    const int src = lane - sub + (sub + kFoldLanes - 1) % kFoldLanes;  // the previous lane of this fold
    const int cnt = t < nblk ? (nblk - 1 - t) / kReduceBlock + 1 : 0;  // records of thread t
    const int maxcnt = (nblk + kReduceBlock - 1) / kReduceBlock;       // the same bound for every lane
    double s[5] = {0.0, 0.0, 0.0, 0.0, 0.0};
    double a = kBIGd, b = 0.0;
    for (int base = 0; base < maxcnt; base += kFoldLanes * kFoldRecs) {
        double r[kFoldRecs][7];
#pragma unroll
        for (int m = 0; m < kFoldRecs; ++m) {
            const int i = base + sub * kFoldRecs + m;
            const int e = min(t + i * kReduceBlock, nblk - 1);
#pragma unroll
            for (int j = 0; j < 7; ++j) r[m][j] = part[(size_t)j * nblk + e];
        }
        // lane `step` adds its records to the running values, which then
        // move on to the next lane (from the last lane back to the first,
        // which starts the next round)
        for (int step = 0; step < kFoldLanes; ++step) {
            if (sub == step) {
#pragma unroll
                for (int m = 0; m < kFoldRecs; ++m) {
                    if (base + sub * kFoldRecs + m >= cnt) break;
#pragma unroll
                    for (int j = 0; j < 5; ++j) s[j] += r[m][j];
                    a = smin(a, r[m][5]);
                    b = smax(b, r[m][6]);
                }
            }
            double ts[5];
#pragma unroll
            for (int j = 0; j < 5; ++j) ts[j] = __shfl(s[j], src, 64);
            const double ta = __shfl(a, src, 64), tb = __shfl(b, src, 64);
            if (sub == (step + 1) % kFoldLanes) {
#pragma unroll
                for (int j = 0; j < 5; ++j) s[j] = ts[j];
                a = ta;
                b = tb;
            }
        }
    }
    if (sub == 0 && t < kReduceBlock) {  // the complete fold is back at the first lane
#pragma unroll
        for (int j = 0; j < 5; ++j) fold[j * kReduceBlock + t] = s[j];
        fold[5 * kReduceBlock + t] = a;
        fold[6 * kReduceBlock + t] = b;
    }
}
__global__ __launch_bounds__(kReduceBlock) void k_reduce_tree(const double* __restrict__ fold, double* __restrict__ run,
                                                        double* __restrict__ hist, int slot, int mode,
                                                        double ratio_dtmax) {
    const int t = (int)threadIdx.x;
    double s[5];
#pragma unroll
    for (int j = 0; j < 5; ++j) s[j] = (mode & 1) ? fold[j * kReduceBlock + t] : 0.0;
    const double a = (mode & 2) ? fold[5 * kReduceBlock + t] : kBIGd;
    const double b = (mode & 2) ? fold[6 * kReduceBlock + t] : 0.0;
    reduce_finish(s, a, b, run, hist, slot, mode, ratio_dtmax);
}

// ---------------------------------------------------------------------------
// Node values (CompNodeVar3D_dist, cal_gradient.cpp:1922-2372): each node
// sums its weighted contributions in the reference's order, then divides by
// WeightNode + TINY.
// Entries are stored per wave of 64 consecutive nodes, entry-major
// (entry k of the wave's lane i at ell_off[w] + 64k + i, padded to the
// wave's largest count), so every entry load of a wave is one coalesced
// 512-byte row; each node still adds its own entries in its order.
template <typename R>
__device__ __forceinline__ void node_body(int p, int w, int nN, const int* __restrict__ nlo,
                                          const int* __restrict__ ell_off, const int2* __restrict__ ell_ab,
                                          const R* __restrict__ ell_w, const double* __restrict__ nden,
                                          const double* __restrict__ q, R* __restrict__ qn) {
    const int lane = (int)threadIdx.x & 63;
    const int e0 = ell_off[w];
    const int K = (ell_off[w + 1] - e0) / 64;  // wave-uniform trip count
    const int cnt = p < nN ? nlo[p + 1] - nlo[p] : 0;
    R acc[5] = {R(0), R(0), R(0), R(0), R(0)};
    // entries in groups of U: the gathers of a group are issued together,
    // then added in entry order
    constexpr int U = 6;
    for (int k = 0; k < K; k += U) {
        int2 ab[U];
        R wt[U], qa[U][5];
#pragma unroll
        for (int i = 0; i < U; ++i) {
            const int kk = (k + i < K) ? k + i : k;
            ab[i] = ell_ab[(size_t)e0 + (size_t)kk * 64 + lane];
            wt[i] = ell_w[(size_t)e0 + (size_t)kk * 64 + lane];
        }
#pragma unroll
        for (int i = 0; i < U; ++i)
#pragma unroll
            for (int j = 0; j < 5; ++j) qa[i][j] = (R)q[(size_t)ab[i].x * 5 + j];
#pragma unroll
        for (int i = 0; i < U; ++i) {
            if (k + i >= cnt) break;
            if (ab[i].y < 0) {
#pragma unroll
                for (int j = 0; j < 5; ++j) acc[j] += qa[i][j] * wt[i];
            } else {
#pragma unroll
                for (int j = 0; j < 5; ++j) {
                    R fq = qa[i][j] + (R)q[(size_t)ab[i].y * 5 + j];
                    fq *= R(0.5);
                    acc[j] += fq * wt[i];
                }
            }
        }
    }
    if (p >= nN) return;
    const R d = (R)nden[p];
#pragma unroll
    for (int j = 0; j < 5; ++j) qn[(size_t)p * 5 + j] = acc[j] / d;
}

template <typename R>
__global__ __launch_bounds__(kBlock) void k_node(int nN, const int* __restrict__ nlo, const int* __restrict__ ell_off,
                                                 const int2* __restrict__ ell_ab, const R* __restrict__ ell_w,
                                                 const double* __restrict__ nden, const double* __restrict__ q,
                                                 R* __restrict__ qn) {
    const int lb = xcd_block();
    node_body<R>(lb * kBlock + (int)threadIdx.x, lb * (kBlock / 64) + (int)threadIdx.x / 64, nN, nlo, ell_off, ell_ab,
                 ell_w, nden, q, qn);
}

// Symmetry-plane velocity projection of the node values (cal_gradient.cpp:2332-2360).
template <typename R>
__global__ void k_node_symm(int nsym, const int* __restrict__ sym_node, const double* __restrict__ sym_n,
                            R* __restrict__ qn) {
    const int s = blockIdx.x * blockDim.x + threadIdx.x;
    if (s >= nsym) return;
    const size_t p = (size_t)sym_node[s] * 5;
    const R xs = (R)sym_n[3 * s], ys = (R)sym_n[3 * s + 1], zs = (R)sym_n[3 * s + 2];
    const R un = qn[p + 1], vn = qn[p + 2], wn = qn[p + 3];
    const R vv = un * xs + vn * ys + wn * zs;
    qn[p + 1] = un - vv * xs;
    qn[p + 2] = vn - vv * ys;
    qn[p + 3] = wn - vv * zs;
}

// Green-Gauss gradient (CompGradientQ_Gauss_Node, cal_gradient.cpp:1740-1795,
// 1889-1897): face values from the node values (interior faces, SYMM and
// INTERFACE boundary faces) or the face-centre average of cell and ghost;
// outputs in the reference's per-variable blocks of nC+nB.
template <int MAXF, typename R>
__device__ __forceinline__ void grad_body(int c, int nC, int n, const int* __restrict__ cfo,
                                          const int* __restrict__ cf, const int2* __restrict__ fcell,
                                          const typename Real<R>::vec4* __restrict__ fgeo,
                                          const int* __restrict__ fno, const int* __restrict__ fn,
                                          const int* __restrict__ btype, const double* __restrict__ q,
                                          const R* __restrict__ qn, const double* __restrict__ vol,
                                          R* __restrict__ gx, R* __restrict__ gy, R* __restrict__ gz) {
    if (c >= nC) return;
    R ax[5] = {R(0), R(0), R(0), R(0), R(0)}, ay[5] = {R(0), R(0), R(0), R(0), R(0)},
      az[5] = {R(0), R(0), R(0), R(0), R(0)};
    int fs[MAXF];
    const int nf = cell_faces<MAXF>(cfo, cf, c, fs);
    int2 cc[MAXF];
    typename Real<R>::vec4 g[MAXF];
    // tetrahedral meshes: every face is a triangle and its nodes sit at 3f
    int tn[MAXF == 4 ? 12 : 1];
#pragma unroll
    for (int s = 0; s < MAXF; ++s) {
        cc[s] = fcell[fs[s]];
        g[s] = fgeo[fs[s]];
        if constexpr (MAXF == 4) {
#pragma unroll
            for (int i = 0; i < 3; ++i) tn[3 * s + i] = fn[3 * fs[s] + i];
        }
    }
#pragma unroll
    for (int s = 0; s < MAXF; ++s) {
        if (s >= nf) break;
        const int f = fs[s];
        R qs[5];
        bool node_mean = true;
        if (cc[s].y >= nC) {
            const int t = btype[cc[s].y - nC];
            node_mean = (t == BC_INTERFACE || t == BC_SYMM);
        }
        if (node_mean) {
            R sum[5] = {R(0), R(0), R(0), R(0), R(0)};
            R cnt;
            if constexpr (MAXF == 4) {
                R v0[5], v1[5], v2[5];
#pragma unroll
                for (int j = 0; j < 5; ++j) {
                    v0[j] = qn[(size_t)tn[3 * s] * 5 + j];
                    v1[j] = qn[(size_t)tn[3 * s + 1] * 5 + j];
                    v2[j] = qn[(size_t)tn[3 * s + 2] * 5 + j];
                }
#pragma unroll
                for (int j = 0; j < 5; ++j) {
                    sum[j] += v0[j];
                    sum[j] += v1[j];
                    sum[j] += v2[j];
                }
                cnt = R(3.0);
            } else {
                const int j0 = fno[f], j1 = fno[f + 1];
                cnt = (R)(j1 - j0);
                for (int m = j0; m < j1; ++m) {
#pragma unroll
                    for (int j = 0; j < 5; ++j) sum[j] += qn[(size_t)fn[m] * 5 + j];
                }
            }
#pragma unroll
            for (int j = 0; j < 5; ++j) qs[j] = sum[j] / cnt;
        } else {
#pragma unroll
            for (int j = 0; j < 5; ++j)
                qs[j] = R(0.5) * ((R)q[(size_t)cc[s].x * 5 + j] + (R)q[(size_t)cc[s].y * 5 + j]);
        }
        const bool minus = (cc[s].y < nC) && (cc[s].y == c);
#pragma unroll
        for (int j = 0; j < 5; ++j) {
            const R sa = qs[j] * g[s].w;
            const R tx = sa * g[s].x, ty = sa * g[s].y, tz = sa * g[s].z;
            if (minus) {
                ax[j] -= tx;
                ay[j] -= ty;
                az[j] -= tz;
            } else {
                ax[j] += tx;
                ay[j] += ty;
                az[j] += tz;
            }
        }
    }
    const R vc = (R)vol[c];
#pragma unroll
    for (int j = 0; j < 5; ++j) {
        gx[(size_t)j * n + c] = ax[j] / vc;
        gy[(size_t)j * n + c] = ay[j] / vc;
        gz[(size_t)j * n + c] = az[j] / vc;
    }
}

// The same gradient for tetrahedral cells, from tables laid out by cell: the
// unit normals pointing away from the cell with their areas (sgeo), the four
// nodes (cnode; node s is the one off the face of slot s) and a word of
// choices (gsel, k_tet_tables).  Subtracting q_f*A*n for a face whose second
// cell this is equals adding q_f*A*(-n) exactly, so the sums are the same
// bits as grad_body's.
//
// Bound: the gathers.  Each node's 5 values are one scattered 40-byte record,
// and a wave's load of 64 of them costs the CU's address and tag units a
// cycle or more per lane, so the cell's four records are gathered once, where
// gathering three per face took twelve.  A face's sum is (a + b) + c with c
// the node its face list names last; which node that is, is the face's choice
// of two bits, taken by selects (a + b commutes; a leading 0 + would only turn
// a sum of negative zeros positive, which the accumulators do anyway).
// Measured alone, before and after: 6.0M cells FP64 650 -> 440 us (1.8 GB of
// compulsory reads and writes, 4.1 TB/s), 2.9M cells FP32 215 -> 134 us; with
// the slot geometry stored slot by slot (slot_at) 397 us, 4.5 TB/s.
template <typename R>
__device__ __forceinline__ void grad_tet_body(int c, int nC, int n, const int* __restrict__ snb,
                                              const typename Real<R>::vec4* __restrict__ sgeo,
                                              const int4* __restrict__ cnode, const unsigned short* __restrict__ gsel,
                                              const double* __restrict__ q, const R* __restrict__ qn,
                                              const double* __restrict__ vol, R* __restrict__ gx,
                                              R* __restrict__ gy, R* __restrict__ gz) {
    if (c >= nC) return;
    const int4 nd = cnode[c];
    const unsigned sel = gsel[c];
    typename Real<R>::vec4 g[4];
#pragma unroll
    for (int s = 0; s < 4; ++s) g[s] = sgeo[slot_at(s, c, nC)];
    R v[4][5];
    load5r(qn + (size_t)nd.x * 5, v[0]);
    load5r(qn + (size_t)nd.y * 5, v[1]);
    load5r(qn + (size_t)nd.z * 5, v[2]);
    load5r(qn + (size_t)nd.w * 5, v[3]);
    const R vc = (R)vol[c];
    R ax[5] = {R(0), R(0), R(0), R(0), R(0)}, ay[5] = {R(0), R(0), R(0), R(0), R(0)},
      az[5] = {R(0), R(0), R(0), R(0), R(0)};
#pragma unroll
    for (int s = 0; s < 4; ++s) {
        constexpr int I[4] = {1, 0, 0, 0}, J[4] = {2, 2, 1, 1}, L[4] = {3, 3, 3, 2};  // the face's nodes
        const R(&vi)[5] = v[I[s]], (&vj)[5] = v[J[s]], (&vk)[5] = v[L[s]];
        const unsigned last = (sel >> (2 * s)) & 3u;
        R qs[5];
#pragma unroll
        for (int j = 0; j < 5; ++j) {
            const R a = last == 0 ? vj[j] : vi[j], b = last == 2 ? vj[j] : vk[j];
            const R e = last == 1 ? vj[j] : vi[j], d = last == 2 ? vk[j] : e;
            qs[j] = ((a + b) + d) / R(3.0);
        }
        if ((sel >> (8 + s)) & 1u) {
            const size_t o = (size_t)snb[(size_t)c * 4 + s] * 5;
#pragma unroll
            for (int j = 0; j < 5; ++j) qs[j] = R(0.5) * ((R)q[(size_t)c * 5 + j] + (R)q[o + j]);
        }
#pragma unroll
        for (int j = 0; j < 5; ++j) {
            const R sa = qs[j] * g[s].w;
            ax[j] += sa * g[s].x;
            ay[j] += sa * g[s].y;
            az[j] += sa * g[s].z;
        }
    }
#pragma unroll
    for (int j = 0; j < 5; ++j) {
        // nothing in the iteration reads the gradient: streaming stores keep
        // its 120 bytes per cell from displacing the sweeps' data in the
        // caches (it runs beside the sweeps' thin tails)
        __builtin_nontemporal_store(ax[j] / vc, &gx[(size_t)j * n + c]);
        __builtin_nontemporal_store(ay[j] / vc, &gy[(size_t)j * n + c]);
        __builtin_nontemporal_store(az[j] / vc, &gz[(size_t)j * n + c]);
    }
}

template <typename R>
__global__ __launch_bounds__(kBlock) void k_grad_tet(int nC, int n, const int* __restrict__ snb,
                                                     const typename Real<R>::vec4* __restrict__ sgeo,
                                                     const int4* __restrict__ cnode, const unsigned short* __restrict__ gsel,
                                                     const double* __restrict__ q, const R* __restrict__ qn,
                                                     const double* __restrict__ vol, R* __restrict__ gx,
                                                     R* __restrict__ gy, R* __restrict__ gz) {
    grad_tet_body<R>(xcd_block() * kBlock + (int)threadIdx.x, nC, n, snb, sgeo, cnode, gsel, q, qn, vol, gx, gy,
                     gz);
}

// k_grad_tet on a small grid whose workgroups claim blocks of kBlock cells:
// workgroup b takes the next unclaimed block of XCD x = b mod 8's span
// (blocks x*span .. (x+1)*span-1, span = nblk / 8, the blocks xcd_block()
// puts on that XCD) from counter x, until the span is done.  The next
// block is claimed while the current one is worked on.  The last workgroup
// to find its span done sets the counter back to zero for the next launch
// (each of the G/8 workgroups of an XCD ends with exactly one claim past
// the span, so the claim returning span + G/8 - 1 is the last).  nblk and
// the grid G are multiples of 8; the counters are 64 ints apart and start
// at zero.
//
// Launched on one workgroup per CU on the context's second stream, beside
// the sweeps' thin tails (6.0M cells, reference order): the gradient takes
// as long as on the full grid (23,440 workgroups), but its waves crowd the
// tails' CUs less (FP64 iteration 3.63 -> 3.57 ms; mixed 3.04 -> 2.99).
// Beside wide sweep levels (the shallower 2/128 order, no thin tail): FP64
// 3.01 -> 2.95 ms, mixed 2.31 -> 2.28; a fixed share per workgroup instead
// of claims left the late-starting workgroups' shares to the end there (the
// gradient 1.40 -> 2.3 ms).
template <typename R>
__global__ __launch_bounds__(kBlock) void k_grad_tet_claim(int nblk, int nC, int n, const int* __restrict__ snb,
                                                           const typename Real<R>::vec4* __restrict__ sgeo,
                                                           const int4* __restrict__ cnode,
                                                           const unsigned short* __restrict__ gsel,
                                                           const double* __restrict__ q, const R* __restrict__ qn,
                                                           const double* __restrict__ vol, R* __restrict__ gx,
                                                           R* __restrict__ gy, R* __restrict__ gz, int* counters) {
    __shared__ int claimed;
    const int x = (int)blockIdx.x % kXcd, per = (int)gridDim.x / kXcd, span = nblk / kXcd;
    int* const ctr = counters + x * 64;
    if (threadIdx.x == 0) claimed = atomicAdd(ctr, 1);
    __syncthreads();
    int k = claimed;
    while (k < span) {
        __syncthreads();  // every thread has read `claimed`
        int next = 0;
        if (threadIdx.x == 0) next = atomicAdd(ctr, 1);
        grad_tet_body<R>((x * span + k) * kBlock + (int)threadIdx.x, nC, n, snb, sgeo, cnode, gsel, q, qn, vol,
                         gx, gy, gz);
        if (threadIdx.x == 0) claimed = next;
        __syncthreads();
        k = claimed;
    }
    if (threadIdx.x == 0 && k == span + per - 1) __hip_atomic_store(ctr, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// The gradient of one iteration and the residual / time step / Diag pass of
// the next, on tetrahedral meshes, in one launch.  One launch instead of
// two lets each wave overlap the gradient's node gathers with the flux
// pass's neighbour gathers (the HBM bytes stay those of the two passes: the
// gathers in between evict the shared slot data).  The gradient feeds
// nothing the next iteration computes, and the two write disjoint arrays,
// so every value is the same as with two launches.
template <bool MIXED, typename R>
__global__ __launch_bounds__(kBlock) void k_grad_flux_ts(int nC, int n, const int* __restrict__ snb,
                                                        const typename Real<R>::vec4* __restrict__ sgeo_r,
                                                        const int4* __restrict__ cnode, const unsigned short* __restrict__ gsel,
                                                        const double* __restrict__ q, const R* __restrict__ qn,
                                                        const double* __restrict__ vol, R* __restrict__ gx,
                                                        R* __restrict__ gy, R* __restrict__ gz,
                                                        const double4* __restrict__ sgeo, const double* __restrict__ sdn,
                                                        const int* __restrict__ sflip, double* __restrict__ res,
                                                        double* __restrict__ dt, double* __restrict__ diag,
                                                        double* __restrict__ part, FlowConst K, double cfl,
                                                        double cfl_min, float* __restrict__ q32,
                                                        float* __restrict__ diag32) {
    const int c = xcd_block() * kBlock + (int)threadIdx.x;
    grad_tet_body<R>(c, nC, n, snb, sgeo_r, cnode, gsel, q, qn, vol, gx, gy, gz);  // no-op past nC
    flux_ts_slot_body<4, MIXED>(c, nC, snb, sgeo, sdn, sflip, q, vol, res, dt, diag,
                                part + blockIdx.x, (int)gridDim.x, K, cfl, cfl_min, q32, diag32);
}

template <int MAXF, typename R>
__global__ __launch_bounds__(kBlock) void k_grad(int nC, int n, const int* __restrict__ cfo,
                                                 const int* __restrict__ cf, const int2* __restrict__ fcell,
                                                 const typename Real<R>::vec4* __restrict__ fgeo,
                                                 const int* __restrict__ fno, const int* __restrict__ fn,
                                                 const int* __restrict__ btype, const double* __restrict__ q,
                                                 const R* __restrict__ qn, const double* __restrict__ vol,
                                                 R* __restrict__ gx, R* __restrict__ gy, R* __restrict__ gz) {
    grad_body<MAXF, R>(xcd_block() * kBlock + (int)threadIdx.x, nC, n, cfo, cf, fcell, fgeo, fno, fn, btype, q, qn,
                       vol, gx, gy, gz);
}
