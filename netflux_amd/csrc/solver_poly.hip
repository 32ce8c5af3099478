// Mixed-element FP64 step on the GPU (poly.hpp).  Per-cell slot layout:
// slot s of cell c is its s-th face in increasing reference face index, and
// every per-slot array is [slot][...][N] so a wave's 64 cells read each
// slot field with one coalesced load.
//   w      [6][N]     NONE, or bit 31 = the cell is the face's j side,
//                     bit 30 = boundary, bits 0-29 = neighbour cell or ghost id
//   ns     [6][N]     the neighbour's slot of the same face
//   geo    [6][6][N]  S of the face (as stored, i -> j), then r of this side
//   U, R   [5][N];  V [5][NT] (cells, then ghosts);  FV [7][5][P], P = max(N,
//   ghosts): reconstructed face values of each slot, and (slot 6) the ghosts
//   of the boundary faces' values;  grad [15][N], psi [5][N]
// A stage is two kernels: sweep A (gradient, min/max, limiter, face values;
// second order only; the CFL steps where asked) and sweep B (flux balance,
// stage update, primvars of the new state, residual sums).  Boundary ghosts
// are formed at the end of the sweep that stores what they depend on, one face
// per lane of the block's first lanes (in launches of their own a step took
// 91.0 against 79.3 us at 12^3, 444 against 437 us at 80^3).  Each follows the CPU solver's loops
// (src/Solver.cpp:54-230, include/Numerics.hpp:86-292) with the same
// operations in the same order; gradient, limiter and R are stored only when
// they are to be exported.
//
// U^n stays in Ua (it is U_old of the next stages), stages write Ub, the last
// one Ua.  Primvars: X of U^n, Y of U1, Z of U2; sweep B of the last stage
// stores X.  The CFL step of the primvars the last stage reads is the next
// step's dt (src/Solver.cpp:248), reduced with the residual by one kernel.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cfloat>
#include <cmath>
#include <cstdio>
#include <cstring>
#include <initializer_list>
#include <map>
#include <memory>
#include <new>
#include <vector>

#include "fp64_math.hpp"
#include "host_pipe.hpp"
#include "physics.hpp"
#include "poly.hpp"

namespace nf {

namespace {
constexpr int PB = 256;
constexpr uint32_t NONE = 0xFFFFFFFFu, SIDE_J = 0x80000000u;
using V3 = Vec3T<double>;

struct PolyDev {
    uint32_t N, NT, G;
    size_t P;  // plane stride of FV
    const uint32_t *w;
    const uint8_t *ns;
    const double *geo, *vol, *dS;
    // boundary faces in device cell order: cell i, its slot, ghost j, S, type
    const uint32_t *bi, *bj;
    const uint8_t *bslot, *bbc;
    const double *bS;
    const uint32_t *boff;  // [blocks + 1] first boundary face of each block's cells
    FarField<double> fs;
    const int *stop;  // kernels return if one of stop[0 .. nstop) is set
    int nstop;
};
constexpr uint32_t BND = 0x40000000u, IDX = 0x3FFFFFFFu;

__device__ __forceinline__ bool stopped(const PolyDev &m) {
    for (int q = 0; q < m.nstop; ++q)
        if (m.stop[q]) return true;
    return false;
}

__device__ __forceinline__ double geo(const PolyDev &m, int s, int q, uint32_t c) {
    return m.geo[((size_t)s * 6 + q) * m.N + c];
}

// sum or minimum over the block in a fixed tree; valid in thread 0
template <bool MIN>
__device__ __forceinline__ double tree(double v, double *sh) {
    sh[threadIdx.x] = v;
    __syncthreads();
    for (int h = PB / 2; h > 0; h >>= 1) {
        if ((int)threadIdx.x < h) {
            const double a = sh[threadIdx.x], b = sh[threadIdx.x + h];
            sh[threadIdx.x] = MIN ? smin(a, b) : a + b;
        }
        __syncthreads();
    }
    return sh[0];
}

// set_constant_ghost_values (src/Solver.cpp:300-330) of boundary face b
__device__ __forceinline__ void ghost_cell(const PolyDev &m, uint32_t b, double *V) {
    const uint32_t i = m.bi[b], j = m.bj[b];
    double vd[5], vg[5];
#pragma unroll
    for (int k = 0; k < 5; ++k) vd[k] = V[k * (size_t)m.NT + i];
    const V3 S = {m.bS[b], m.bS[m.G + b], m.bS[2 * (size_t)m.G + b]};
    ghost_value<double>((int)m.bbc[b], vd, S, m.fs, vg);
#pragma unroll
    for (int k = 0; k < 5; ++k) V[k * (size_t)m.NT + j] = vg[k];
}
// ghost of its reconstructed face state (src/Solver.cpp:210-212)
__device__ __forceinline__ void ghost_face(const PolyDev &m, uint32_t b, double *FV) {
    const uint32_t i = m.bi[b], s = m.bslot[b];
    double vd[5], vg[5];
#pragma unroll
    for (int k = 0; k < 5; ++k) vd[k] = FV[(s * 5 + k) * m.P + i];
    const V3 S = {m.bS[b], m.bS[m.G + b], m.bS[2 * (size_t)m.G + b]};
    ghost_d((int)m.bbc[b], vd, S, m.fs, vg);
#pragma unroll
    for (int k = 0; k < 5; ++k) FV[(30 + k) * m.P + (m.bj[b] - m.N)] = vg[k];
}
// The block's boundary faces, one per lane of its first lanes.  The range is
// loaded at the start of a sweep and kept there by the asm: at its end every
// block would wait for these scalar loads.
struct BndFaces {
    uint32_t b0, b1;
};
__device__ __forceinline__ BndFaces bnd_faces(const PolyDev &m, uint32_t lb) {
    BndFaces r{m.boff[lb], m.boff[lb + 1]};
    asm volatile("" : "+s"(r.b0), "+s"(r.b1));
    return r;
}
template <typename F>
__device__ __forceinline__ void block_ghosts(BndFaces r, F ghost) {
    if (r.b0 == r.b1) return;  // the same for the whole block
    __syncthreads();           // every lane's values are stored
    for (uint32_t b = r.b0 + threadIdx.x; b < r.b1; b += PB) ghost(b);
}

__global__ __launch_bounds__(PB) void k_poly_prim(const double *U, double *V, uint32_t N, uint32_t NT) {
    const uint32_t c = blockIdx.x * PB + threadIdx.x;
    if (c >= N) return;
    double u[5], v[5];
    for (int k = 0; k < 5; ++k) u[k] = U[k * (size_t)N + c];
    cons_to_prim_d(u, v);
    for (int k = 0; k < 5; ++k) V[k * (size_t)NT + c] = v[k];
}

__global__ __launch_bounds__(PB) void k_poly_ghost(PolyDev m, double *V) {
    const uint32_t b = blockIdx.x * PB + threadIdx.x;
    if (b < m.G && !stopped(m)) ghost_cell(m, b, V);
}

// calc_timestep of a cell (src/Solver.cpp:232-274)
__device__ __forceinline__ double cell_step(const PolyDev &m, uint32_t c, const double *v, double CFL) {
    const double cs = sound_speed_prim(v);
    const double sx = (std::fabs(v[1]) + cs) * m.dS[c];
    const double sy = (std::fabs(v[2]) + cs) * m.dS[(size_t)m.N + c];
    const double sz = (std::fabs(v[3]) + cs) * m.dS[2 * (size_t)m.N + c];
    return CFL * m.vol[c] / ((sx + sy) + sz);
}

struct SweepA {
    const double *V;
    int limiter;
    double *FV;
    double *grad, *psi;  // exported, or null
    double CFL;
    double *dt_part, *dt_cell;  // per-block minimum of the cells' CFL steps, the steps themselves; or null
};

// Green-Gauss (Numerics.hpp:86-128), max/min (:253-292), Barth (:148-250)
// and the reconstructed face values (Solver.hpp:81-112) of one cell.  The
// gradient terms divide by the cell volume through one refined reciprocal
// (rdiv: the quotient of a plain division), the Barth limiter takes two
// divisions per variable over the largest positive and most negative face
// Delta_2 (barth_psi_hilo), and the face-centroid vectors are read once.
// Bound by HBM: 600 bytes per hexahedron (288 of geometry, 240 of face values).
__global__ __launch_bounds__(PB) void k_poly_sweepA(PolyDev m, SweepA a) {
    __shared__ double sh[PB];
    const uint32_t lb = logical_block(blockIdx.x, gridDim.x, 1);  // XCD-contiguous
    const BndFaces br = bnd_faces(m, lb);
    if (stopped(m)) return;  // the same for every thread of the block
    const bool live = lb * PB + threadIdx.x < m.N;
    const uint32_t c = live ? lb * PB + threadIdx.x : m.N - 1;
    const size_t NT = m.NT, N = m.N;
    const double *V = a.V;
    double vc[5];
#pragma unroll
    for (int k = 0; k < 5; ++k) vc[k] = V[k * NT + c];
    const Rcp ivol = rcp_of(m.vol[c]);
    uint32_t w[6];
    int nfc = 0;
#pragma unroll
    for (int s = 0; s < 6; ++s) {
        w[s] = m.w[s * N + c];
        if (w[s] != NONE) nfc = s + 1;
    }
    double g[15];
#pragma unroll
    for (int q = 0; q < 15; ++q) g[q] = 0.0;
    double vmax[5], vmin[5];
#pragma unroll
    for (int k = 0; k < 5; ++k) vmax[k] = vmin[k] = vc[k];
#pragma unroll
    for (int s = 0; s < 6; ++s) {
        // loads before the slot test (absent slots read the cell's own
        // entries, in bounds), so that later faces' loads need not wait
        const uint32_t n = s < nfc ? (w[s] & IDX) : c;
        const double Sx = geo(m, s, 0, c), Sy = geo(m, s, 1, c), Sz = geo(m, s, 2, c);
        double vnb[5];
#pragma unroll
        for (int k = 0; k < 5; ++k) vnb[k] = V[k * NT + n];
        if (s >= nfc) break;
        // cell j subtracts the term: the sign goes into S, exactly (0.5 (v_i +
        // v_j) does not depend on the side); maxima of {v, v_j} as in the
        // tetrahedral sweep.  With selects by side and both signs' sums a step of
        // 12^3 / 48^3 / 96^3 hexahedra took 79.0 / 124.5 / 769 us, so 76.8 /
        // 120.3 / 766: it is the arithmetic of small meshes, large ones are
        // bound by the gathers.
        const uint32_t mneg = (w[s] & SIDE_J) ? 0x80000000u : 0u;
        const double Tx = flip(Sx, mneg), Ty = flip(Sy, mneg), Tz = flip(Sz, mneg);
#pragma unroll
        for (int k = 0; k < 5; ++k) {
            const double uf = 0.5 * (vc[k] + vnb[k]);
            g[k] += rdiv(uf * Tx, ivol);
            g[k + 5] += rdiv(uf * Ty, ivol);
            g[k + 10] += rdiv(uf * Tz, ivol);
            vmax[k] = dmax(vmax[k], vnb[k]);
            vmin[k] = dmin(vmin[k], vnb[k]);
        }
    }
    V3d r[6];
#pragma unroll
    for (int s = 0; s < 6; ++s)
        r[s] = s < nfc ? V3d{geo(m, s, 3, c), geo(m, s, 4, c), geo(m, s, 5, c)} : V3d{0.0, 0.0, 0.0};
    double ps[5];
#pragma unroll
    for (int k = 0; k < 5; ++k) {
        ps[k] = 1.0;  // SolverData.cpp:17 (no limiter)
        if (a.limiter) {
            double hi = 0.0, lo = 0.0;
#pragma unroll
            for (int s = 0; s < 6; ++s) {
                if (s >= nfc) break;
                const double D = (g[k] * r[s].x + g[k + 5] * r[s].y) + g[k + 10] * r[s].z;
                hi = dmax(hi, D);
                lo = dmin(lo, D);
            }
            ps[k] = barth_psi_hilo(hi, lo, vmax[k], vmin[k], vc[k]);
        }
    }
    if (live) {
#pragma unroll
        for (int s = 0; s < 6; ++s) {
            if (s >= nfc) break;
#pragma unroll
            for (int k = 0; k < 5; ++k) {
                const double D = (g[k] * r[s].x + g[k + 5] * r[s].y) + g[k + 10] * r[s].z;
                a.FV[(s * 5 + k) * m.P + c] = vc[k] + ps[k] * D;
            }
        }
        if (a.grad) {
            for (int q = 0; q < 15; ++q) a.grad[q * N + c] = g[q];
            for (int k = 0; k < 5; ++k) a.psi[k * N + c] = ps[k];
        }
    }
    block_ghosts(br, [&](uint32_t b) { ghost_face(m, b, a.FV); });
    if (a.dt_part) {
        const double x = cell_step(m, c, vc, a.CFL);
        if (a.dt_cell && live) a.dt_cell[c] = x;  // local time stepping: each cell's own CFL step
        const double t = tree<true>(live ? smin(DBL_MAX, x) : DBL_MAX, sh);
        if (threadIdx.x == 0) a.dt_part[lb] = t;
    }
}

struct SweepB {
    const double *V, *FV;  // FV == nullptr: first order (face values = cell values)
    const double *U, *Uo;  // state entering the stage, U^n
    double *Uout;          // (may alias either)
    double *Vout;          // primvars and cell ghosts of Uout, or null
    double *R;             // stored when not null
    double *res_part;      // per-block sums of R_rho^2, or null
    int *bad;              // cells with a non-finite flux balance are counted, or null
    int flux;              // 0 Rusanov, 1 HLLC
    int kind;              // 0: U + dt/vol R, 1: RK3 stage 2, 2: RK3 stage 3, -1: no update
    double dt;
    const double *dtp;    // the step's dt in device memory (device-resident run), or null: dt
    const double *dtc;    // per-cell steps (local time stepping), or null
    const int *zero_old;  // U_old counts as zero while set (the first step)
};

// the stage update (src/Solver.cpp:83-133) of a cell
__device__ __forceinline__ void stage_update(const PolyDev &m, const SweepB &a, uint32_t c, bool live, const double *R) {
    const size_t N = m.N;
    const double vol = m.vol[c], dt = a.dtc ? a.dtc[c] : (a.dtp ? *a.dtp : a.dt);
    const bool zero = a.kind > 0 && *a.zero_old;
    double un[5], v[5];
#pragma unroll
    for (int k = 0; k < 5; ++k) {
        const double u = a.U[k * N + c], uo = a.kind > 0 && !zero ? a.Uo[k * N + c] : 0.0;
        if (a.kind == 0) un[k] = u + dt / vol * R[k];
        else if (a.kind == 1) un[k] = 3.0 / 4.0 * uo + 1.0 / 4.0 * u + 1.0 / 4.0 * dt / vol * R[k];
        else un[k] = 1.0 / 3.0 * uo + 2.0 / 3.0 * u + 2.0 / 3.0 * dt / vol * R[k];
    }
    if (live) {
#pragma unroll
        for (int k = 0; k < 5; ++k) a.Uout[k * N + c] = un[k];
        if (a.Vout) {
            cons_to_prim_d(un, v);
#pragma unroll
            for (int k = 0; k < 5; ++k) a.Vout[k * (size_t)m.NT + c] = v[k];
        }
    }
}

// inviscid_fluxes (src/Solver.cpp:144-230) gathered per cell, the validity
// check (src/SolverData.cpp:66-79) and the stage update.  Bound by HBM: about
// 570 bytes per hexahedron (144 of face vectors, 240 of face values, which
// the neighbours' reads find in L2).  The primvars stored here instead of in
// a pass over U, U^n left in place instead of copied to U_old, the residual
// and dt partials formed where their inputs are in registers: a step of 7
// launches instead of 17, 102 -> 79 us at 12^3, 234 -> 216 at 64^3, 804 -> 775
// at 96^3 hexahedra.
__global__ __launch_bounds__(PB) void k_poly_sweepB(PolyDev m, SweepB a) {
    __shared__ double sh[PB];
    const uint32_t lb = logical_block(blockIdx.x, gridDim.x, 1);  // XCD-contiguous
    const BndFaces br = bnd_faces(m, lb);
    if (stopped(m)) return;  // the same for every thread of the block
    const bool live = lb * PB + threadIdx.x < m.N;
    const uint32_t c = live ? lb * PB + threadIdx.x : m.N - 1;
    const size_t NT = m.NT, N = m.N;
    double R[5] = {0.0, 0.0, 0.0, 0.0, 0.0};
    // slot words first, then every face's loads without waiting on them;
    // absent slots read the cell's own entries (in bounds)
    uint32_t w[6], qs[6];
    int nfc = 0;
#pragma unroll
    for (int s = 0; s < 6; ++s) {
        w[s] = m.w[s * N + c];
        qs[s] = m.ns[s * N + c];
    }
#pragma unroll
    for (int s = 0; s < 6; ++s)
        if (w[s] != NONE) nfc = s + 1;
#pragma unroll
    for (int s = 0; s < 6; ++s) {
        // the other side: the neighbour's slot of this face, or the ghost
        const uint32_t id = w[s] & IDX;
        const bool bnd = s < nfc && (w[s] & BND);
        const uint32_t n = s < nfc ? (bnd && a.FV ? id - m.N : id) : c, q = s < nfc ? (bnd ? 6u : qs[s]) : (uint32_t)s;
        const V3 S = {geo(m, s, 0, c), geo(m, s, 1, c), geo(m, s, 2, c)};
        double own[5], oth[5], UO[5], UN[5], F[5];
#pragma unroll
        for (int k = 0; k < 5; ++k) own[k] = a.FV ? a.FV[(s * 5 + k) * m.P + c] : a.V[k * NT + c];
#pragma unroll
        for (int k = 0; k < 5; ++k) oth[k] = a.FV ? a.FV[(q * 5 + k) * m.P + n] : a.V[k * NT + n];
        if (s >= nfc) break;
        const bool sj = (w[s] & SIDE_J) != 0;
        prim_to_cons(own, UO);
        prim_to_cons(oth, UN);
        if (a.flux == 1) {
            double ul[5], ur[5];  // the face's i and j sides
#pragma unroll
            for (int k = 0; k < 5; ++k) ul[k] = sj ? UN[k] : UO[k], ur[k] = sj ? UO[k] : UN[k];
            hllc_d(ul, ur, S, F);
        } else {
            rusanov_side(UO, UN, S, sj ? 0x80000000u : 0u, F);  // = rusanov(ul, ur, S)
        }
        if (sj) {
            for (int k = 0; k < 5; ++k) R[k] += F[k];
        } else {
            for (int k = 0; k < 5; ++k) R[k] -= F[k];
        }
    }
    bool ok = true;
#pragma unroll
    for (int k = 0; k < 5; ++k) {
        if (a.R && live) a.R[k * N + c] = R[k];
        ok = ok && std::isfinite(R[k]);
    }
    if (!ok && a.bad && live) atomicAdd(a.bad, 1);
    if (a.kind >= 0) {
        stage_update(m, a, c, live, R);
        if (a.Vout) block_ghosts(br, [&](uint32_t b) { ghost_cell(m, b, a.Vout); });
    }
    if (a.res_part) {
        const double s = tree<false>(live ? R[0] * R[0] : 0.0, sh);
        if (threadIdx.x == 0) a.res_part[lb] = s;
    }
}

// the stage update alone, where the flux balance R had no bad cell (m.stop
// covers its counter)
__global__ __launch_bounds__(PB) void k_poly_update(PolyDev m, SweepB a) {
    const uint32_t lb = blockIdx.x;
    const BndFaces br = bnd_faces(m, lb);
    if (stopped(m)) return;
    const bool live = lb * PB + threadIdx.x < m.N;
    const uint32_t c = live ? lb * PB + threadIdx.x : m.N - 1;
    double R[5];
#pragma unroll
    for (int k = 0; k < 5; ++k) R[k] = a.R[k * (size_t)m.N + c];
    stage_update(m, a, c, live, R);
    if (a.Vout) block_ghosts(br, [&](uint32_t b) { ghost_cell(m, b, a.Vout); });
}

// per-block minimum of the cell steps of the primvars V
__global__ __launch_bounds__(PB) void k_poly_dt(PolyDev m, const double *V, double CFL, double *part, double *dt_cell) {
    __shared__ double sh[PB];
    if (stopped(m)) return;  // the same for every thread of the block
    const uint32_t c = blockIdx.x * PB + threadIdx.x;
    double t = DBL_MAX;
    if (c < m.N) {
        double v[5];
        for (int k = 0; k < 5; ++k) v[k] = V[k * (size_t)m.NT + c];
        const double x = cell_step(m, c, v, CFL);
        if (dt_cell) dt_cell[c] = x;
        t = smin(t, x);
    }
    t = tree<true>(t, sh);
    if (threadIdx.x == 0) part[blockIdx.x] = t;
}

// Run state on the device: flags [0] stop, [1] converged, [2] invalid dt, [3]
// steps completed (the index of the step in progress), so a graph of several
// steps can be replayed unchanged.
struct RunDev {
    int *flags;            // null: a step driven from the host
    double *dtdev;         // the next step's dt
    double *dts, *hres;    // per step of a run: dt, residual
    double *runp;          // {drop, ref}: ref is the first residual since the state was set, or negative when this
                           // run's first step is that residual (a first residual of 0 never converges)
    int *zero_old;         // U_old counts as zero (before the first step)
    int *bad;              // [3] bad cells of each stage (checked steps)
    double *host;          // residual, dt, bad[3]: pinned, or where there was none dev_res
};

// partials in a fixed order: each thread a strided sum (or minimum), then a tree
template <bool MIN>
__device__ __forceinline__ double all_parts(const double *part, uint32_t nb, double *sh) {
    constexpr int Q = 8;  // loads in flight
    double v = MIN ? DBL_MAX : 0.0;
    for (uint32_t i0 = threadIdx.x; i0 < nb; i0 += Q * PB) {
        double x[Q];
#pragma unroll
        for (int q = 0; q < Q; ++q) x[q] = part[i0 + q * PB < nb ? i0 + q * PB : i0];
#pragma unroll
        for (int q = 0; q < Q; ++q)
            if (i0 + q * PB < nb) v = MIN ? smin(v, x[q]) : v + x[q];
    }
    return tree<MIN>(v, sh);
}
__device__ __forceinline__ bool valid_dt(double dt) { return (dt - dt == 0.0) && dt > 0.0; }

// dt of the first step: minimum of the block partials, or the one in place;
// and a run's flags, drop and reference
__global__ __launch_bounds__(PB) void k_poly_begin(RunDev r, const double *part, uint32_t nb, double drop, double ref) {
    __shared__ double sh[PB];
    double dt = 0.0;
    if (part) dt = all_parts<true>(part, nb, sh);
    if (threadIdx.x) return;
    if (part) r.dtdev[0] = dt;
    else dt = r.dtdev[0];
    r.host[1] = dt;
    if (!r.flags) return;
    const bool ok = valid_dt(dt);
    r.flags[0] = r.flags[2] = ok ? 0 : 1;
    r.flags[1] = r.flags[3] = 0;
    r.runp[0] = drop;
    r.runp[1] = ref;
    r.dts[0] = dt;
}

// The end of a step, one block: the residual (sum of the block partials, its
// square root), the drop test, and the next step's dt with its test.
__global__ __launch_bounds__(PB) void k_poly_end(RunDev r, const double *res_part, const double *dt_part, uint32_t nb) {
    __shared__ double sh[2][PB];
    if (r.flags && r.flags[0]) return;
    const double s = all_parts<false>(res_part, nb, sh[0]), dt = all_parts<true>(dt_part, nb, sh[1]);
    if (threadIdx.x) return;
    const double res = sqrt(s);
    if (!r.flags) {
        r.host[0] = res;
        r.host[1] = dt;
        bool bad = false;
        for (int q = 0; q < 3; ++q) {
            bad = bad || r.bad[q];
            r.host[2 + q] = r.bad[q];
            r.bad[q] = 0;
        }
        if (bad) return;
        *r.zero_old = 0;
        r.dtdev[0] = dt;
        return;
    }
    const int k = r.flags[3];
    r.hres[k] = res;
    r.flags[3] = k + 1;
    *r.zero_old = 0;
    r.dtdev[0] = dt;
    r.dts[k + 1] = dt;
    const double drop = r.runp[0], ref = r.runp[1];
    const double r0 = ref >= 0.0 ? ref : r.hres[0];
    if (drop > 0.0 && r0 > 0.0 && res / r0 <= drop) {
        r.flags[1] = 1;
        r.flags[0] = 1;
    }
    if (!valid_dt(dt)) {  // an error only if a further step was asked for
        r.flags[2] = 1;
        r.flags[0] = 1;
    }
}

__global__ void k_poly_set(int *p, int v) { *p = v; }

// reference-order AoS [N][cols] <-> [cols][N] in device cell order
__global__ __launch_bounds__(PB) void k_poly_aos_in(const double *aos, const uint32_t *perm, double *soa, uint32_t N,
                                                    int cols) {
    const uint32_t d = blockIdx.x * PB + threadIdx.x;
    if (d >= N) return;
    const size_t r = (size_t)cols * perm[d];
    for (int k = 0; k < cols; ++k) soa[k * (size_t)N + d] = aos[r + k];
}
__global__ __launch_bounds__(PB) void k_poly_aos_out(const double *soa, const uint32_t *perm, double *aos, uint32_t N,
                                                     int cols) {
    const uint32_t d = blockIdx.x * PB + threadIdx.x;
    if (d >= N) return;
    const size_t r = (size_t)cols * perm[d];
    for (int k = 0; k < cols; ++k) aos[r + k] = soa[k * (size_t)N + d];
}
struct Five {
    double v[5];
};
__global__ __launch_bounds__(PB) void k_poly_fill(double *U, Five u, double *X, Five x, size_t NT, uint32_t n) {
    const uint32_t q = blockIdx.x * PB + threadIdx.x;
    if (q >= n) return;
    for (int k = 0; k < 5; ++k) {
        U[k * (size_t)n + q] = u.v[k];
        X[k * NT + q] = x.v[k];
    }
}
}  // namespace

struct PolyPath {
    hipStream_t st = nullptr;
    nf_params prm{};
    PolyDev m{};
    nf_fv_sizes sizes{};
    double *Ua = nullptr, *Ub = nullptr, *X = nullptr, *Y = nullptr, *Z = nullptr, *FV = nullptr;
    double *grad = nullptr, *psi = nullptr, *R = nullptr, *dt_part = nullptr, *res_part = nullptr;
    double *dtc = nullptr;  // [N] per-cell steps (local time stepping)
    RunDev run{};           // run.flags: set for the kernels of a device-resident run only
    double *dev_res = nullptr, res[5] = {};  // results without pinned memory, and on the host (read_results)
    int *flags = nullptr;
    int64_t run_cap = 0;
    uint32_t *boff = nullptr;
    hipGraphExec_t graph = nullptr;  // check_every steps of nf_run, captured once per K and buffers
    int graph_K = 0;
    bool aux_valid = false;  // grad / psi / R hold nf_eval_flux_balance of the current state
    // run state since the last set_state / set_freestream
    bool split = false;      // a failed stage left the state in Ub (U_old still in Ua)
    bool x_prim = false;     // X holds prim of the state, ghosts included
    bool dt_valid = false;   // dtdev (and dt) hold the next step's dt; else it is that of X
    bool old_zero = false;   // U_old counts as zero
    double dt = 0.0;
    // kernel timing (nf_time_kernels): HIP events around each launch
    bool timing = false;
    std::vector<std::pair<const char *, std::pair<hipEvent_t, hipEvent_t>>> pending;
    std::map<std::string, std::pair<double, int>> ktime;
    std::vector<uint32_t> perm;  // device cell -> reference cell
    uint32_t *perm_dev = nullptr;  // the same on the device (made on first state transfer)
    HostPipe *pipe = nullptr;      // the context's: large arrays across the boundary
    double *stage = nullptr;       // [15][N] AoS staging of state and field transfers
    std::vector<double> hist;    // residual norm of each step (flux balance of U^n)
    double time = 0.0;
    bool converged = false;
    std::vector<void *> owned;
    double *state() const { return split ? Ub : Ua; }
    bool second() const { return prm.spatial_order == NF_SECOND_ORDER; }
    bool rk3() const { return prm.time_scheme == NF_TVD_RK3; }
    uint32_t blocks() const { return (m.N + PB - 1) / PB; }
    ~PolyPath() {
        if (st) (void)hipStreamSynchronize(st);
        if (graph) (void)hipGraphExecDestroy(graph);
        for (void *p : owned) (void)hipFree(p);
        if (run.host && run.host != dev_res) PinnedPool::get().give_record(run.host);
    }
};

namespace {
#define PHIP(expr)                                                                  \
    do {                                                                            \
        hipError_t e_ = (expr);                                                     \
        if (e_ != hipSuccess) {                                                     \
            (void)hipGetLastError(); /* not reported again by the next call */      \
            err = std::string(#expr) + ": " + hipGetErrorString(e_);                \
            return NF_E_HIP;                                                        \
        }                                                                           \
    } while (0)

template <typename T> int alloc(PolyPath *P, T **p, size_t n, std::string &err) {
    PHIP(hipMalloc((void **)p, std::max<size_t>(n, 1) * sizeof(T)));
    P->owned.push_back(*p);
    return NF_OK;
}
// several arrays in one allocation (a context of 2k cells has 28 arrays, and
// as many calls were a tenth of its creation)
struct Slot {
    void **p;
    size_t bytes;
    template <typename T> Slot(T **q, size_t n) : p((void **)q), bytes((std::max<size_t>(n, 1) * sizeof(T) + 255) & ~(size_t)255) {}
};
int alloc_all(PolyPath *P, std::initializer_list<Slot> slots, std::string &err) {
    size_t n = 0;
    for (const Slot &q : slots) n += q.bytes;
    char *base = nullptr;
    int rc;
    if ((rc = alloc(P, &base, n, err))) return rc;
    for (const Slot &q : slots) {
        *q.p = base;
        base += q.bytes;
    }
    return NF_OK;
}
template <typename T> int upload(T *dst, const std::vector<T> &src, std::string &err) {
    PHIP(hipMemcpy(dst, src.data(), src.size() * sizeof(T), hipMemcpyHostToDevice));
    return NF_OK;
}
dim3 grid(size_t n) { return dim3((unsigned)((n + PB - 1) / PB)); }

// AoS [N][cols] in reference cell order <-> SoA [cols][N] in device order
// Reference-order AoS [N][cols] crosses as is; the device reorders it into
// [cols][N] in device cell order (and back), the host never touches it.
int ensure_stage(PolyPath *P, std::string &err) {
    if (P->stage) return NF_OK;
    int rc;
    if ((rc = alloc(P, &P->perm_dev, P->m.N, err)) || (rc = alloc(P, &P->stage, 15 * (size_t)P->m.N, err))) return rc;
    PHIP(hipMemcpy(P->perm_dev, P->perm.data(), (size_t)P->m.N * sizeof(uint32_t), hipMemcpyHostToDevice));
    return NF_OK;
}
int put_soa(PolyPath *P, double *dst, const double *aos, int cols, std::string &err) {
    const uint32_t N = P->m.N;
    int rc;
    if ((rc = ensure_stage(P, err))) return rc;
    PHIP(P->pipe->up(P->stage, aos, (size_t)cols * N * 8, P->st));
    hipLaunchKernelGGL(k_poly_aos_in, grid(N), dim3(PB), 0, P->st, (const double *)P->stage,
                       (const uint32_t *)P->perm_dev, dst, N, cols);
    PHIP(hipGetLastError());
    PHIP(hipStreamSynchronize(P->st));
    return NF_OK;
}
int get_soa(PolyPath *P, const double *src, int cols, double *aos, std::string &err) {
    const uint32_t N = P->m.N;
    int rc;
    if ((rc = ensure_stage(P, err))) return rc;
    hipLaunchKernelGGL(k_poly_aos_out, grid(N), dim3(PB), 0, P->st, src, (const uint32_t *)P->perm_dev, P->stage,
                       N, cols);
    PHIP(hipGetLastError());
    PHIP(P->pipe->down(aos, P->stage, (size_t)cols * N * 8, P->st));
    return NF_OK;
}

int tstart(PolyPath *P, hipEvent_t *e, std::string &err) {
    if (!P->timing) return NF_OK;
    PHIP(hipEventCreate(e));
    PHIP(hipEventRecord(*e, P->st));
    return NF_OK;
}
int tstop(PolyPath *P, const char *name, hipEvent_t e0, std::string &err) {
    if (!P->timing) return NF_OK;
    hipEvent_t e1;
    PHIP(hipEventCreate(&e1));
    PHIP(hipEventRecord(e1, P->st));
    P->pending.push_back({name, {e0, e1}});
    return NF_OK;
}
int tflush(PolyPath *P, std::string &err) {
    PHIP(hipStreamSynchronize(P->st));
    for (auto &q : P->pending) {
        float ms = 0.0f;
        PHIP(hipEventElapsedTime(&ms, q.second.first, q.second.second));
        auto &slot = P->ktime[q.first];
        slot.first += ms;
        slot.second += 1;
        (void)hipEventDestroy(q.second.first);
        (void)hipEventDestroy(q.second.second);
    }
    P->pending.clear();
    return NF_OK;
}

// primvars of U into V, cell ghosts included.  timed: one launch each in the
// kernel timing
int prim_of(PolyPath *P, const double *U, double *V, bool timed, std::string &err) {
    int rc;
    hipEvent_t e = nullptr;
    if (timed && (rc = tstart(P, &e, err))) return rc;
    hipLaunchKernelGGL(k_poly_prim, grid(P->m.N), dim3(PB), 0, P->st, U, V, P->m.N, P->m.NT);
    if (timed && ((rc = tstop(P, "poly_prim", e, err)) || (rc = tstart(P, &e, err)))) return rc;
    if (P->m.G) {
        PolyDev m = P->m;
        m.nstop = 0;
        hipLaunchKernelGGL(k_poly_ghost, grid(m.G), dim3(PB), 0, P->st, m, V);
    }
    if (timed && (rc = tstop(P, "poly_ghost", e, err))) return rc;
    PHIP(hipGetLastError());
    return NF_OK;
}

// X = prim of the state (where it is not already)
int ensure_x(PolyPath *P, std::string &err) {
    if (P->x_prim) return NF_OK;
    const int rc = prim_of(P, P->state(), P->X, false, err);
    P->x_prim = rc == NF_OK;
    return rc;
}

// one flux balance from the primvars V: sweep A for second order, sweep B.
// a: what sweep B does with it; dt_part, dt_cell: the CFL steps of V too
int flux_balance(PolyPath *P, const PolyDev &m, const double *V, SweepB a, bool aux, double *dt_part, double *dt_cell,
                 std::string &err) {
    int rc;
    hipEvent_t e = nullptr;
    if (P->second()) {
        if ((rc = tstart(P, &e, err))) return rc;
        const SweepA x{V, P->prm.limiter != NF_LIMITER_NONE ? 1 : 0, P->FV, aux ? P->grad : nullptr,
                       aux ? P->psi : nullptr, P->prm.CFL, dt_part, dt_cell};
        hipLaunchKernelGGL(k_poly_sweepA, dim3(P->blocks()), dim3(PB), 0, P->st, m, x);
        if ((rc = tstop(P, "poly_sweepA", e, err))) return rc;
    } else if (dt_part) {
        hipLaunchKernelGGL(k_poly_dt, dim3(P->blocks()), dim3(PB), 0, P->st, m, V, P->prm.CFL, dt_part, dt_cell);
    }
    a.V = V;
    a.FV = P->second() ? P->FV : nullptr;
    a.flux = P->prm.inv_flux_scheme == NF_FLUX_HLLC ? 1 : 0;
    a.zero_old = P->run.zero_old;
    if ((rc = tstart(P, &e, err))) return rc;
    hipLaunchKernelGGL(k_poly_sweepB, dim3(P->blocks()), dim3(PB), 0, P->st, m, a);
    PHIP(hipGetLastError());
    return tstop(P, "poly_sweepB", e, err);
}

// The stages of one step (Solver::step, src/Solver.cpp:34-52, 83-133): dt
// given, or (device-resident run) from dtdev, with kernels that return once
// flags[0] is set.  With the flux-balance check (host-driven steps) an update
// runs only where no cell of its or an earlier stage was bad.  Leaves the
// partials of the residual and of the next dt.
int stages(PolyPath *P, bool on_device, double dt, std::string &err) {
    const bool rk3 = P->rk3(), second = P->second(), lts = P->prm.local_time_step != 0;
    const bool check = P->prm.check_physical_validity != 0;
    const int n = rk3 ? 3 : 1;
    int rc;
    if ((rc = ensure_x(P, err))) return rc;
    // (a first-order Euler step's sweep B reads its neighbours' values in X)
    const bool store_x = rk3 || second;
    double *const Vin[3] = {P->X, P->Y, P->Z};
    for (int s = 0; s < n; ++s) {
        const bool last = s + 1 == n;
        PolyDev m = P->m;
        m.stop = on_device ? P->flags : P->run.bad;
        m.nstop = on_device ? 1 : (check ? s : 0);
        SweepB a{};
        a.U = s == 0 ? P->state() : P->Ub;
        a.Uo = P->Ua;
        a.Uout = last ? P->Ua : P->Ub;
        a.Vout = last ? (store_x ? P->X : nullptr) : Vin[s + 1];
        a.R = check ? P->R : nullptr;
        a.res_part = s == 0 ? P->res_part : nullptr;
        a.bad = check ? P->run.bad + s : nullptr;
        a.kind = check ? -1 : s;
        a.dt = dt;
        a.dtp = on_device ? P->run.dtdev : nullptr;
        a.dtc = lts ? P->dtc : nullptr;
        // (kernel timing: the primvars and ghosts of the stage in launches of their own)
        if (P->timing && (rc = prim_of(P, a.U, Vin[s], true, err))) return rc;
        if ((rc = flux_balance(P, m, Vin[s], a, false, last || (lts && s == 0) ? P->dt_part : nullptr,
                               lts && s == 0 ? P->dtc : nullptr, err)))
            return rc;
        if (check) {
            m.nstop = s + 1;
            a.kind = s;
            a.zero_old = P->run.zero_old;
            hipLaunchKernelGGL(k_poly_update, dim3(P->blocks()), dim3(PB), 0, P->st, m, a);
        }
    }
    P->x_prim = store_x;
    PHIP(hipGetLastError());
    return NF_OK;
}

// where begin and step_end leave their results, taken by the first of them
void ensure_host(PolyPath *P) {
    if (!P->run.host) P->run.host = static_cast<double *>(PinnedPool::get().record());
    if (!P->run.host) P->run.host = P->dev_res;
}
// the results, after the work enqueued so far
int read_results(PolyPath *P, std::string &err) {
    if (P->run.host == P->dev_res)
        PHIP(hipMemcpyAsync(P->res, P->dev_res, sizeof P->res, hipMemcpyDeviceToHost, P->st));
    PHIP(hipStreamSynchronize(P->st));
    if (P->run.host != P->dev_res) std::copy(P->run.host, P->run.host + 5, P->res);
    return NF_OK;
}

int step_end(PolyPath *P, bool on_device, std::string &err) {
    ensure_host(P);
    RunDev r = P->run;
    r.flags = on_device ? P->flags : nullptr;
    hipLaunchKernelGGL(k_poly_end, dim3(1), dim3(PB), 0, P->st, r, (const double *)P->res_part,
                       (const double *)P->dt_part, P->blocks());
    PHIP(hipGetLastError());
    return NF_OK;
}

// dt of the first step where it is not in place, and (on_device) a run's start
int begin(PolyPath *P, bool on_device, double drop, double ref, std::string &err) {
    ensure_host(P);
    RunDev r = P->run;
    r.flags = on_device ? P->flags : nullptr;
    if (!P->dt_valid) {
        PolyDev m = P->m;
        m.nstop = 0;
        hipLaunchKernelGGL(k_poly_dt, dim3(P->blocks()), dim3(PB), 0, P->st, m, (const double *)P->X, P->prm.CFL,
                           P->dt_part, (double *)nullptr);
    }
    hipLaunchKernelGGL(k_poly_begin, dim3(1), dim3(PB), 0, P->st, r,
                       (const double *)(P->dt_valid ? nullptr : P->dt_part), P->blocks(), drop, ref);
    PHIP(hipGetLastError());
    return NF_OK;
}

int set_old_zero(PolyPath *P, bool zero, std::string &err) {
    P->old_zero = zero;
    hipLaunchKernelGGL(k_poly_set, dim3(1), dim3(1), 0, P->st, P->run.zero_old, zero ? 1 : 0);
    PHIP(hipGetLastError());
    return NF_OK;
}

std::string bad_cells(int n) {
    return std::to_string(n) + " cells with unphysical values detected in the flux_balance field of the Euler solver";
}

}  // namespace

int poly_create(const PrimalMesh &pm, const FVGrid &g, const nf_params &p, hipStream_t st, HostPipe &pipe,
                PolyPath **out, std::string &err) {
    (void)pm;
    *out = nullptr;
    if (p.precision != NF_PREC_FP64) {
        err = "a mixed-element mesh runs in FP64 only";
        return NF_E_ARG;
    }
    std::unique_ptr<PolyPath> hold(new PolyPath);
    PolyPath *P = hold.get();
    P->st = st;
    P->pipe = &pipe;
    P->prm = p;
    const uint32_t N = g.N, NT = g.NT, Fint = g.Fint, F = g.F;
    P->sizes = {N, NT, Fint, F, (uint32_t)g.pfirst.size()};
    if (NT - 1 > IDX) {
        err = "mesh too large for the mixed-element path";
        return NF_E_MESH;
    }
    // device numbering (cell_order); each cell keeps its faces in increasing
    // reference face index, so every sum keeps the reference's order
    if (p.cell_order == NF_ORDER_RCM) P->perm = rcm_order(g);
    else if (p.cell_order == NF_ORDER_MORTON) P->perm = morton_order(g);
    else {
        P->perm.resize(N);
        for (uint32_t c = 0; c < N; ++c) P->perm[c] = c;
    }
    std::vector<uint32_t> iperm(N);
    for (uint32_t d = 0; d < N; ++d) iperm[P->perm[d]] = d;
    // slots: the faces of each cell in increasing face index
    std::vector<uint32_t> w((size_t)6 * N, NONE);
    std::vector<uint8_t> ns((size_t)6 * N, 0), cnt(N, 0);
    std::vector<double> geo((size_t)36 * N, 0.0);
    const uint32_t G = F - Fint;
    // boundary faces in device cell order: bat[b] = reference boundary face
    std::vector<uint32_t> bat(G), bpos(G);
    for (uint32_t b = 0; b < G; ++b) bat[b] = b;
    auto bcell = [&](uint32_t b) { return iperm[g.ij[2 * (size_t)(Fint + b)]]; };
    std::stable_sort(bat.begin(), bat.end(), [&](uint32_t a, uint32_t b) { return bcell(a) < bcell(b); });
    for (uint32_t b = 0; b < G; ++b) bpos[bat[b]] = b;
    std::vector<uint32_t> bi(G), bj(G), boff((N + PB - 1) / PB + 1, 0);
    std::vector<double> bS((size_t)3 * G);
    std::vector<uint8_t> bbc(G), bslot(G);
    for (size_t q = 0; q < g.pfirst.size(); ++q)
        for (uint32_t f = g.pfirst[q]; f < g.pfirst[q] + g.pn[q]; ++f) bbc[bpos[f - Fint]] = (uint8_t)g.pbc[q];
    auto put_geo = [&](uint32_t c, int s, uint32_t f, const std::vector<double> &r) {
        for (int d = 0; d < 3; ++d) {
            geo[((size_t)s * 6 + d) * N + c] = g.S[3 * (size_t)f + d];
            geo[((size_t)s * 6 + 3 + d) * N + c] = r[3 * (size_t)f + d];
        }
    };
    for (uint32_t f = 0; f < F; ++f) {
        const uint32_t i = iperm[g.ij[2 * (size_t)f]], jr = g.ij[2 * (size_t)f + 1];
        const uint32_t j = jr < N ? iperm[jr] : jr;  // ghosts keep their reference id
        if (cnt[i] >= 6 || (j < N && cnt[j] >= 6)) {
            err = "cell with more than six faces";
            return NF_E_MESH;
        }
        const int si = cnt[i]++;
        if (j < N) {
            const int sj = cnt[j]++;
            w[(size_t)si * N + i] = j;
            ns[(size_t)si * N + i] = (uint8_t)sj;
            w[(size_t)sj * N + j] = i | SIDE_J;
            ns[(size_t)sj * N + j] = (uint8_t)si;
            put_geo(j, sj, f, g.rj);
        } else {
            const uint32_t b = bpos[f - Fint];
            w[(size_t)si * N + i] = j | BND;
            bi[b] = i;
            bj[b] = j;
            bslot[b] = (uint8_t)si;
            boff[i / PB + 1]++;
            for (int d = 0; d < 3; ++d) bS[(size_t)d * G + b] = g.S[3 * (size_t)f + d];
        }
        put_geo(i, si, f, g.ri);
    }
    for (size_t q = 1; q < boff.size(); ++q) boff[q] += boff[q - 1];
    std::vector<double> vol(N), dS((size_t)3 * N);
    for (uint32_t c = 0; c < N; ++c) {
        vol[c] = g.vol[P->perm[c]];
        for (int d = 0; d < 3; ++d) dS[d * (size_t)N + c] = g.dS[3 * (size_t)P->perm[c] + d];
    }
    uint32_t *dw, *dbi, *dbj;
    uint8_t *dns, *dbbc, *dbslot;
    double *dgeo, *dvol, *ddS, *dbS;
    const size_t plane = std::max(N, G);
    const uint32_t nblk = (N + PB - 1) / PB;
    int rc;
    if ((rc = alloc_all(P, {{&dw, w.size()}, {&dns, ns.size()}, {&dgeo, geo.size()}, {&dvol, N},
                            {&ddS, 3 * (size_t)N}, {&dbi, G}, {&dbj, G}, {&dbS, 3 * (size_t)G}, {&dbbc, G},
                            {&dbslot, G}, {&P->boff, boff.size()}},
                        err)))
        return rc;
    if ((rc = upload(dw, w, err)) || (rc = upload(dns, ns, err)) || (rc = upload(dgeo, geo, err)) ||
        (rc = upload(dvol, vol, err)) || (rc = upload(ddS, dS, err)) || (rc = upload(dbi, bi, err)) ||
        (rc = upload(dbj, bj, err)) || (rc = upload(dbS, bS, err)) || (rc = upload(dbbc, bbc, err)) ||
        (rc = upload(dbslot, bslot, err)) || (rc = upload(P->boff, boff, err)))
        return rc;
    P->m = {N, NT, G, plane, dw, dns, dgeo, dvol, ddS, dbi, dbj, dbslot, dbbc, dbS,
            P->boff, make_farfield<double>(p.primvars_inf), nullptr, 0};
    if ((rc = alloc_all(P, {{&P->Ua, 5 * (size_t)N}, {&P->Ub, 5 * (size_t)N}, {&P->X, 5 * (size_t)NT},
                            {&P->Y, 5 * (size_t)NT}, {&P->Z, 5 * (size_t)NT}, {&P->FV, 35 * plane},
                            {&P->grad, 15 * (size_t)N}, {&P->psi, 5 * (size_t)N}, {&P->R, 5 * (size_t)N},
                            {&P->dt_part, nblk}, {&P->res_part, nblk}, {&P->dtc, N}, {&P->flags, 4},
                            {&P->run.dtdev, 1}, {&P->dev_res, 5}, {&P->run.runp, 2}, {&P->run.zero_old, 1}, {&P->run.bad, 3}},
                        err)))
        return rc;
    PHIP(hipMemset(P->run.bad, 0, 3 * sizeof(int)));
    if ((rc = poly_set_freestream(P, err))) return rc;
    *out = hold.release();
    return NF_OK;
}

void poly_destroy(PolyPath *P) { delete P; }

nf_fv_sizes poly_sizes(const PolyPath *P) { return P->sizes; }

// set_freestream_values (src/SolverData.cpp:50-58)
static void reset_run(PolyPath *P) {
    P->hist.clear();
    P->time = 0.0;
    P->converged = false;
    P->aux_valid = false;
    P->split = P->dt_valid = P->x_prim = false;
}

int poly_set_freestream(PolyPath *P, std::string &err) {
    const uint32_t N = P->m.N;
    reset_run(P);
    Five U, V;
    prim_to_cons(P->prm.primvars_inf, U.v);
    std::copy(P->prm.primvars_inf, P->prm.primvars_inf + 5, V.v);
    hipLaunchKernelGGL(k_poly_fill, grid(N), dim3(PB), 0, P->st, P->Ua, U, P->X, V, (size_t)P->m.NT, N);
    PHIP(hipGetLastError());
    // (X is V_inf, which the first dt is taken from, and not prim(U) bit for bit)
    int rc;
    if ((rc = set_old_zero(P, P->prm.rk3_zero_old_first_step != 0, err))) return rc;
    PHIP(hipStreamSynchronize(P->st));
    return NF_OK;
}

// U as given, primvars = prim(U); U_old = zero (the reference's first RK3
// step) unless given, and a given U_old must equal U
int poly_set_state(PolyPath *P, const double *U, const double *U_old, std::string &err) {
    const uint32_t N = P->m.N;
    bool zero = P->prm.rk3_zero_old_first_step != 0;
    if (U_old) {
        if (U != U_old && std::memcmp(U, U_old, (size_t)5 * N * sizeof(double)) != 0) {
            err = "U_old must be NULL (zero) or equal to U";
            return NF_E_ARG;
        }
        zero = false;
    }
    int rc;
    reset_run(P);
    if ((rc = put_soa(P, P->Ua, U, 5, err)) || (rc = ensure_x(P, err)) || (rc = set_old_zero(P, zero, err))) return rc;
    PHIP(hipStreamSynchronize(P->st));
    return NF_OK;
}

// the dt the last step left, or that of the primvars as set
int poly_calc_timestep(PolyPath *P, double *dt_out, std::string &err) {
    int rc;
    if (!P->dt_valid) {
        if ((rc = begin(P, false, 0.0, 0.0, err)) || (rc = read_results(P, err))) return rc;
        P->dt = P->res[1];
        P->dt_valid = true;
    }
    const double dt = P->dt;
    if (dt_out) *dt_out = dt;
    if (!((dt - dt == 0.0) && dt > 0.0)) {
        char buf[96];
        std::snprintf(buf, sizeof buf, "Invalid dt calculated (dt = %f)", dt);
        err = buf;
        return NF_E_INVALID_DT;
    }
    return NF_OK;
}

// Solver::step (src/Solver.cpp:34-52, 83-133), one synchronisation
int poly_step(PolyPath *P, double dt, std::string &err) {
    int rc;
    P->aux_valid = false;
    if ((rc = stages(P, false, dt, err)) || (rc = step_end(P, false, err)) || (rc = read_results(P, err))) return rc;
    for (int s = 0; s < 3; ++s) {
        const int n = (int)P->res[2 + s];
        if (n == 0) continue;
        // the state is the failed stage's input, U_old what it was
        P->split = P->split || s > 0;
        P->x_prim = P->dt_valid = false;
        if ((rc = ensure_x(P, err))) return rc;
        err = bad_cells(n);
        return NF_E_NONPHYSICAL;
    }
    P->hist.push_back(P->res[0]);  // the flux balance of U^n (first stage), as in the batched path
    P->time += dt;
    P->dt = P->res[1];
    P->dt_valid = true;
    P->split = P->old_zero = false;
    return NF_OK;
}

// the flux balance of the current state, once, with a primvar buffer of the
// stages: those the next dt or step reads are left as the last step set them
int poly_eval_flux_balance(PolyPath *P, std::string &err) {
    int rc;
    const bool check = P->prm.check_physical_validity != 0, timing = P->timing;
    PolyDev m = P->m;
    m.nstop = 0;
    SweepB a{};
    a.R = P->R;
    a.bad = check ? P->run.bad : nullptr;
    a.kind = -1;
    P->timing = false;
    rc = prim_of(P, P->state(), P->Y, false, err);
    if (!rc) rc = flux_balance(P, m, P->Y, a, true, nullptr, nullptr, err);
    P->timing = timing;
    if (rc) return rc;
    int bad = 0;
    if (check) PHIP(hipMemcpyAsync(&bad, P->run.bad, sizeof bad, hipMemcpyDeviceToHost, P->st));
    PHIP(hipStreamSynchronize(P->st));
    if (bad) {
        PHIP(hipMemset(P->run.bad, 0, sizeof bad));
        err = bad_cells(bad);
        return NF_E_NONPHYSICAL;
    }
    P->aux_valid = true;
    return NF_OK;
}

int poly_get_state(PolyPath *P, double *U, std::string &err) { return get_soa(P, P->state(), 5, U, err); }

// The Driver loop (calc_timestep, step) for n steps, stopping after the step
// whose residual norm is at most drop times the first step's; a run that has
// reached its drop stays stopped until the state is set again.
static int poly_run_host(PolyPath *P, const nf_run_opts *o, nf_run_stats *stats, std::string &err) {
    const double drop = o->residual_drop;
    hipEvent_t e0, e1;
    PHIP(hipEventCreate(&e0));
    PHIP(hipEventCreate(&e1));
    PHIP(hipEventRecord(e0, P->st));
    int done = 0, rc = NF_OK;
    double dt = 0.0;
    if (!(drop > 0.0 && P->converged)) {
        while (done < o->n_steps) {
            if ((rc = poly_calc_timestep(P, &dt, err)) || (rc = poly_step(P, dt, err))) break;
            ++done;
            if (drop > 0.0 && P->hist[0] > 0.0 && P->hist.back() / P->hist[0] <= drop) {
                P->converged = true;
                break;
            }
        }
    }
    float ms = 0.0f;
    (void)hipEventRecord(e1, P->st);
    (void)hipEventSynchronize(e1);
    (void)hipEventElapsedTime(&ms, e0, e1);
    (void)hipEventDestroy(e0);
    (void)hipEventDestroy(e1);
    if (stats) {
        stats->steps_done = done;
        stats->converged = P->converged ? 1 : 0;
        stats->time = P->time;
        stats->last_dt = dt;
        stats->res_first = P->hist.empty() ? 0.0 : P->hist.front();
        stats->res_last = P->hist.empty() ? 0.0 : P->hist.back();
        stats->elapsed_ms = ms;
        stats->fell_back = 0;
        stats->pad = 0;
    }
    return rc;
}

// HIP-event durations of each kernel over n steps of the Driver loop, with
// each stage's primvars and cell ghosts formed once more by the launches that
// form them after a state change
int poly_time_kernels(PolyPath *P, int32_t n_steps, nf_kernel_time *out, int32_t max, int32_t *n_out,
                      std::string &err) {
    if (n_steps < 1 || !out) return NF_E_ARG;
    P->ktime.clear();
    P->timing = true;
    int rc = NF_OK;
    for (int q = 0; q < n_steps && rc == NF_OK; ++q) {
        double dt;
        if ((rc = poly_calc_timestep(P, &dt, err)) == NF_OK) rc = poly_step(P, dt, err);
        const int f = tflush(P, err);
        if (rc == NF_OK) rc = f;
    }
    P->timing = false;
    if (rc) return rc;
    int n = 0;
    for (auto &kv : P->ktime) {
        if (n >= max) break;
        std::snprintf(out[n].name, sizeof out[n].name, "%s", kv.first.c_str());
        out[n].avg_ms = kv.second.first / kv.second.second;
        out[n].calls = kv.second.second;
        ++n;
    }
    if (n_out) *n_out = n;
    return NF_OK;
}

// One step of the device-resident run: the same kernels and values as
// calc_timestep + step, with dt, residual and the stop test on the device.
static int enqueue_run_step(PolyPath *P, std::string &err) {
    int rc;
    if ((rc = stages(P, true, 0.0, err))) return rc;
    return step_end(P, true, err);
}

// nf_run: check_every steps, captured once as a HIP graph (use_graph) or
// launched eagerly, run between host synchronisations; the stop flag ends the
// remaining ones on the device, so the run stops after exactly the step that
// reached the drop, as the host loop does.  With the flux-balance check on (a
// host read per stage) the host loop runs instead.
int poly_run(PolyPath *P, const nf_run_opts *o, nf_run_stats *stats, std::string &err) {
    if (!o || o->n_steps < 0) return NF_E_ARG;
    if (P->prm.check_physical_validity) return poly_run_host(P, o, stats, err);
    const double drop = o->residual_drop;
    int rc;
    P->aux_valid = false;
    if ((int64_t)o->n_steps + 1 > P->run_cap) {  // per-step history buffers, grown (the graph refers to them)
        const int64_t cap = std::max<int64_t>((int64_t)o->n_steps + 1, 1024);
        PHIP(hipStreamSynchronize(P->st));
        if (P->graph) {
            (void)hipGraphExecDestroy(P->graph);
            P->graph = nullptr;
        }
        for (double *old : {P->run.dts, P->run.hres}) {
            if (!old) continue;
            P->owned.erase(std::find(P->owned.begin(), P->owned.end(), (void *)old));
            PHIP(hipFree(old));
        }
        P->run.dts = P->run.hres = nullptr;
        P->run_cap = 0;
        if ((rc = alloc(P, &P->run.dts, cap, err)) || (rc = alloc(P, &P->run.hres, cap, err))) return rc;
        P->run_cap = cap;
    }
    // this run's drop and reference (negative: the run's own first residual)
    if ((rc = begin(P, true, drop, P->hist.empty() ? -1.0 : P->hist.front(), err))) return rc;
    hipEvent_t e0, e1;
    PHIP(hipEventCreate(&e0));
    PHIP(hipEventCreate(&e1));
    PHIP(hipEventRecord(e0, P->st));
    const int K = std::max(1, o->check_every);
    int flags[4] = {0, 0, 0, 0}, queued = 0;
    if (!(drop > 0.0 && P->converged)) {
        while (queued < o->n_steps && !flags[0]) {
            const int chunk = std::min(K, o->n_steps - queued);
            // a graph starts from prim(U) in X, whatever was the case when it
            // was captured, and from the state in Ua (a split state exists only
            // with the flux-balance check, whose runs went to the host loop)
            if ((rc = ensure_x(P, err))) return rc;
            if (o->use_graph && chunk == K && K > 1) {
                if (!P->graph || P->graph_K != K) {
                    if (P->graph) (void)hipGraphExecDestroy(P->graph);
                    P->graph = nullptr;
                    hipGraph_t gr;
                    PHIP(hipStreamBeginCapture(P->st, hipStreamCaptureModeThreadLocal));
                    for (int q = 0; q < K; ++q)
                        if ((rc = enqueue_run_step(P, err))) {
                            (void)hipStreamEndCapture(P->st, &gr);
                            P->x_prim = false;
                            return rc;
                        }
                    PHIP(hipStreamEndCapture(P->st, &gr));
                    const hipError_t ie = hipGraphInstantiate(&P->graph, gr, nullptr, nullptr, 0);
                    (void)hipGraphDestroy(gr);
                    PHIP(ie);
                    P->graph_K = K;
                }
                PHIP(hipGraphLaunch(P->graph, P->st));
                P->x_prim = P->rk3() || P->second();
            } else {
                for (int q = 0; q < chunk; ++q)
                    if ((rc = enqueue_run_step(P, err))) return rc;
            }
            queued += chunk;
            PHIP(hipMemcpyAsync(flags, P->flags, sizeof flags, hipMemcpyDeviceToHost, P->st));
            PHIP(hipStreamSynchronize(P->st));
        }
    }
    float ms = 0.0f;
    (void)hipEventRecord(e1, P->st);
    (void)hipEventSynchronize(e1);
    (void)hipEventElapsedTime(&ms, e0, e1);
    (void)hipEventDestroy(e0);
    (void)hipEventDestroy(e1);
    const int done = flags[3];
    std::vector<double> dts(done + 1), res(done);
    PHIP(hipMemcpy(dts.data(), P->run.dts, (done + 1) * 8, hipMemcpyDeviceToHost));
    if (done > 0) PHIP(hipMemcpy(res.data(), P->run.hres, done * 8, hipMemcpyDeviceToHost));
    P->dt = dts[done];
    P->dt_valid = true;
    if (done > 0) P->old_zero = false;
    for (int k = 0; k < done; ++k) {
        P->time += dts[k];
        P->hist.push_back(res[k]);
    }
    if (flags[1]) P->converged = true;
    if (stats) {
        stats->steps_done = done;
        stats->converged = P->converged ? 1 : 0;
        stats->time = P->time;
        stats->last_dt = done > 0 ? dts[done - 1] : 0.0;
        stats->res_first = P->hist.empty() ? 0.0 : P->hist.front();
        stats->res_last = P->hist.empty() ? 0.0 : P->hist.back();
        stats->elapsed_ms = ms;
        stats->fell_back = 0;
        stats->pad = 0;
    }
    if (flags[2] && !flags[1] && done < o->n_steps) {
        char buf[96];
        std::snprintf(buf, sizeof buf, "Invalid dt calculated (dt = %f)", dts[done]);
        err = buf;
        return NF_E_INVALID_DT;
    }
    return NF_OK;
}

int poly_get_residuals(PolyPath *P, double *out, int32_t max, int32_t *n_out) {
    const int32_t n = (int32_t)std::min<size_t>(P->hist.size(), (size_t)std::max(max, 0));
    std::copy(P->hist.begin(), P->hist.begin() + n, out);
    if (n_out) *n_out = n;
    return NF_OK;
}

int poly_get_field(PolyPath *P, int32_t which, double *out, std::string &err) {
    switch (which) {
    case NF_FIELD_PRIM:  // prim(U) with row stride N for the export
        hipLaunchKernelGGL(k_poly_prim, grid(P->m.N), dim3(PB), 0, P->st, (const double *)P->state(), P->Y, P->m.N,
                           P->m.N);
        PHIP(hipGetLastError());
        return get_soa(P, P->Y, 5, out, err);
    case NF_FIELD_STATE_OLD:
        if (P->old_zero) {
            std::memset(out, 0, 5 * (size_t)P->m.N * 8);
            return NF_OK;
        }
        return get_soa(P, P->Ua, 5, out, err);
    case NF_FIELD_LIMITER:
    case NF_FIELD_GRADIENT:
    case NF_FIELD_RESIDUAL:
        if (!P->aux_valid) {
            err = "call nf_eval_flux_balance first";
            return NF_E_ARG;
        }
        if (which == NF_FIELD_LIMITER) {
            if (P->prm.spatial_order != NF_SECOND_ORDER) {  // psi keeps its initial 1 (SolverData.cpp:17)
                for (size_t q = 0; q < 5 * (size_t)P->m.N; ++q) out[q] = 1.0;
                return NF_OK;
            }
            return get_soa(P, P->psi, 5, out, err);
        }
        if (which == NF_FIELD_GRADIENT) {
            if (P->prm.spatial_order != NF_SECOND_ORDER) {
                std::memset(out, 0, 15 * (size_t)P->m.N * 8);
                return NF_OK;
            }
            return get_soa(P, P->grad, 15, out, err);
        }
        return get_soa(P, P->R, 5, out, err);
    default:
        err = "unknown field";
        return NF_E_ARG;
    }
}

}  // namespace nf
