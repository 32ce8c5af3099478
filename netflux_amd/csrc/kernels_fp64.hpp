// FP64 stage kernels of the explicit Euler step.
//
// Mapping: one tetrahedron per lane.  The lane visits its four faces in slot
// order -- slot s is the cell's s-th face in increasing reference face index
// -- so every per-cell accumulation (Green-Gauss gradient, flux balance,
// Delta S) adds the same terms in the same order as the reference's
// face-ordered scatter loops, and FP64 results are identical to a serial
// evaluation of the reference formulas, with no atomics and no colouring.
// Geometry (volume, centroid, face normals, centroid-to-face vectors) is
// recomputed from the four nodes with the reference formulas instead of
// being streamed from memory.
//
//   sweep A (per stage): V -> Green-Gauss gradient, neighbour min/max, Barth
//            limiter, limited face values of the four faces
//            (+ Delta S and the CFL time step when requested).
//   sweep B (per stage): face values -> Rusanov fluxes of the four faces,
//            flux balance, RK stage combination, prim(U) of the new state.
//   Boundary faces read their ghost state from small per-boundary-face
//   buffers: ghosts of the cell-centre states (for the gradient and min/max)
//   and of the reconstructed face states (for the boundary flux).  k_ghost
//   fills them, or, on small meshes (FUSE), the end of the sweep before.
//
// Several meshes (instances) can share one launch: their cells are
// concatenated, each instance padded to whole blocks of 256 cells, and every
// block looks up its instance for the time step, the first-step flag, the
// stop flag and the error counters (InstState).
//
// Layouts: cell fields are tiled by 64 cells (one wavefront):
//   V, U  : [tile][5][64]          FV : [tile][4 slots][5][64]
// so a wave's own-cell loads and stores are fully coalesced; cnodes and nbr
// are [N][4] u32, fcode [N], nodes [n_nodes][4] (x, y, z, pad).
#pragma once
#include <hip/hip_runtime.h>

#include <cstdint>

#include "face_record.hpp"
#include "fp64_math.hpp"
#include "physics.hpp"

namespace nf {

// sweep A reads neighbours in the lane's own 64-cell tile (1) or in its
// block (2, with block barriers) from LDS
#ifndef NF_A_LDS
#define NF_A_LDS 2
#endif
// sweep A writes its face values with 16-byte stores (needs NF_A_LDS)
#ifndef NF_A_STX4
#define NF_A_STX4 1
#endif
// waves per SIMD the sweeps are compiled for (0: the compiler's choice)
#ifndef NF_SWEEP_WAVES
#define NF_SWEEP_WAVES 0
#endif
#if NF_SWEEP_WAVES
#define NF_SWEEP_ATTR __attribute__((amdgpu_waves_per_eu(NF_SWEEP_WAVES, NF_SWEEP_WAVES)))
#else
#define NF_SWEEP_ATTR
#endif
#ifndef NF_SWEEPB_WAVES
#define NF_SWEEPB_WAVES 0
#endif
#if NF_SWEEPB_WAVES
#define NF_SWEEPB_ATTR __attribute__((amdgpu_waves_per_eu(NF_SWEEPB_WAVES, NF_SWEEPB_WAVES)))
#else
#define NF_SWEEPB_ATTR NF_SWEEP_ATTR
#endif

constexpr int BLOCK = 256;  // threads of the auxiliary kernels; instance padding unit
constexpr int TILE = 64;    // cells per layout tile
constexpr uint32_t FACE_LDS = 53728;  // most LDS bytes of a block of k_sweepA_face (three per CU)

// load through a global-address-space pointer (keeps the compiler from
// falling back to flat loads, which also count against the LDS counter)
__device__ __forceinline__ double ldg(const double *p) {
    return *(const __attribute__((address_space(1))) double *)p;
}

__device__ __forceinline__ size_t tix(uint32_t c, int k) {  // [tile][5][64]
    return ((size_t)(c >> 6) * 5 + k) * TILE + (c & 63u);
}
__device__ __forceinline__ size_t fix(uint32_t c, uint32_t s, int k) {  // [tile][4][5][64]
    return (((size_t)(c >> 6) * 4 + s) * 5 + k) * TILE + (c & 63u);
}

// Per-instance run state, one record per mesh of the context.
struct InstState {
    double dt;         // time step of the current step
    double time;       // sum of completed steps' dt
    double rref;       // residual the drop is measured against (0: the first step's)
    int nstep;         // completed steps
    int err;           // NF_E_INVALID_DT once raised
    int stop;          // nonzero: kernels skip this instance
    int converged;     // residual drop reached
    int bad_flux;      // cells with non-finite flux balance (checked runs)
    int bad_state;     // cells with rho <= 0, p <= 0 or NaN after an update
    int uold_zero;     // U_old is all zeros (before the first step)
    int pad;
};

struct DevMesh {
    double three, six;       // 3.0 and 6.0, divisors of the centroid / volume formulas
    const double *nodes;
    const uint32_t *cnodes;
    // per 64-cell group: its distinct nodes' coordinates, SoA, entries
    // [grp_off[g], grp_off[g+1]); cell_ln: per cell 4 x u16, the byte
    // offsets of its nodes in the group's [node][3] table
    const uint32_t *grp_off;
    const double *gx, *gy, *gz;
    const uint2 *cell_ln;
    const uint32_t *nbr;
    // per BLOCK cells, null if some block has too many records: faces between
    // two of its cells, numbers [foff[b], foff[b+1]), and records of its other
    // cell sides, [roff[b], roff[b+1]).  Per record: hal, the cell of the
    // face's other side (or bit 31 and boundary face); rec, that side's record
    // (face_record.hpp); rS [tile][3][64], the face vector.  Per cell
    // 4 x u16: cell_nb, where a slot's neighbour state is -- below BLOCK the
    // block's own cell, then the records' -- and bit 15 on a boundary slot;
    // cell_fx, the place of a slot's side among the block's 2 nf + nr (owner
    // sides of its faces, their other sides, records) and bit 15 on an owner's
    // side.  nstride: most nodes of a node table; nent: most nf + nr
    const uint32_t *foff, *roff, *hal, *rec;
    const uint2 *cell_nb, *cell_fx;
    const double *rS, *vol;
    uint32_t nstride, nent;
    const uint32_t *fcode;
    const uint32_t *blk_inst;  // [blocks] instance of each 256-cell block (32-bit: scalar loads)
    const uint32_t *inst_end;  // [instances] one past the instance's last device cell
    InstState *st;             // [instances]
};

// The lane's cell, its instance, and whether it is a real cell.  Dead lanes
// of the last block of an instance mirror the instance's last cell and store
// nothing.
struct LaneCell {
    uint32_t c, inst, lb;  // cell, instance, logical block
    bool live;
};
template <int B>
__device__ __forceinline__ LaneCell lane_cell(const DevMesh &m, int xcd_remap) {
    const uint32_t lb = logical_block(blockIdx.x, gridDim.x, xcd_remap);
    const uint32_t c0 = lb * B + threadIdx.x;
    const uint32_t inst = m.blk_inst[(lb * B) / BLOCK];
    const uint32_t end = m.inst_end[inst];
    return {c0 < end ? c0 : end - 1, inst, lb, c0 < end};
}

// The boundary faces of a block's cells (numbered in device cell order).
// Loaded by a sweep before anything else, kept there by the asm: at its end
// every block would wait for these scalar loads.
struct BndRange {
    uint32_t b0, b1;
};
template <int B>
__device__ __forceinline__ BndRange bnd_range(const uint32_t *boff, uint32_t lb) {
    BndRange r{boff[lb * (B / 128)], boff[(lb + 1) * (B / 128)]};
    asm volatile("" : "+s"(r.b0), "+s"(r.b1));
    return r;
}

struct CellGeo {
    V3d p0, p1, p2, p3;
    V3d cen;
    double vol;
    Rcp ivol;
};

// Node loads of cell c from the node array (boundary-face kernels).
__device__ __forceinline__ void load_nodes(const DevMesh &m, uint32_t c, CellGeo &g) {
    const uint4 q = *reinterpret_cast<const uint4 *>(m.cnodes + 4 * (size_t)c);
    auto node = [&](uint32_t n) {
        const double2 a = *reinterpret_cast<const double2 *>(m.nodes + 4 * (size_t)n);
        return V3d{a.x, a.y, m.nodes[4 * (size_t)n + 2]};
    };
    g.p0 = node(q.x);
    g.p1 = node(q.y);
    g.p2 = node(q.z);
    g.p3 = node(q.w);
}

// volume, centroid and 1/volume of loaded nodes
__device__ __forceinline__ void cell_geo(const DevMesh &m, CellGeo &g) {
    // tetrahedron_calc_volume / _centroid (src/geometry/GeometryUtilities.cpp:289-316)
    const V3d ab = vsub(g.p1, g.p0), ac = vsub(g.p2, g.p0), ad = vsub(g.p3, g.p0);
    g.vol = rdiv(dot3(vcross(ab, ac), ad), rcp_of(m.six));
    g.cen = vscl(1.0 / 4, vadd(vadd(vadd(g.p0, g.p1), g.p2), g.p3));
    g.ivol = rcp_of(g.vol);
}

__device__ __forceinline__ void load_cell(const DevMesh &m, uint32_t c, CellGeo &g) {
    load_nodes(m, c, g);
    cell_geo(m, g);
}

// Node coordinates in LDS, [entry][3].  l holds the byte offsets of the four
// cell nodes' entries, 16 bits each: one byte permute selects a face's node,
// its three coordinates follow at constant offsets (with separate rows and
// the offsets in four registers the selects were 5 % of sweep A's
// instructions).
struct NodeView {
    const double *lds;
    uint2 l;
};
__device__ __forceinline__ V3d nv_node(const NodeView &v, uint32_t q) {
    const uint32_t o = __builtin_amdgcn_perm(v.l.y, v.l.x, 0x0c0c0100u + q * 0x0202u);
    const double *w = reinterpret_cast<const double *>(reinterpret_cast<const char *>(v.lds) + o);
    return {w[0], w[1], w[2]};
}

// Per-lane staging (boundary-face kernels): lane t writes its four nodes at
// entries 4 t + q; only its own entries are read, so no barrier is needed.
template <int B>
__device__ __forceinline__ NodeView stage_nodes(double *lds, const CellGeo &g) {
    const uint32_t t = threadIdx.x;
    const V3d P[4] = {g.p0, g.p1, g.p2, g.p3};
    const uint32_t o = 96 * t;
    NodeView v{lds, make_uint2(o | (o + 24) << 16, (o + 48) | (o + 72) << 16)};
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        lds[12 * t + 3 * q] = P[q].x;
        lds[12 * t + 3 * q + 1] = P[q].y;
        lds[12 * t + 3 * q + 2] = P[q].z;
    }
    return v;
}

// Per-wave node table (sweeps): the wave's 64 cells (one group) load their
// distinct nodes once, coalesced, into the wave's LDS slice (at most 256
// entries); each lane then takes its cell's nodes from there.  The loads are
// issued here, before the sweep's state gathers, so that waiting for them
// does not wait for the gathers (memory counters retire in order).  p is the
// lane's device cell position (padding included).  Only lanes of the same
// wave exchange data through the slice, so no block barrier is needed.
struct NodeTableLoad {
    double x, y, z;
    uint32_t n;
    uint2 q;
};
__device__ __forceinline__ NodeTableLoad node_table_issue(const DevMesh &m, uint32_t p) {
    const uint32_t gi = p >> 6, lane = p & 63u;
    const uint32_t o0 = m.grp_off[gi], n = m.grp_off[gi + 1] - o0;
    NodeTableLoad t;
    t.n = n;
    t.q = m.cell_ln[p];
    // up to 256 nodes: four per lane at most; the first 64 here, the rest
    // (rare: only very irregular orderings) in node_table_finish
    const uint32_t i = lane < n ? lane : 0;
    t.x = m.gx[o0 + i];
    t.y = m.gy[o0 + i];
    t.z = m.gz[o0 + i];
    return t;
}
template <int B>
__device__ __forceinline__ NodeView node_table_finish(const DevMesh &m, uint32_t p, const NodeTableLoad &t,
                                                      double *lds, CellGeo &g, uint32_t stride = 256) {
    const uint32_t lane = p & 63u, wv = threadIdx.x >> 6;
    double *w = lds + wv * 3 * stride;  // [stride][3] per wave
    if (lane < t.n) {
        w[3 * lane] = t.x;
        w[3 * lane + 1] = t.y;
        w[3 * lane + 2] = t.z;
    }
    if (t.n > 64) {  // uniform per wave
        const uint32_t o0 = m.grp_off[p >> 6];
        for (uint32_t i = lane + 64; i < t.n; i += 64) {
            w[3 * i] = m.gx[o0 + i];
            w[3 * i + 1] = m.gy[o0 + i];
            w[3 * i + 2] = m.gz[o0 + i];
        }
    }
    // LDS operations of one wave complete in order; the fences keep the
    // compiler from moving the reads above the writes
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    NodeView v{w, t.q};
    g.p0 = nv_node(v, 0);
    g.p1 = nv_node(v, 1);
    g.p2 = nv_node(v, 2);
    g.p3 = nv_node(v, 3);
    return v;
}

// Face normal oriented i->j (triangle formula of src/geometry/
// GeometryUtilities.cpp:318-324, flip of src/geometry/FV_Grid.cpp:247-250)
// and centroid-to-face vector (triangle_calc_centroid, :326-329) from the
// face element's node order.
__device__ __forceinline__ void face_geo(const DevMesh &m, const CellGeo &g, const NodeView &nv, uint32_t byte,
                                         V3d &S, V3d *r) {
    const V3d a = nv_node(nv, byte & 3u), b = nv_node(nv, (byte >> 2) & 3u), c = nv_node(nv, (byte >> 4) & 3u);
    S = vscl(0.5, vcross(vsub(b, a), vsub(c, a)));
    if (byte & 0x40u) S = vscl(-1, S);
    if (r) {
        const V3d s = vadd(vadd(a, b), c);
        const Rcp i3 = rcp_of(m.three);
        const V3d fc = {rdiv(s.x, i3), rdiv(s.y, i3), rdiv(s.z, i3)};
        *r = vsub(fc, g.cen);
    }
}

// wave + block min / sum over all threads; result valid in thread 0.  The min
// skips NaN inputs, as the reference's running std::min(delta_time, x) does
// (x = NaN compares false and leaves delta_time), whatever lane holds them.
template <bool MIN, int B>
__device__ __forceinline__ double block_reduce(double v, double *sh) {
    if (MIN && !(v == v)) v = DBL_MAX;
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
        const double w = __shfl_xor(v, o, 64);
        v = MIN ? ((w < v) ? w : v) : v + w;
    }
    const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
    if (lane == 0) sh[wid] = v;
    __syncthreads();
    if (threadIdx.x == 0) {
        v = sh[0];
        for (int q = 1; q < B / 64; ++q) v = MIN ? ((sh[q] < v) ? sh[q] : v) : v + sh[q];
    }
    return v;
}

// CFL step of a cell (src/Solver.cpp:254-266) with Delta S over its interior
// faces (src/Solver.cpp:287-297), in slot order
__device__ __forceinline__ double cell_dt(const double *Vc, const V3d *S, const uint32_t *w, double vol, double CFL) {
    double d0 = 0.0, d1 = 0.0, d2 = 0.0;
#pragma unroll
    for (int s = 0; s < 4; ++s) {
        if (!(w[s] & 0x80000000u)) {
            d0 += 0.5 * fabs(S[s].x);
            d1 += 0.5 * fabs(S[s].y);
            d2 += 0.5 * fabs(S[s].z);
        }
    }
    const double cs = sound_speed_prim(Vc);
    const double sx = (fabs(Vc[1]) + cs) * d0;
    const double sy = (fabs(Vc[2]) + cs) * d1;
    const double sz = (fabs(Vc[3]) + cs) * d2;
    return CFL * vol / ((sx + sy) + sz);
}

// Stage combination of Solver::TVD_RK3 / explicit_euler (src/Solver.cpp:
// 98-132) with f = (stage weight x dt) / volume: kind 1 U + f R, kind 2
// 3/4 U_old + 1/4 U + f R, kind 3 1/3 U_old + 2/3 U + f R (U_old = 0 on the
// first step of a zero-U_old run).  Shared by the fused sweeps and the checked
// stage update, so both give the same bits in a translation unit.
__device__ __forceinline__ void stage_combine(int kind, bool zero_old, double f, const double *Up,
                                              const double *Uop, const double *R, double *Un) {
    if (kind == 1) {
#pragma unroll
        for (int k = 0; k < 5; ++k) Un[k] = Up[k] + f * R[k];
    } else if (kind == 2) {
#pragma unroll
        for (int k = 0; k < 5; ++k) {
            const double uo = zero_old ? 0.0 : Uop[k];
            Un[k] = 3.0 / 4.0 * uo + 1.0 / 4.0 * Up[k] + f * R[k];
        }
    } else {
#pragma unroll
        for (int k = 0; k < 5; ++k) {
            const double uo = zero_old ? 0.0 : Uop[k];
            Un[k] = 1.0 / 3.0 * uo + 2.0 / 3.0 * Up[k] + f * R[k];
        }
    }
}

// Checked stage (check_physical_validity): the sweep stores R [tile][5][64]
// and f [cell] instead of updating; this pass updates only if no cell of the
// instance had a non-finite flux balance.  Otherwise the instance stops with
// U untouched and bad_flux holding that one evaluation's count, as the
// reference throws at the end of evaluate_flux_balance before any update
// (src/Solver.cpp:80, src/SolverData.cpp:66-79).  One lane per device cell,
// BLOCK-cell blocks (the instance padding unit).
struct ApplyArgs {
    const double *U, *Uo;
    double *Uout;
    void *Vout;  // prim(Uout): double (FP64 path, may be null) or float (mixed path)
    const double *Rst, *fst;
    int kind;
};

template <typename VT>
__device__ __forceinline__ void apply_stage_cell(const DevMesh &m, const ApplyArgs &a) {
    const uint32_t inst = m.blk_inst[blockIdx.x];
    InstState &st = m.st[inst];
    if (st.stop) return;
    if (st.bad_flux > 0) {
        if (threadIdx.x == 0) st.stop = 1;
        return;
    }
    const uint32_t c = blockIdx.x * BLOCK + threadIdx.x;
    if (c >= m.inst_end[inst]) return;
    const bool zero_old = st.uold_zero;
    const double *uo = (a.kind == 1 || zero_old) ? a.U : a.Uo;
    double Up[5], Uop[5], R[5], Un[5], Vnew[5];
#pragma unroll
    for (int k = 0; k < 5; ++k) {
        Up[k] = a.U[tix(c, k)];
        Uop[k] = uo[tix(c, k)];
        R[k] = a.Rst[tix(c, k)];
    }
    stage_combine(a.kind, zero_old, a.fst[c], Up, Uop, R, Un);
    cons_to_prim_d(Un, Vnew);
#pragma unroll
    for (int k = 0; k < 5; ++k) a.Uout[tix(c, k)] = Un[k];
    if (a.Vout) {
#pragma unroll
        for (int k = 0; k < 5; ++k) static_cast<VT *>(a.Vout)[tix(c, k)] = (VT)Vnew[k];
    }
    if (!(Vnew[0] > 0.0) || !(Vnew[4] > 0.0) || !(Un[4] > 0.0)) atomicAdd(&st.bad_state, 1);
}

#ifndef NF_DEVICE_HELPERS_ONLY
// ---------------------------------------------------------------------------
// boundary ghost states; boundary faces are numbered in device cell order
struct BndArgs {
    const uint32_t *bface;       // device cell | slot << 29
    const uint32_t *boff;        // [cells/128 + 1] first boundary face of each 128 device cells
    const uint16_t *binst;       // instance
    const uint8_t *bbc;          // boundary type
    const double *bS;            // [3][nb] S_ij of each boundary face (cell -> ghost)
    uint32_t nb;                 // boundary faces
    const uint32_t *brec;        // record of each boundary face (GhostOf::REC)
    const FarField<double> *fs;  // [instances]
    double *out;                 // [nb/64][5][64], tiled like V
};

// what a ghost is formed from: V (set_constant_ghost_values, src/Solver.cpp:
// 300-330), the primvars of the state U, or the reconstructed face states FV
// (src/Solver.cpp:210-212), or their records
enum class GhostOf { V, U, FV, REC };

// The face vector comes precomputed from the host face graph: the same cross
// product and sign the sweeps evaluate from the nodes, so the same bits.
template <GhostOf OF>
__device__ __forceinline__ void bnd_ghost(const BndArgs &a, uint32_t b, uint32_t inst, const double *src) {
    const uint32_t w = a.bface[b], c = w & 0x1FFFFFFFu;
    const V3d S = {a.bS[b], a.bS[a.nb + b], a.bS[2 * (size_t)a.nb + b]};
    double Vd[5], Vg[5];
#pragma unroll
    for (int k = 0; k < 5; ++k)
        Vd[k] = OF == GhostOf::FV ? src[fix(c, w >> 29, k)] : src[tix(OF == GhostOf::REC ? a.brec[b] : c, k)];
    if (OF == GhostOf::U) {
        const double Ud[5] = {Vd[0], Vd[1], Vd[2], Vd[3], Vd[4]};
        cons_to_prim_d(Ud, Vd);
    }
    ghost_d((int)a.bbc[b], Vd, S, a.fs[inst], Vg);
#pragma unroll
    for (int k = 0; k < 5; ++k) a.out[tix(b, k)] = Vg[k];
}

// Ghosts of the block's boundary faces, at the end of a sweep that stored
// src.  The block's faces are taken by its first lanes, one face per lane, so
// the long farfield branch (two pow) runs in as few waves as it can.
template <int B, GhostOf OF>
__device__ __forceinline__ void bnd_ghosts(const BndArgs &a, BndRange r, uint32_t inst, const double *src) {
    if (r.b0 == r.b1) return;  // the same for the whole block
    __syncthreads();           // every wave's part of src is stored
    for (uint32_t b = r.b0 + threadIdx.x; b < r.b1; b += B) bnd_ghost<OF>(a, b, inst, src);
}

// Ghosts of every boundary face in a launch of its own.  Also those of
// stopped instances: they have to match the state when it runs again.
template <GhostOf OF>
__global__ __launch_bounds__(BLOCK) void k_ghost(BndArgs a, const double *src) {
    const uint32_t b = blockIdx.x * BLOCK + threadIdx.x;
    if (b < a.nb) bnd_ghost<OF>(a, b, a.binst[b], src);
}

// ---------------------------------------------------------------------------
struct SweepAArgs {
    const double *V;   // [tile][5][64] primvars (FROM_U = false) or the state U (FROM_U)
    const double *Gc;  // [nb/64][5][64] ghost of the cell-centre state
    double *FV;        // [tile][4][5][64]; k_sweepA_face: per block [5][nf] fluxes of its own faces
    double *H;         // k_sweepA_face: [tile][5][64] face values of the records
    double *dt_part;   // per-block CFL dt minimum, or null
    double *dt_cell;   // [N] per-cell CFL step (local time stepping), or null
    double CFL;
    int xcd_remap;
    double *grad_aux;  // [N][15] column-major 5x3 per cell, or null
    double *psi_aux;   // [N][5] or null
    const uint32_t *aux_row;  // device cell -> row of grad_aux and psi_aux (reference cell)
    BndArgs bnd;       // FUSE: ghosts of the reconstructed face states (out: Gf)
    int hllc;          // k_sweepA_face: the flux
};

// One 64-cell tile of sweep A: its loads (tileA_issue) and the rest
// (tileA_run).
//
// ORDER: 0 first order, 1 second order without limiter, 2 second order Barth.
// FROM_U: a.V holds the stage's state U and the sweep evaluates the
// primvars itself (cons_to_prim of the own cell and of the neighbours it
// gathers; neighbours in the tile come from the LDS copy of the own values),
// so that sweep B need not store them.
struct TileA {
    uint32_t c, p;  // cell (clamped for padding lanes), device position
    bool live;
    uint32_t code, w[4];
    NodeTableLoad ntl;
    double Vc[5], Vn[4][5];
    const double *nsrc[4];
    bool loc[4];
};

template <int ORDER, int B, bool FROM_U>
__device__ __forceinline__ void tileA_issue(const DevMesh &m, const SweepAArgs &a, TileA &t) {
    const uint32_t c = t.c, p = t.p;
    // all loads first: own state, neighbour states (or ghost states), nodes
    t.code = m.fcode[c];
    const uint4 w4 = *reinterpret_cast<const uint4 *>(m.nbr + 4 * (size_t)c);
    t.w[0] = w4.x, t.w[1] = w4.y, t.w[2] = w4.z, t.w[3] = w4.w;
    t.ntl = node_table_issue(m, p);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int k = 0; k < 5; ++k) t.Vc[k] = a.V[tix(c, k)];  // (U if FROM_U: converted in tileA_run)
    // neighbour (or ghost) states; ghosts are tiled like V, so every source
    // has the same stride and the five loads share one address.  A neighbour
    // in the lane's own block (83 % of interior faces in Morton order at
    // 256 cells; 71 % within one 64-cell tile) is read from the block's copy
    // of its states in LDS instead (NF_A_LDS): the gathers are exec-masked
    // to the other lanes, which is what saves time (the texture path's work
    // grows with the lanes that access memory).  Every cell of the block is
    // a lane of it and live, since neighbours are real cells.  The gathers go first: the waits for the node and state loads
    // then cover them too (masked loads cannot be counted), which measured
    // faster than issuing them after the LDS copies (1.04 vs 0.93 ms).
#pragma unroll
    for (int s = 0; s < 4; ++s) {
        const uint32_t idx = t.w[s] & 0x1FFFFFFFu;
        t.nsrc[s] = ((t.w[s] & 0x80000000u) ? a.Gc : a.V) + tix(idx, 0);
        t.loc[s] = NF_A_LDS && !(t.w[s] & 0x80000000u) &&
                   (NF_A_LDS == 2 ? (idx / B) == (p / B) : (idx >> 6) == (p >> 6));
    }
    if (ORDER != 0) {
#pragma unroll
        for (int s = 0; s < 4; ++s)
            if (!t.loc[s]) {
#pragma unroll
                for (int k = 0; k < 5; ++k) t.Vn[s][k] = ldg(t.nsrc[s] + k * TILE);
            }
    }
}

// the tile's gradient, limiter and face values; returns the cell's CFL step
// (DBL_MAX for padding lanes or without a.dt_part)
template <int ORDER, int B, bool FROM_U>
__device__ __forceinline__ double tileA_run(const DevMesh &m, const SweepAArgs &a, TileA &t, double *lds,
                                            double *ldsv) {
    const uint32_t c = t.c, p = t.p, code = t.code;
    const bool live = t.live;
    const uint32_t *w = t.w;
    const bool *loc = t.loc;
    double *Vc = t.Vc;
    double(*Vn)[5] = t.Vn;
    if (FROM_U) {
        const double Uc[5] = {Vc[0], Vc[1], Vc[2], Vc[3], Vc[4]};
        cons_to_prim_d(Uc, Vc);
    }
    double *vt = ldsv + (NF_A_LDS ? (threadIdx.x >> 6) * 5 * TILE : 0);
    if (NF_A_LDS && ORDER != 0) {
#pragma unroll
        for (int k = 0; k < 5; ++k) vt[k * TILE + (p & 63u)] = Vc[k];
    }
    CellGeo g;
    // (its wave-level fences also order the state writes above before the
    // reads below)
    const NodeView nv = node_table_finish<B>(m, p, t.ntl, lds, g);
    if (NF_A_LDS == 2 && ORDER != 0) __syncthreads();  // every wave's states are in LDS
    cell_geo(m, g);
    V3d S[4], r[4];
#pragma unroll
    for (int s = 0; s < 4; ++s) face_geo(m, g, nv, (code >> (8 * s)) & 0xFFu, S[s], &r[s]);
    __builtin_amdgcn_sched_barrier(0);
    if (FROM_U && ORDER != 0) {
        // gathered neighbour states to primvars (ghost values already are)
#pragma unroll
        for (int s = 0; s < 4; ++s)
            if (!loc[s] && !(w[s] & 0x80000000u)) {
                const double Un[5] = {Vn[s][0], Vn[s][1], Vn[s][2], Vn[s][3], Vn[s][4]};
                cons_to_prim_d(Un, Vn[s]);
            }
    }
    if (NF_A_LDS && ORDER != 0) {
#pragma unroll
        for (int s = 0; s < 4; ++s)
            if (loc[s]) {
                const uint32_t idx = w[s] & 0x1FFFFFFFu, j = idx & 63u;
                const double *src = NF_A_LDS == 2 ? ldsv + ((idx >> 6) - (p & ~(uint32_t)(B - 1)) / TILE) * 5 * TILE : vt;
#pragma unroll
                for (int k = 0; k < 5; ++k) Vn[s][k] = src[k * TILE + j];
            }
        if (NF_A_LDS == 2) __syncthreads();  // before the slices are reused for the stores
    }

    if (ORDER == 0) {
        if (live) {
#pragma unroll
            for (int s = 0; s < 4; ++s)
#pragma unroll
                for (int k = 0; k < 5; ++k) a.FV[fix(c, s, k)] = Vc[k];
        }
    } else {
        // face normals as the cell adds them: -S where the cell is the
        // reference's neighbour j (cell j subtracts tmp/vol); in place, as
        // the time step below uses |S| only
#pragma unroll
        for (int s = 0; s < 4; ++s) {
            const uint32_t mneg = ((code >> (8 * s + 7)) & 1u) ? 0u : 0x80000000u;
            S[s] = {flip(S[s].x, mneg), flip(S[s].y, mneg), flip(S[s].z, mneg)};
        }
        // One variable at a time: gradient row k, its neighbour min/max, the
        // Barth factor and the face values depend on variable k only.
#pragma unroll
        for (int k = 0; k < 5; ++k) {
            // Green-Gauss (include/Numerics.hpp:112-127): cell i adds tmp/vol,
            // cell j subtracts it, faces in reference order
            double g0 = 0.0, g1 = 0.0, g2 = 0.0;
            double vmax = Vc[k], vmin = Vc[k];
#pragma unroll
            for (int s = 0; s < 4; ++s) {
                // 0.5 (V_i + V_j) is symmetric in i, j; the non-owner subtracts
                // (through the flipped S: the sign carries through the
                // product and the division exactly)
                const double uf = 0.5 * (Vc[k] + Vn[s][k]);
                g0 = g0 + rdiv(uf * S[s].x, g.ivol);
                g1 = g1 + rdiv(uf * S[s].y, g.ivol);
                g2 = g2 + rdiv(uf * S[s].z, g.ivol);
                if (ORDER == 2) {
                    // neighbour min/max (include/Numerics.hpp:276-291): the
                    // maximum of {v, v_j} over the faces, one v_j at a time
                    vmax = dmax(vmax, Vn[s][k]);
                    vmin = dmin(vmin, Vn[s][k]);
                }
            }
            double delta[4];
#pragma unroll
            for (int s = 0; s < 4; ++s) delta[s] = (g0 * r[s].x + g1 * r[s].y) + g2 * r[s].z;
            const double psi = (ORDER == 2) ? barth_psi_d(delta, vmax, vmin, Vc[k]) : 1.0;
            // limited reconstruction (include/Numerics.hpp:135-145)
            if (NF_A_LDS && NF_A_STX4) {
                // The wave's four rows (s, k) of the tile are written with
                // 16-byte stores: the values pass through the LDS slice (free
                // once the neighbour states are read), and lane l stores the
                // values of lanes 2(l%32), 2(l%32)+1 of slots l/32 and l/32+2.
                // Padding lanes store too: no real cell reads their entries.
                const uint32_t lane = p & 63u;
                __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
                __builtin_amdgcn_wave_barrier();
                __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
#pragma unroll
                for (int s = 0; s < 4; ++s) vt[s * TILE + lane] = Vc[k] + psi * delta[s];
                __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
                __builtin_amdgcn_wave_barrier();
                __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
                const double2 v0 = reinterpret_cast<const double2 *>(vt)[lane];
                const double2 v1 = reinterpret_cast<const double2 *>(vt)[lane + TILE];
                double *row = a.FV + fix(p & ~63u, lane >> 5, k) + 2 * (lane & 31u);
                *reinterpret_cast<double2 *>(row) = v0;
                *reinterpret_cast<double2 *>(row + 2 * 5 * TILE) = v1;
            } else if (live) {
#pragma unroll
                for (int s = 0; s < 4; ++s) a.FV[fix(c, s, k)] = Vc[k] + psi * delta[s];
            }
            if (live) {
                if (a.grad_aux) {
                    const size_t row = a.aux_row[c];
                    a.grad_aux[15 * row + k] = g0;
                    a.grad_aux[15 * row + k + 5] = g1;
                    a.grad_aux[15 * row + k + 10] = g2;
                    a.psi_aux[5 * row + k] = psi;
                }
            }
            __builtin_amdgcn_sched_barrier(0);
        }
    }
    double dtc = DBL_MAX;
    if (a.dt_part) {
        const double tc = cell_dt(Vc, S, w, g.vol, a.CFL);
        dtc = (live && tc < DBL_MAX) ? tc : DBL_MAX;  // NaN/+inf never win std::min
        if (a.dt_cell && live) a.dt_cell[c] = tc;
    }
    return dtc;
}

template <int ORDER, int B, bool FROM_U, bool FUSE>
__global__ __launch_bounds__(B) NF_SWEEP_ATTR void k_sweepA(DevMesh m, SweepAArgs a) {
    __shared__ double sh[B / 64];
    __shared__ double lds[12 * B];
    __shared__ __align__(16) double ldsv[NF_A_LDS ? 5 * B : 2];  // [wave][5][64] own states
    const LaneCell L = lane_cell<B>(m, a.xcd_remap);
    BndRange br{0, 0};
    if (FUSE) br = bnd_range<B>(a.bnd.boff, L.lb);
    if (m.st[L.inst].stop) return;
    TileA t;
    t.c = L.c;
    t.live = L.live;
    t.p = L.lb * B + threadIdx.x;
    tileA_issue<ORDER, B, FROM_U>(m, a, t);
    __builtin_amdgcn_sched_barrier(0);
    const double dtc = tileA_run<ORDER, B, FROM_U>(m, a, t, lds, ldsv);
    if (FUSE) bnd_ghosts<B, GhostOf::FV>(a.bnd, br, L.inst, a.FV);
    if (a.dt_part) {
        const double v = block_reduce<true, B>(dtc, sh);
        if (threadIdx.x == 0) a.dt_part[L.lb] = v;
    }
}

// Second-order sweeps over the faces of blocks of 256 cells, as long as every
// block's LDS fits: with the Morton order (at most some 330 records per block)
// and the input order of a generated box (360), not with reverse Cuthill-McKee,
// whose fronts give a block up to 1,024 records.  Of a block's 1,024 cell sides
// some 830 belong to 415 faces between its own cells; the other 200 are its
// records.  Sweep A gathers and converts the records' outside states once,
// one per lane, and keeps them in LDS beside the block's own; reconstructs
// every cell; passes the face values through LDS; and one lane per face then
// evaluates the flux of a face of the block, once instead of once from either
// side.  It stores those fluxes and the records' face values, 97 B per cell;
// sweep B evaluates the records' fluxes only, and sums every cell's four in
// slot order.  Against the sweeps that gather per lane and pass all 160 B of
// face values through memory (k_sweepA, k_sweepB): 470 instead of 650 B per
// cell and stage, 620 instead of 1,024 flux evaluations per block.  TVD-RK3
// step, farfield box / bump channel: 63k / 60k cells 63.5 / 63.5 -> 60.7 /
// 61.5 us, 215k / 202k 156 / 149 -> 136 / 130, 998k / 1,054k 488 / 510 -> 382
// / 415, 3.95M / 4.14M 1,929 / 1,904 -> 1,471 / 1,593.
//
// Sweep A is bound by its phases between barriers: the vector units are busy
// 60 % of its time, memory moves 2.9 TB/s (207 B per cell).  52 KB of LDS hold three blocks per
// CU; the face values in two halves (33 KB, 128 registers, four blocks) cost
// more in barriers than they gain: 382 -> 410 us at 998k cells.
template <int ORDER, bool FROM_U, bool FUSE>
__global__ __launch_bounds__(BLOCK) __attribute__((amdgpu_waves_per_eu(3, 3))) void k_sweepA_face(DevMesh m, SweepAArgs a) {
    constexpr int B = BLOCK;
    static_assert(ORDER != 0, "a first-order sweep needs no neighbours");
    __shared__ double sh[B / 64];
    // node tables and [cell][5] the states of the block and of its halo; later
    // [5][1024] the face values of all cell sides and [3][512] face vectors
    extern __shared__ __align__(16) double lds[];
    double *vs = lds + 12 * m.nstride;
    const LaneCell L = lane_cell<B>(m, a.xcd_remap);
    const uint32_t f0 = m.foff[L.lb], nf = m.foff[L.lb + 1] - f0, r0 = m.roff[L.lb], nr = m.roff[L.lb + 1] - r0;
    BndRange br{0, 0};
    if (FUSE) br = bnd_range<B>(a.bnd.boff, L.lb);
    if (m.st[L.inst].stop) return;
    const uint32_t c = L.c, t = threadIdx.x, p = L.lb * B + t;
    const bool live = L.live;

    const uint32_t hw = m.hal[r0 + (t < nr ? t : 0)];  // (one entry past the end is there)
    const uint32_t code = m.fcode[c];
    const uint2 nb = m.cell_nb[p], fx = m.cell_fx[p];
    const NodeTableLoad ntl = node_table_issue(m, p);
    __builtin_amdgcn_sched_barrier(0);
    double Vc[5], Vh[5];
#pragma unroll
    for (int k = 0; k < 5; ++k) Vc[k] = a.V[tix(c, k)];
    auto halo_load = [&](uint32_t w) {
        const double *src = ((w & 0x80000000u) ? a.Gc : a.V) + tix(w & 0x1FFFFFFFu, 0);
#pragma unroll
        for (int k = 0; k < 5; ++k) Vh[k] = ldg(src + k * TILE);
    };
    auto halo_store = [&](uint32_t h, uint32_t w) {
        if (FROM_U && !(w & 0x80000000u)) {  // (ghosts are primvars already)
            const double Uh[5] = {Vh[0], Vh[1], Vh[2], Vh[3], Vh[4]};
            cons_to_prim_d(Uh, Vh);
        }
#pragma unroll
        for (int k = 0; k < 5; ++k) vs[5 * (B + h) + k] = Vh[k];
    };
    if (t < nr) halo_load(hw);
    __builtin_amdgcn_sched_barrier(0);
    CellGeo g;
    const NodeView nv = node_table_finish<B>(m, p, ntl, lds, g, m.nstride);
    if (FROM_U) {
        const double Uc[5] = {Vc[0], Vc[1], Vc[2], Vc[3], Vc[4]};
        cons_to_prim_d(Uc, Vc);
    }
#pragma unroll
    for (int k = 0; k < 5; ++k) vs[5 * t + k] = Vc[k];
    if (t < nr) halo_store(t, hw);
    for (uint32_t h = t + B; h < nr; h += B) {
        const uint32_t w = m.hal[r0 + h];
        halo_load(w);
        halo_store(h, w);
    }
    cell_geo(m, g);
    V3d S[4], r[4];
#pragma unroll
    for (int s = 0; s < 4; ++s) face_geo(m, g, nv, (code >> (8 * s)) & 0xFFu, S[s], &r[s]);
    __syncthreads();  // every wave's states are in LDS

    const uint32_t nbw[4] = {nb.x & 0xFFFFu, nb.x >> 16, nb.y & 0xFFFFu, nb.y >> 16};
    const double *vn[4];
#pragma unroll
    for (int s = 0; s < 4; ++s) vn[s] = vs + 5 * (nbw[s] & 0x7FFFu);
    // face normals as the cell adds them: -S where the cell is the
    // reference's neighbour j (cell j subtracts tmp/vol); in place, as
    // the time step below uses |S| only
#pragma unroll
    for (int s = 0; s < 4; ++s) {
        const uint32_t mneg = ((code >> (8 * s + 7)) & 1u) ? 0u : 0x80000000u;
        S[s] = {flip(S[s].x, mneg), flip(S[s].y, mneg), flip(S[s].z, mneg)};
    }
    double Vf[4][5];
    // one variable at a time, as in tileA_run; the face values wait in registers
    // until every wave has read its neighbours' states
#pragma unroll
    for (int k = 0; k < 5; ++k) {
        const double Vk = vs[5 * t + k];  // (kept there: ten registers fewer)
        double Vn[4];
#pragma unroll
        for (int s = 0; s < 4; ++s) Vn[s] = vn[s][k];
        double g0 = 0.0, g1 = 0.0, g2 = 0.0;
        double vmax = Vk, vmin = Vk;
#pragma unroll
        for (int s = 0; s < 4; ++s) {
            const double uf = 0.5 * (Vk + Vn[s]);
            g0 = g0 + rdiv(uf * S[s].x, g.ivol);
            g1 = g1 + rdiv(uf * S[s].y, g.ivol);
            g2 = g2 + rdiv(uf * S[s].z, g.ivol);
            if (ORDER == 2) {
                vmax = dmax(vmax, Vn[s]);
                vmin = dmin(vmin, Vn[s]);
            }
        }
        double delta[4];
#pragma unroll
        for (int s = 0; s < 4; ++s) delta[s] = (g0 * r[s].x + g1 * r[s].y) + g2 * r[s].z;
        const double psi = (ORDER == 2) ? barth_psi_d(delta, vmax, vmin, Vk) : 1.0;
#pragma unroll
        for (int s = 0; s < 4; ++s) Vf[s][k] = Vk + psi * delta[s];
        if (live && a.grad_aux) {
            const size_t o = a.aux_row[c];
            a.grad_aux[15 * o + k] = g0;
            a.grad_aux[15 * o + k + 5] = g1;
            a.grad_aux[15 * o + k + 10] = g2;
            a.psi_aux[5 * o + k] = psi;
        }
        // without a limiter computed here: sunk to their stores, they would keep
        // the gradients of all variables alive (168 registers and spills;
        // channel of 1.05M cells 422 -> 413 us; with it 382 -> 387)
        if (ORDER == 1) asm volatile("" : "+v"(Vf[0][k]), "+v"(Vf[1][k]), "+v"(Vf[2][k]), "+v"(Vf[3][k]));
        __builtin_amdgcn_sched_barrier(0);
    }
    double tc = DBL_MAX;
    if (a.dt_part) {
#pragma unroll
        for (int k = 0; k < 5; ++k) Vc[k] = vs[5 * t + k];
        uint32_t w[4];
#pragma unroll
        for (int s = 0; s < 4; ++s) w[s] = nbw[s] << 16;  // (bit 31: boundary)
        tc = cell_dt(Vc, S, w, g.vol, a.CFL);
        if (a.dt_cell && live) a.dt_cell[c] = tc;
    }
    __syncthreads();
    // every side's values, and each own face's vector from its owner, to LDS
    double *fS = lds + 5 * 4 * B;
    if (live) {
        const uint32_t pos[4] = {fx.x & 0x7FFFu, (fx.x >> 16) & 0x7FFFu, fx.y & 0x7FFFu, (fx.y >> 16) & 0x7FFFu};
#pragma unroll
        for (int s = 0; s < 4; ++s) {
#pragma unroll
            for (int k = 0; k < 5; ++k) lds[k * 4 * B + pos[s]] = Vf[s][k];
            if (pos[s] < nf) {
                fS[pos[s]] = S[s].x;
                fS[2 * B + pos[s]] = S[s].y;
                fS[4 * B + pos[s]] = S[s].z;
            }
        }
    }
    __syncthreads();
    for (uint32_t h = t; h < nr; h += B) {
#pragma unroll
        for (int k = 0; k < 5; ++k) a.H[tix(r0 + h, k)] = lds[k * 4 * B + 2 * nf + h];
    }
    for (uint32_t f = t; f < nf; f += B) {
        double Vo[5], Vn[5], UO[5], UN[5], F[5];
#pragma unroll
        for (int k = 0; k < 5; ++k) {
            Vo[k] = lds[k * 4 * B + f];
            Vn[k] = lds[k * 4 * B + nf + f];
        }
        const V3d Sf = {fS[f], fS[2 * B + f], fS[4 * B + f]};
        prim_to_cons(Vo, UO);
        prim_to_cons(Vn, UN);
        if (a.hllc) hllc_d(UO, UN, Sf, F);
        else rusanov_side(UO, UN, Sf, 0u, F);
#pragma unroll
        for (int k = 0; k < 5; ++k) a.FV[5 * (size_t)f0 + k * (size_t)nf + f] = F[k];
    }
    if (FUSE) bnd_ghosts<B, GhostOf::REC>(a.bnd, br, L.inst, a.H);
    if (a.dt_part) {
        const double v = block_reduce<true, B>((live && tc < DBL_MAX) ? tc : DBL_MAX, sh);
        if (t == 0) a.dt_part[L.lb] = v;
    }
}

// Faces and records of the blocks, numbered in the order of the cells' slots.
// COUNT: foff[b + 1], roff[b + 1] = their numbers.  Otherwise, from the
// offsets, the tables of DevMesh but rec, and side_rec [cell][4], the record
// of each side.
struct FaceTables {
    uint32_t *foff, *roff, *hal, *rec, *brec, *side_rec;
    uint2 *cell_nb, *cell_fx;
};
template <bool COUNT>
__global__ __launch_bounds__(BLOCK) void k_block_faces(DevMesh m, FaceTables o) {
    __shared__ uint32_t sum[BLOCK];      // faces | records << 16
    __shared__ uint16_t face[4 * BLOCK];
    __shared__ uint2 last[2];
    const uint32_t b = blockIdx.x, t = threadIdx.x, p0 = b * BLOCK, p = p0 + t;
    const bool live = p < m.inst_end[m.blk_inst[b]];
    const uint4 w4 = *reinterpret_cast<const uint4 *>(m.nbr + 4 * (size_t)p);
    const uint32_t w[4] = {w4.x, w4.y, w4.z, w4.w};
    bool out[4], first[4];
    uint32_t j[4], n = 0;
#pragma unroll
    for (uint32_t q = 0; q < 4; ++q) {
        const uint32_t idx = w[q] & 0x1FFFFFFFu;
        out[q] = (w[q] & 0x80000000u) || idx / BLOCK != b;
        j[q] = 4 * (idx - p0) + ((w[q] >> 29) & 3u);  // the other side's place in the block
        first[q] = !out[q] && 4 * t + q < j[q];
        if (live) n += (first[q] ? 1u : 0u) + (out[q] ? 0x10000u : 0u);
    }
    sum[t] = n;
    __syncthreads();
    for (uint32_t d = 1; d < BLOCK; d *= 2) {
        const uint32_t v = t >= d ? sum[t - d] : 0;
        __syncthreads();
        sum[t] += v;
        __syncthreads();
    }
    const uint32_t nf = sum[BLOCK - 1] & 0xFFFFu, nr = sum[BLOCK - 1] >> 16;
    if (COUNT) {
        if (t == 0) o.foff[b + 1] = nf, o.roff[b + 1] = nr;
        return;
    }
    uint32_t f = (sum[t] - n) & 0xFFFFu, h = (sum[t] - n) >> 16, nb[4], fx[4];
#pragma unroll
    for (uint32_t q = 0; q < 4; ++q)
        if (live && first[q]) face[4 * t + q] = (uint16_t)f++;
    __syncthreads();
    const uint32_t code = m.fcode[p];
#pragma unroll
    for (uint32_t q = 0; q < 4; ++q) {
        if (!live) continue;
        const uint32_t own = (code >> (8 * q + 7)) & 1u;
        if (out[q]) {
            const uint32_t r = o.roff[b] + h;
            o.hal[r] = w[q] & 0x9FFFFFFFu;
            o.side_rec[4 * (size_t)p + q] = r;
            nb[q] = (w[q] & 0x80000000u) >> 16 | (BLOCK + h);
            fx[q] = own << 15 | (2 * nf + h++);
        } else {
            const uint32_t g = face[first[q] ? 4 * t + q : j[q]];
            nb[q] = j[q] / 4;
            fx[q] = own << 15 | (own ? g : nf + g);
        }
    }
    if (live) {
        const uint2 a = make_uint2(nb[0] | nb[1] << 16, nb[2] | nb[3] << 16);
        const uint2 c = make_uint2(fx[0] | fx[1] << 16, fx[2] | fx[3] << 16);
        o.cell_nb[p] = a;
        o.cell_fx[p] = c;
        if (t == BLOCK - 1 || p + 1 == m.inst_end[m.blk_inst[b]]) last[0] = a, last[1] = c;
    }
    __syncthreads();
    if (!live) o.cell_nb[p] = last[0], o.cell_fx[p] = last[1];  // padding: as the last cell
}

// rec and brec, once every block has numbered its records
__global__ __launch_bounds__(BLOCK) void k_link_records(DevMesh m, FaceTables o) {
    const uint32_t b = blockIdx.x, p = b * BLOCK + threadIdx.x;
    if (b + 1 == gridDim.x && threadIdx.x == 0) {  // (read, not used, by a block without records)
        const uint32_t n = o.roff[gridDim.x];
        o.hal[n] = 0;
        o.rec[n] = 0;
    }
    if (p >= m.inst_end[m.blk_inst[b]]) return;
    const uint32_t code = m.fcode[p];
    for (uint32_t q = 0; q < 4; ++q) {
        const uint32_t w = m.nbr[4 * (size_t)p + q], idx = w & 0x1FFFFFFFu;
        const bool bnd = w & 0x80000000u;
        if (!bnd && idx / BLOCK == b) continue;
        const uint32_t r = o.side_rec[4 * (size_t)p + q];
        if (bnd) o.brec[idx] = r;
        o.rec[r] = rec_word(bnd, (code >> (8 * q + 7)) & 1u,
                            bnd ? idx : o.side_rec[4 * (size_t)idx + ((w >> 29) & 3u)]);
    }
}

// Face vectors of the records and cell volumes, with the sweeps' arithmetic.
__global__ __launch_bounds__(BLOCK) void k_rec_geo(DevMesh m, double *rS, double *vol) {
    __shared__ double lds[12 * BLOCK];
    const LaneCell L = lane_cell<BLOCK>(m, 0);
    const uint32_t p = L.lb * BLOCK + threadIdx.x;
    const uint32_t nf = m.foff[L.lb + 1] - m.foff[L.lb], r0 = m.roff[L.lb], code = m.fcode[L.c];
    const uint2 fx = m.cell_fx[p];
    const NodeTableLoad ntl = node_table_issue(m, p);
    CellGeo g;
    const NodeView nv = node_table_finish<BLOCK>(m, p, ntl, lds, g);
    cell_geo(m, g);
    vol[p] = g.vol;
    if (!L.live) return;
    const uint32_t pos[4] = {fx.x & 0x7FFFu, (fx.x >> 16) & 0x7FFFu, fx.y & 0x7FFFu, (fx.y >> 16) & 0x7FFFu};
#pragma unroll
    for (int s = 0; s < 4; ++s) {
        if (pos[s] < 2 * nf) continue;
        V3d S;
        face_geo(m, g, nv, (code >> (8 * s)) & 0xFFu, S, nullptr);
        const uint32_t r = r0 + pos[s] - 2 * nf;
        const size_t o = ((size_t)(r >> 6) * 3) * TILE + (r & 63u);
        rS[o] = S.x;
        rS[o + TILE] = S.y;
        rS[o + 2 * TILE] = S.z;
    }
}

// ---------------------------------------------------------------------------
struct SweepBArgs {
    const double *FV;       // [tile][4][5][64]; k_sweepB_face: per block [5][nf] fluxes
    const double *H;        // k_sweepB_face: [tile][5][64] face values of the records
    const double *Gf;       // [nb/64][5][64] ghost of the reconstructed face state
    const double *U;        // [tile][5][64] state entering the stage
    const double *Uo;       // U_old (U^n)
    double *Uout;           // (may alias U)
    const double *dt_cell;  // per-cell step (local time stepping), or null
    int kind;               // 1: U + dt/vol R, 2: RK3 stage 2, 3: RK3 stage 3
    double *res_part;       // per-block sum of R_rho^2, or null
    int check;
    int xcd_remap;
    double *R_aux;          // [N][5] or null: store R, skip the update
    const uint32_t *aux_row;  // device cell -> row of R_aux (reference cell)
    double *Rst, *fst;      // checked stage: R [tile][5][64] and f [cell] for k_apply, no update
    BndArgs bnd;            // FUSE: ghosts of the updated cell states (out: Gc), where it updates
};

// The end of sweep B of a cell with flux balance R: checks, what is kept of R,
// the stage's update and the residual.
template <int B, bool FUSE>
__device__ __forceinline__ void finish_cell(const DevMesh &m, const SweepBArgs &a, const LaneCell &L, BndRange br,
                                            InstState &st, const double *R, bool zero_old, const double *Up,
                                            const double *Uop, const Rcp &ivol, double *sh) {
    const uint32_t c = L.c;
    const bool live = L.live;
    if (live && a.check) {
        bool ok = true;
#pragma unroll
        for (int k = 0; k < 5; ++k) ok = ok && (R[k] - R[k] == 0.0);
        if (!ok) atomicAdd(&st.bad_flux, 1);
    }
    if (a.R_aux) {
        if (live) {
#pragma unroll
            for (int k = 0; k < 5; ++k) a.R_aux[5 * (size_t)a.aux_row[c] + k] = R[k];
        }
    } else {
        const double dt = a.dt_cell ? a.dt_cell[c] : st.dt;
        // Solver::TVD_RK3 / explicit_euler (src/Solver.cpp:98-132)
        const double f = rdiv(a.kind == 1 ? dt : (a.kind == 2 ? 1.0 / 4.0 * dt : 2.0 / 3.0 * dt), ivol);
        if (a.Rst) {
            if (live) {
#pragma unroll
                for (int k = 0; k < 5; ++k) a.Rst[tix(c, k)] = R[k];
                a.fst[c] = f;
            }
        } else {
            double Un[5], Vnew[5];
            stage_combine(a.kind, zero_old, f, Up, Uop, R, Un);
            cons_to_prim_d(Un, Vnew);
            if (live) {
#pragma unroll
                for (int k = 0; k < 5; ++k) a.Uout[tix(c, k)] = Un[k];
                if (!(Vnew[0] > 0.0) || !(Vnew[4] > 0.0) || !(Un[4] > 0.0)) atomicAdd(&st.bad_state, 1);
            }
            if (FUSE) bnd_ghosts<B, GhostOf::U>(a.bnd, br, L.inst, a.Uout);
        }
    }
    if (a.res_part) {
        const double r2 = live ? R[0] * R[0] : 0.0;
        const double v = block_reduce<false, B>(r2, sh);
        if (threadIdx.x == 0) a.res_part[L.lb] = v;
    }
}

// FLUX: 0 Rusanov, 1 HLLC
template <int B, int FLUX, bool FUSE>
__global__ __launch_bounds__(B) NF_SWEEPB_ATTR void k_sweepB(DevMesh m, SweepBArgs a) {
    __shared__ double sh[B / 64];
    __shared__ double lds[12 * B];
    const LaneCell L = lane_cell<B>(m, a.xcd_remap);
    BndRange br{0, 0};
    if (FUSE) br = bnd_range<B>(a.bnd.boff, L.lb);
    InstState &st = m.st[L.inst];
    if (st.stop) return;
    const uint32_t c = L.c;
    const bool live = L.live;

    const uint32_t code = m.fcode[c];
    const uint4 w4 = *reinterpret_cast<const uint4 *>(m.nbr + 4 * (size_t)c);
    const uint32_t w[4] = {w4.x, w4.y, w4.z, w4.w};
    const NodeTableLoad ntl = node_table_issue(m, L.lb * B + threadIdx.x);
    __builtin_amdgcn_sched_barrier(0);
    CellGeo g;
    NodeView nv;
    double R[5] = {0.0, 0.0, 0.0, 0.0, 0.0};
    const bool zero_old = st.uold_zero;
    double Up[5], Uop[5];
    {
        // loaded first, outside the stage-kind branches (stage 1 and a zero
        // U_old read U twice: same lines, no branch)
        const double *uo = (a.kind == 1 || zero_old) ? a.U : a.Uo;
#pragma unroll
        for (int k = 0; k < 5; ++k) {
            Up[k] = a.U[tix(c, k)];
            Uop[k] = uo[tix(c, k)];
        }
    }
    // face values of both sides, one face at a time, the next face's loads
    // issued before the current face is computed
    double Vo4[4][5], Vn4[4][5];
    auto load_face = [&](int s) {
        const uint32_t idx = w[s] & 0x1FFFFFFFu, sn = (w[s] >> 29) & 3u;
        const bool bnd = w[s] & 0x80000000u;
        const double *src = bnd ? a.Gf + tix(idx, 0) : a.FV + fix(idx, sn, 0);
#pragma unroll
        for (int k = 0; k < 5; ++k) {
            Vo4[s][k] = a.FV[fix(c, s, k)];
            Vn4[s][k] = src[k * TILE];
        }
    };
    load_face(0);
    nv = node_table_finish<B>(m, L.lb * B + threadIdx.x, ntl, lds, g);
    cell_geo(m, g);
#pragma unroll
    for (int s = 0; s < 4; ++s) {
        if (s + 1 < 4) load_face(s + 1);
        __builtin_amdgcn_sched_barrier(0);
        const uint32_t byte = (code >> (8 * s)) & 0xFFu;
        V3d S;
        face_geo(m, g, nv, byte, S, nullptr);
        // interior faces (src/Solver.cpp:171-192), boundary faces (:197-229)
        double UO[5], UN[5], F[5];
        prim_to_cons(Vo4[s], UO);
        prim_to_cons(Vn4[s], UN);
        const uint32_t mneg = (byte & 0x80u) ? 0u : 0x80000000u;
        if (FLUX == 1) {
            // F(U_i side, U_j side, S_ij) on both cells of the face
            const bool own = byte & 0x80u;
            double UL[5], UR[5];
#pragma unroll
            for (int k = 0; k < 5; ++k) {
                UL[k] = own ? UO[k] : UN[k];
                UR[k] = own ? UN[k] : UO[k];
            }
            hllc_d(UL, UR, S, F);
        } else {
            rusanov_side(UO, UN, S, mneg, F);
        }
#pragma unroll
        for (int k = 0; k < 5; ++k) R[k] = R[k] + flip(F[k], mneg ^ 0x80000000u);  // R_i -= F, R_j += F
        // the face's flux is complete here: without this the compiler sinks
        // every face's arithmetic below the last face's loads, and all four
        // faces' values are live at once
        asm volatile("" : "+v"(R[0]), "+v"(R[1]), "+v"(R[2]), "+v"(R[3]), "+v"(R[4]) : : "memory");
    }
    finish_cell<B, FUSE>(m, a, L, br, st, R, zero_old, Up, Uop, g.ivol, sh);
}

// The records' fluxes, then every cell's flux balance from LDS.  273 B per cell
// move at 5.7 TB/s (998k cells: 48 us): bound by memory, with the vector units
// busy 23 % of the time.  Five waves per SIMD spill: 382 -> 472 us per step.
template <int FLUX, bool FUSE>
__global__ __launch_bounds__(BLOCK) void k_sweepB_face(DevMesh m, SweepBArgs a) {
    constexpr int B = BLOCK;
    __shared__ double sh[B / 64];
    extern __shared__ __align__(16) double fl[];  // [5][nent] fluxes of the block's faces, then of its records
    const LaneCell L = lane_cell<B>(m, a.xcd_remap);
    const uint32_t f0 = m.foff[L.lb], nf = m.foff[L.lb + 1] - f0, r0 = m.roff[L.lb], nr = m.roff[L.lb + 1] - r0;
    BndRange br{0, 0};
    if (FUSE) br = bnd_range<B>(a.bnd.boff, L.lb);
    InstState &st = m.st[L.inst];
    if (st.stop) return;
    const uint32_t c = L.c, t = threadIdx.x;
    const uint32_t rw = m.rec[r0 + (t < nr ? t : 0)];  // (one entry past the end is there)
    const uint2 fx = m.cell_fx[L.lb * B + t];
    double F[2][5];  // (a block has at most 2 B faces)
#pragma unroll
    for (int q = 0; q < 2; ++q)
        if (t + q * B < nf) {
#pragma unroll
            for (int k = 0; k < 5; ++k) F[q][k] = a.FV[5 * (size_t)f0 + k * (size_t)nf + t + q * B];
        }
    const bool zero_old = st.uold_zero;
    const double vol = m.vol[c];
    double Up[5], Uop[5];
    {
        const double *uo = (a.kind == 1 || zero_old) ? a.U : a.Uo;
#pragma unroll
        for (int k = 0; k < 5; ++k) {
            Up[k] = a.U[tix(c, k)];
            Uop[k] = uo[tix(c, k)];
        }
    }
    auto rec_flux = [&](uint32_t h, uint32_t w) {
        const uint32_t r = r0 + h;
        const double *src = ((w & REC_BOUNDARY) ? a.Gf : a.H) + tix(rec_index(w), 0);
        const double *sp = m.rS + (size_t)(r >> 6) * 3 * TILE + (r & 63u);
        double Vo[5], Vn[5], UO[5], UN[5], G[5];
#pragma unroll
        for (int k = 0; k < 5; ++k) {
            Vo[k] = a.H[tix(r, k)];
            Vn[k] = ldg(src + k * TILE);
        }
        const V3d S = {sp[0], sp[TILE], sp[2 * TILE]};
        prim_to_cons(Vo, UO);
        prim_to_cons(Vn, UN);
        const bool own = w & REC_OWNER;
        if (FLUX == 1) {
            double UL[5], UR[5];
#pragma unroll
            for (int k = 0; k < 5; ++k) {
                UL[k] = own ? UO[k] : UN[k];
                UR[k] = own ? UN[k] : UO[k];
            }
            hllc_d(UL, UR, S, G);
        } else {
            rusanov_side(UO, UN, S, own ? 0u : 0x80000000u, G);
        }
#pragma unroll
        for (int k = 0; k < 5; ++k) fl[k * m.nent + nf + h] = G[k];
    };
    if (t < nr) rec_flux(t, rw);
    for (uint32_t h = t + B; h < nr; h += B) rec_flux(h, m.rec[r0 + h]);
#pragma unroll
    for (int q = 0; q < 2; ++q)
        if (t + q * B < nf) {
#pragma unroll
            for (int k = 0; k < 5; ++k) fl[k * m.nent + t + q * B] = F[q][k];
        }
    __syncthreads();
    double R[5] = {0.0, 0.0, 0.0, 0.0, 0.0};
    const uint32_t fw[4] = {fx.x & 0xFFFFu, fx.x >> 16, fx.y & 0xFFFFu, fx.y >> 16};
#pragma unroll
    for (int s = 0; s < 4; ++s) {
        const uint32_t pos = fw[s] & 0x7FFFu, e = pos < nf ? pos : pos - nf;
        const uint32_t sub = (fw[s] & 0x8000u) << 16;  // R_i -= F, R_j += F
#pragma unroll
        for (int k = 0; k < 5; ++k) R[k] = R[k] + flip(fl[k * m.nent + e], sub);
    }
    finish_cell<B, FUSE>(m, a, L, br, st, R, zero_old, Up, Uop, rcp_of(vol), sh);
}

__global__ __launch_bounds__(BLOCK) void k_apply(DevMesh m, ApplyArgs a) { apply_stage_cell<double>(m, a); }

// prim of a tiled state: V = prim(U)
__global__ __launch_bounds__(BLOCK) void k_prim(const double *U, double *V, uint32_t N) {
    const uint32_t c = blockIdx.x * BLOCK + threadIdx.x;
    if (c >= N) return;
    double u[5], v[5];
#pragma unroll
    for (int k = 0; k < 5; ++k) u[k] = U[tix(c, k)];
    cons_to_prim_d(u, v);
#pragma unroll
    for (int k = 0; k < 5; ++k) V[tix(c, k)] = v[k];
}

// State across the boundary: reference-order AoS [N][5] (copied to the
// device as is) to the instance's device tiles, padding cells zero; perm is
// the instance's device cell -> reference cell map.
__global__ __launch_bounds__(BLOCK) void k_state_in(const double *aos, const uint32_t *perm, double *dev,
                                                    uint32_t N, uint32_t Npad) {
    const uint32_t p = blockIdx.x * BLOCK + threadIdx.x;
    if (p >= Npad) return;
    const size_t r = p < N ? 5 * (size_t)perm[p] : 0;
#pragma unroll
    for (int k = 0; k < 5; ++k) dev[tix(p, k)] = p < N ? aos[r + k] : 0.0;
}
// and back: device tiles (FP64, or FP32 primvars) to reference-order AoS
template <typename T>
__global__ __launch_bounds__(BLOCK) void k_state_out(const T *dev, const uint32_t *perm, double *aos, uint32_t N) {
    const uint32_t p = blockIdx.x * BLOCK + threadIdx.x;
    if (p >= N) return;
    const size_t r = 5 * (size_t)perm[p];
#pragma unroll
    for (int k = 0; k < 5; ++k) aos[r + k] = (double)dev[tix(p, k)];
}
// one state in every cell, padding cells zero
struct CellState {
    double v[5];
};
__global__ __launch_bounds__(BLOCK) void k_state_fill(CellState s, double *dev, uint32_t N, uint32_t Npad) {
    const uint32_t p = blockIdx.x * BLOCK + threadIdx.x;
    if (p >= Npad) return;
#pragma unroll
    for (int k = 0; k < 5; ++k) dev[tix(p, k)] = p < N ? s.v[k] : 0.0;
}
#endif  // NF_DEVICE_HELPERS_ONLY

}  // namespace nf
