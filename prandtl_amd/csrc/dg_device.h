// Device side of the DGSEM RHS (gfx950): tables and arguments, launch shapes,
// mesh and index helpers and the viscous kernel k_visc.
// Included by the library's host translation unit and by the per-order
// instantiation units.
//
// Two kernels per RHS evaluation:
//
//  k_visc_l (dg_visc_lines.h: boxes, corrected mode) or k_visc (meshes,
//  faithful mode, gradient output), parabolic only  u -> BR1 lifting of the entropy variables,
//      EntropyGrad2PrimGrad, viscous flux, contravariant transform and the
//      weak-form derivative sum D^ Fv of the volume term; writes the raw
//      viscous volume sum (nv-1 per node) and the face-normal component of
//      the viscous flux at every face node of the element (nv-1 per face
//      node).  Restates DGSEMOperator.cpp:82-159, LiftingBR1.cpp:10-272 and
//      DGSEMIntegrator.cpp:617-641,705-738 (and 435-549 for the face side).
//      The volume sum holds this element's half of the viscous face terms.
//
//  k_rhs_l (dg_lines.h; dg_points.h's k_rhs_p in 1-D and on small meshes)
//      the inviscid flux differencing,
//      surface fluxes, modal indicator and subcell FV blending, plus the
//      viscous volume/face terms from k_visc, then either writes the RHS
//      (Operator::Mult) or the RK3 stage combination.
//
// Both are also built for forced workgroup sizes (64, 128 or 256 threads,
// "launch shapes"); prandtl_autotune picks one per context by timing them on
// the caller's state.
#pragma once
#include <hip/hip_runtime.h>

#include <cmath>
#include <cstdint>
#include <cstdio>
#include <algorithm>
#include <cstring>
#include <filesystem>
#include <fstream>
#include <new>
#include <string>
#include <type_traits>
#include <vector>

#include "../../include/prandtl_hip.h"
#include "dg_physics.h"
#include "mesh.h"

namespace prandtl {

constexpr int MAXNP = 8;

#ifndef PRANDTL_WAVES
#define PRANDTL_WAVES 3
#endif

struct Tables {
    double D[MAXNP * MAXNP];    // D_ij (row-major), DGSEMIntegrator.cpp:58-69
    double Dh[MAXNP * MAXNP];   // D + E            (lines 71-74, un-transposed)
    double Dh2[MAXNP * MAXNP];  // 2D + E           (lines 76-80, un-transposed)
    double V1i[MAXNP * MAXNP];  // inverse 1-D shifted-Legendre Vandermonde
    double w[MAXNP];            // LGL weights on [0,1]
    double x[MAXNP];            // LGL nodes on [0,1]
    double subn[3][MAXNP];      // subcell normal magnitude per interface (1199-1304)
};

struct Geo {
    int n[3];
    int NE;
    double nrm[3];   // adj(r,r) = face measure of an r-face
    double inv_n0, inv_n01;   // 1 / n[0], 1 / (n[0] n[1]): box element index arithmetic
    double invJ;     // 1/J
    double aface;    // 1/(w_0 J)
    double nsc, insc;   // meshes: the power of two that brings the largest normal near 1, and its inverse
    int bcmask;      // boundary type (BC_*) of side (r, s) in bits 3(2r+s)..+2; 0: periodic box
    const double *bcs;    // device outer states of inflow / specified-state boundaries, 5 per
                          // box side [3][2] (Cartesian) or per attribute (unstructured meshes)
    // general geometry of quadrilateral and hexahedral meshes (null on
    // Cartesian boxes), local faces f = 2r + side; per-node tables hold DIM*DIM
    // adjugate entries, per-point normals DIM components
    const double *met;    // [4][NE*K] adjugate row r, component d at 2r+d
    const double *jac;    // [NE*K] Jacobian determinant
    const int *fface;     // [NE*4] bit 0: first element of the face; bits 1-3 boundary type; 4+: attribute-1
    const int *fnb;       // [NE*4*NFP] neighbour node e2*K + n2 of each interior face point
    const int *fnf;       // [NE*4] 2 (e2*4 + f2) + reversed: the neighbour's face of each interior face
    const double *fnor;   // [NE*4*NFP*2] normal outward of the face's first element
    const double *fxy;    // [NE*4*NFP*2] boundary face points' coordinates (quadrilateral meshes)
    const double *bfn;    // null, or per attribute [16]: a split outer state [kind, n0, n1, n2,
                          // offset, speed, below[5], above[5]] (0 kind: the constant state)
    const double *subn;   // [NE][2][NFP][NP-1][2] subcell interface normals
    const double *corner; // [NE][4][2] or [NE][8][3] element corners: the RHS forms its metrics from
                          // them, in 3-D k_visc too (met is not stored there)
    // axisymmetric quadrilateral meshes (null otherwise)
    const double *rnode;  // [NE*K] r = y of each node
    const int *axm;       // [NE*K] -1 off the axis, else 2 d + (1: radial RHS zeroed), d the descriptor
    const int *axj;       // [nax][3] element-local nodes j1, j2 (ray fit), jn (floor fallback); -1 none
    const double *axr;    // [nax][3] their r
    double axis_floor;    // density floor of the axis reconstruction
};

struct KArgs {
    Tables tab;
    Geo geo;
    Phys phys;
    int blend, parabolic, ec, quirks;
    int mode;             // 0: out = rhs; 1: out = y + dt rhs; 2: out = c0 u0 + c1 (y + dt rhs)
    double dt, c0, c1;
    const double *dtp;    // if set, dt is read from device memory (graph replays)
    const double *tp;     // if set, the time of the step's first stage (device memory)
    double tc;            // this stage's time is *tp + tc dt (RK3SSPSolver: 0, 1, 1/2)
    const double *y;      // the state (axisymmetric: the weighted state r U)
    const double *u0;
    double *out;
    const void *visc;     // [nv-1][NE][K]            (FP32 in the mixed form)
    const void *fvf;      // [NE][2 dim][nv-1][Nfp]   (FP32 in the mixed form)
    double *alpha;        // [NE]
    double *eta;          // [NE]
    double *lam;          // per-block running maxima [gridDim.x]
    const int *skip;      // if set and nonzero, the launch does nothing (a finished device loop)
};

// A (N+1)x(N+1) derivative matrix M with M[N-a][N-m] = -M[a][m] in even-odd
// form, H = NP/2 rows: e, o = (M[a][m] +- M[a][N-m]) / 2 at 4a + m, c the
// middle column, r the middle row (odd NP).
struct EvenOdd {
    double e[16], o[16], c[4], r[4];
};

struct VArgs {
    Tables tab;
    EvenOdd eD;           // D
    double iw0;           // 1/w_0

    Geo geo;
    Phys phys;
    int quirks;
    const double *y;
    void *visc;
    void *fvf;
    double *grad;         // optional [dim][nv][NE][K]
    const int *skip;      // as KArgs::skip
};

constexpr int cmx(int a, int b) { return a > b ? a : b; }
constexpr int r64(int x) { return ((x + 63) / 64) * 64; }
// NP^d: nodes per element (d = DIM) and per face (d = DIM - 1)
constexpr int npow(int NP, int d) { return d <= 0 ? 1 : NP * npow(NP, d - 1); }

// Launch shapes of both kernels: 0 natural, 1..3 forced blocks of 64, 128
// and 256 threads (autotuned per case).
constexpr int NSHAPES = PRANDTL_SHAPES;
constexpr int shape_fb(int shape) { return shape == 1 ? 64 : shape == 2 ? 128 : shape == 3 ? 256 : 0; }

// Launch shape of k_visc: one thread per node, BLOCK / K elements per
// workgroup.
constexpr int visc_block(int DIM, int NP, int FB)
{
    const int K = npow(NP, DIM);
    return FB ? FB : K > 256 ? r64(K) : 256;
}
constexpr bool visc_shape_ok(int DIM, int NP, int shape)
{
    if (shape == 0) return true;
    if (shape < 0 || shape >= NSHAPES) return false;
    const int K = npow(NP, DIM);
    const int fb = shape_fb(shape);
    return K <= fb && fb != visc_block(DIM, NP, 0);
}
template <int DIM, int NP, int FB = 0> struct VCfg {
    static constexpr int NV = DIM + 2;
    static constexpr int K = npow(NP, DIM);
    static constexpr int NFP = npow(NP, DIM - 1);
    static constexpr int BLOCK = visc_block(DIM, NP, FB);
    static constexpr int EPB = BLOCK / K;
    // waves per SIMD to ask the register allocator for
    static constexpr int WAVES = K > 256 ? 2 : BLOCK <= 128 ? 4 : PRANDTL_WAVES;
    static_assert(EPB >= 1, "one node per thread");
};

template <int DIM, int NP>
__device__ __forceinline__ int line_node(int r, int l, int m)
{
    if (DIM == 2) return r == 0 ? l * NP + m : m * NP + l;
    const int a = l % NP, b = l / NP;
    if (r == 0) return (b * NP + a) * NP + m;
    if (r == 1) return (b * NP + m) * NP + a;
    return (m * NP + b) * NP + a;
}

template <int DIM, int NP>
__device__ __forceinline__ int line_of(int r, int i, int j, int k)
{
    if (DIM == 2) return r == 0 ? j : i;
    if (r == 0) return k * NP + j;
    if (r == 1) return k * NP + i;
    return j * NP + i;
}

template <int NP> __device__ __forceinline__ int pair_index(int a, int b)
{
    // a < b; pairs ordered (0,1),(0,2),...,(0,N),(1,2),...
    return a * NP - (a * (a + 1)) / 2 + (b - a - 1);
}

__device__ __forceinline__ int xcd_remap(int bid, int nb)
{
    // blocks are dispatched round-robin over the 8 XCDs; give each XCD a
    // contiguous range of element groups so face neighbours share its L2
    const int q = nb >> 3, rr = nb & 7;
    const int x = bid & 7, k = bid >> 3;
    return (x < rr) ? x * (q + 1) + k : rr * (q + 1) + (x - rr) * q + k;
}

// q = e / d for 0 <= e < 2^31 and d >= 1 given dinv = 1/d: the truncated
// double-precision product is off by at most one, and one remainder test
// corrects it (cheaper than an integer division by a run-time divisor).
__device__ __forceinline__ int quot(int e, int d, double dinv)
{
    int q = (int)((double)e * dinv);
    const int rr = e - q * d;
    q += (rr >= d) ? 1 : 0;
    q -= (rr < 0) ? 1 : 0;
    return q;
}

// (i, j, k) of box element e, elements numbered x fastest
__device__ __forceinline__ void box_index(const Geo &g, int e, int *idx)
{
    const int n01 = g.n[0] * g.n[1];
    const int k = quot(e, n01, g.inv_n01);
    const int rem = e - k * n01;
    const int j = quot(rem, g.n[0], g.inv_n0);
    idx[0] = rem - j * g.n[0];
    idx[1] = j;
    idx[2] = k;
}

// The step size of a stage: the device value when the caller keeps dt on the
// device, else the argument.  Written as a branch on the pointer with the
// loaded value passed through an empty asm: a choice between the two loads
// would be compiled to one flat load through a selected address, and a
// flat load still in flight makes the next memory wait drain every
// outstanding load.
__device__ __forceinline__ double step_dt(const KArgs &A)
{
    double dt = A.dt;
    if (A.dtp) {
        double d = *A.dtp;
        asm volatile("" : "+v"(d));
        dt = d;
    }
    return dt;
}

// a, b or c for r = 0, 1, 2 where r differs between the lanes of a wave:
// the three values pass through an empty asm first, so the choice is between
// values, not a load through a selected address of the argument struct
__device__ __forceinline__ double lane_pick3(double a, double b, double c, int r)
{
    asm volatile("" : "+v"(a), "+v"(b), "+v"(c));
    return r == 0 ? a : r == 1 ? b : c;
}

// The element beside e's face (r, side), periodic, for callers whose direction
// r differs between the lanes of a wave (one thread per line or per face point
// of several directions).
// Indexing the argument struct with a per-lane r is a vector load from
// argument memory that the thread waits for before its state loads can
// issue; so is a select between the three fields, which the compiler turns
// into one load through a selected address.  The empty asm takes the three
// scalar-loaded values as they are, and the select is then between values.
__device__ __forceinline__ int neighbor_lane(const Geo &g, int e, int r, int side)
{
    int idx[3];
    box_index(g, e, idx);
    int n0 = g.n[0], n1 = g.n[1], n2 = g.n[2];
    asm volatile("" : "+s"(n0), "+s"(n1), "+s"(n2));
    const int nr = r == 0 ? n0 : r == 1 ? n1 : n2;
    idx[r] = side ? (idx[r] + 1 == nr ? 0 : idx[r] + 1) : (idx[r] == 0 ? nr - 1 : idx[r] - 1);
    return (idx[2] * g.n[1] + idx[1]) * g.n[0] + idx[0];
}

// Boundary type of element e's face (r, side), BC_PERIODIC for a face with
// a neighbour.
__device__ __forceinline__ int boundary_of(const Geo &g, int e, int r, int side)
{
    int ix[3];
    box_index(g, e, ix);
    const int idx = ix[r];
    const int nr = r == 0 ? g.n[0] : r == 1 ? g.n[1] : g.n[2];
    const bool at = side ? idx == nr - 1 : idx == 0;
    return at ? (g.bcmask >> (3 * (2 * r + side))) & 7 : BC_PERIODIC;
}

__device__ __forceinline__ double wave_max(double v)
{
    for (int off = 32; off > 0; off >>= 1) {
        const double o = __shfl_xor(v, off, 64);
        v = (v < o) ? o : v;
    }
    return v;
}

// Running maximum wave speed: each block keeps its own slot (one thread, a
// plain read-modify-write, no contention); prandtl_max_wave_speed reduces
// the slots when asked.  old: the slot's value, read by thread 0 when the
// block started (only this block writes the slot during a launch).  Non-finite speeds are ignored, as std::max(current,
// NaN) does in the reference (DGSEMIntegrator.cpp:270).
template <int BLOCK>
__device__ __forceinline__ void block_lam_max(double lam, double old, double *slots, double *sred, int slot)
{
    lam = wave_max(lam);
    const int w = threadIdx.x >> 6, lane = threadIdx.x & 63;
    if (lane == 0) sred[w] = lam;
    __syncthreads();
    if (threadIdx.x == 0) {
        double m = sred[0];
        for (int i = 1; i < (BLOCK + 63) / 64; i++) m = (m < sred[i]) ? sred[i] : m;
        if (old < m) slots[slot] = m;
    }
}

// Launch shapes of the RHS in two and three dimensions: which workgroup sizes
// a caller may force (PRANDTL_SHAPES).  The set is part of the interface, callers
// keep shapes that autotune found: it is that of workgroups with a thread for each
// of an element's nodes and pairs' jobs (rshape), other than the one that was the
// natural one for those.  Every size in it holds an element's lines.
struct RShape {
    int K, WORK, EPB, BLOCK;
};
constexpr RShape rshape(int DIM, int NP, bool BLEND, int FB)
{
    const int K = npow(NP, DIM);
    const int NFP = npow(NP, DIM - 1);
    const int JP = NFP * (NP * (NP - 1) / 2 + (BLEND ? NP - 1 : 0));
    const int WORK = cmx(K, cmx(JP, 2 * DIM * NFP));
    const int EPB = K > 128 ? 1 : cmx(1, (FB ? FB : 256) / WORK);
    const int BLOCK = FB ? FB : K > 256 ? r64(K) : (r64(EPB * WORK) > 512 ? 512 : r64(EPB * WORK));
    return RShape{K, WORK, EPB, BLOCK};
}
constexpr bool rhs_shape_ok(int DIM, int NP, bool BLEND, int shape)
{
    if (shape == 0) return true;
    if (shape < 0 || shape >= NSHAPES || DIM == 1) return false;
    const RShape n = rshape(DIM, NP, BLEND, 0);
    const RShape f = rshape(DIM, NP, BLEND, shape_fb(shape));
    return f.EPB * f.K <= f.BLOCK && !(f.EPB == n.EPB && f.BLOCK == n.BLOCK);
}

// DGSEMOperator::RecoverStateFromWeighted (DGSEMOperator.cpp:161-424) for one
// node q: U = rU / r off the axis; on it (low-order axis reconstruction, as
// an "axis" boundary selects) each of rho, rho u_z, rho E from the ray fit
// through the origin over the nodes j1, j2 of the node's descriptor,
// minmod-limited against 1.5 f_j / r_j and capped at 10 |f_j1| / r_j1 (one
// node: its f / r), radial momentum 0; a density below the floor, or a
// non-finite one or energy, takes node jn's state instead.  The nodes are
// chosen on the host from the geometry.
__device__ __forceinline__ double ax_minmod(double a, double b)
{
    if (a * b <= 0.0) return 0.0;
    const double m = fmin(fabs(a), fabs(b));
    return a > 0.0 ? m : -m;
}

__device__ __forceinline__ double ax_clamp(double x, double m)
{
    if (!isfinite(x)) return 0.0;
    if (fabs(x) <= m) return x;
    return x > 0.0 ? m : (x < 0.0 ? -m : 0.0);
}

// What a node's recovery loads in any case.  Apart from the rest, so that a
// thread with several nodes has all of these loads in flight at once.
struct AxNode {
    int code;
    double r, u[4];
};

__device__ __forceinline__ AxNode axis_load(const double *rU, const Geo &g, size_t NK, size_t q)
{
    AxNode n;
    n.code = g.axm[q];
    n.r = g.rnode[q];
#pragma unroll
    for (int v = 0; v < 4; v++) n.u[v] = rU[v * NK + q];
    return n;
}

__device__ __forceinline__ void axis_state(const double *rU, const Geo &g, int K, size_t NK, size_t q, const AxNode &n,
                                           double U[4])
{
    if (n.code < 0) {
#pragma unroll
        for (int v = 0; v < 4; v++) U[v] = n.u[v] / n.r;
        return;
    }
    const int d = n.code >> 1;
    const size_t eb = q - q % (size_t)K;
    const int j1 = g.axj[3 * d], j2 = g.axj[3 * d + 1], jn = g.axj[3 * d + 2];
    const double r1 = g.axr[3 * d], r2 = g.axr[3 * d + 1], rn = g.axr[3 * d + 2];
    double f1s[4], f2s[4], fns[4];   // (loaded together; no node: node 0, unused)
#pragma unroll
    for (int v = 0; v < 4; v++) {
        f1s[v] = rU[v * NK + eb + (j1 < 0 ? 0 : j1)];
        f2s[v] = rU[v * NK + eb + (j2 < 0 ? 0 : j2)];
        fns[v] = rU[v * NK + eb + jn];
    }
    auto fit = [&](int comp) -> double {
        if (j1 < 0) return 0.0;
        const double f1 = f1s[comp], f2 = f2s[comp];
        const double fref = fabs(f1);
        const double cap = (fref < 1e-12) ? INFINITY : 10.0 * fref / fmax(r1, 1e-14);
        if (j2 >= 0) {
            const double m = (r1 * f1 + r2 * f2) / fmax(r1 * r1 + r2 * r2, 1e-14);
            return ax_clamp(ax_minmod(m, ax_minmod(1.5 * (f1 / r1), 1.5 * (f2 / r2))), cap);
        }
        return ax_clamp(f1 / r1, cap);
    };
    const double rho = fit(0), mz = fit(1), E = fit(3);
    if (!isfinite(rho) || rho < g.axis_floor || !isfinite(E)) {
#pragma unroll
        for (int v = 0; v < 4; v++) U[v] = fns[v] / rn;
        U[2] = 0.0;
    } else {
        U[0] = rho;
        U[1] = mz;
        U[2] = 0.0;
        U[3] = E;
    }
}

// Adjugate rows (row r = Ja^r, the contravariant metric) and determinant of
// a hexahedron's trilinear map at reference point xi, from its corners c
// ([8][3], MFEM's vertex order): the metrics the host builds per node, here
// recomputed where they are used, which saves the 80 bytes per node of a
// stored table.
__device__ __forceinline__ void hex_metrics(const double *c, double x0, double x1, double x2, double *adj,
                                            double &det)
{
    constexpr int CV[8] = {0, 1, 3, 2, 4, 5, 7, 6};   // vertex k -> bits (x + 2y + 4z) of its corner
    double J[3][3];
#pragma unroll
    for (int a = 0; a < 3; a++)
#pragma unroll
        for (int b = 0; b < 3; b++) J[a][b] = 0.0;
    const double xi[3] = {x0, x1, x2};
#pragma unroll
    for (int k = 0; k < 8; k++) {
        double f[3], df[3];
#pragma unroll
        for (int d = 0; d < 3; d++) {
            const bool one = (CV[k] >> d) & 1;
            f[d] = one ? xi[d] : 1.0 - xi[d];
            df[d] = one ? 1.0 : -1.0;
        }
        const double dN[3] = {df[0] * f[1] * f[2], f[0] * df[1] * f[2], f[0] * f[1] * df[2]};
#pragma unroll
        for (int a = 0; a < 3; a++)
#pragma unroll
            for (int b = 0; b < 3; b++) J[a][b] += dN[b] * c[3 * k + a];
    }
    adj[0] = J[1][1] * J[2][2] - J[1][2] * J[2][1];
    adj[1] = J[0][2] * J[2][1] - J[0][1] * J[2][2];
    adj[2] = J[0][1] * J[1][2] - J[0][2] * J[1][1];
    adj[3] = J[1][2] * J[2][0] - J[1][0] * J[2][2];
    adj[4] = J[0][0] * J[2][2] - J[0][2] * J[2][0];
    adj[5] = J[0][2] * J[1][0] - J[0][0] * J[1][2];
    adj[6] = J[1][0] * J[2][1] - J[1][1] * J[2][0];
    adj[7] = J[0][1] * J[2][0] - J[0][0] * J[2][1];
    adj[8] = J[0][0] * J[1][1] - J[0][1] * J[1][0];
    det = J[0][0] * adj[0] + J[0][1] * adj[3] + J[0][2] * adj[6];
}

// Face point l (a + NP b, a and b the other two coordinates in increasing
// order) of a 3-D element's node on a face of direction r.
template <int NP> __device__ __forceinline__ int face_point_3(int node, int r)
{
    const int i = node % NP, j = (node / NP) % NP, k = node / (NP * NP);
    return r == 0 ? j + NP * k : (r == 1 ? i + NP * k : i + NP * j);
}

// ---------------------------------------------------------------------------
// k_visc: entropy variables, BR1 lifting, gradient conversion, viscous fluxes
// ---------------------------------------------------------------------------
// MIXED: the mixed-precision form.  Entropy variables stay FP64; each
// element's are shifted by their value at node 0 (in FP64) and the BR1
// derivatives, gradient conversion, viscous flux and D^ sums then run in
// FP32 on those offsets (D annihilates constants, so the shift leaves the
// derivatives unchanged while keeping their significant digits).  The
// outputs visc and fvf are FP32 in that form.
// OPEN: a box with boundary sides; their face points take the boundary
// type's lifting flux (LiftingBR1.cpp:311-407) instead of the neighbour jump.
// GEN: a quadrilateral or hexahedral mesh (per-node metrics, face tables; traces are
// Fv.n with the face's normal).
// RED (meshes in corrected mode, without gradient output): the velocity and
// temperature gradients alone (entgrad2velgrad), so the first entropy
// variable and its logarithms are left out except at boundary points: 16^3
// hexahedra N = 3 22.3 -> 18.5 us.
template <int DIM, int NP, bool MIXED, int FB, bool OPEN = false, bool GEN = false, bool RED = false>
__global__ void __launch_bounds__((VCfg<DIM, NP, FB>::BLOCK))
__attribute__((amdgpu_waves_per_eu(VCfg<DIM, NP, FB>::WAVES))) k_visc(const VArgs A)
{
    using C = VCfg<DIM, NP, FB>;
    constexpr int MC = DIM * DIM;   // adjugate entries per node (general geometry)
    using R = typename std::conditional<MIXED, float, double>::type;
    if (A.skip && *A.skip) return;   // uniform: before any barrier
    constexpr int NV = C::NV, K = C::K, NFP = C::NFP, EPB = C::EPB, BLOCK = C::BLOCK;
    constexpr int V0 = RED ? 1 : 0, NW = NV - V0;   // entropy variables from V0
    // phase 1 (lifting) needs the entropy variables and neighbour traces,
    // phase 2 (viscous divergence) the contravariant fluxes: one LDS region
    constexpr int P1 = EPB * NW * K + EPB * 2 * DIM * NW * NFP;
    constexpr int P2 = EPB * DIM * (NV - 1) * K;
    constexpr int SCR = P1 > P2 ? P1 : P2;

    __shared__ R sD[NP * NP];
    __shared__ R sDh[NP * NP];
    __shared__ double sUl[EPB][NV];   // state of node K-1 (the faithful stale state)
    __shared__ double sCn[GEN && DIM == 3 ? EPB : 1][GEN && DIM == 3 ? 24 : 1];   // hexahedron corners
    __shared__ double sWref[EPB][NV];
    __shared__ R sScr[SCR];
    R (*sW)[NW][K] = reinterpret_cast<R (*)[NW][K]>(sScr);
    R (*sWN)[2 * DIM][NW][NFP] = reinterpret_cast<R (*)[2 * DIM][NW][NFP]>(sScr + EPB * NW * K);
    R (*sFV)[DIM][NV - 1][K] = reinterpret_cast<R (*)[DIM][NV - 1][K]>(sScr);

    const int t = threadIdx.x;
    for (int i = t; i < NP * NP; i += BLOCK) {
        sD[i] = (R)A.tab.D[(i / NP) * MAXNP + i % NP];
        sDh[i] = (R)A.tab.Dh[(i / NP) * MAXNP + i % NP];
    }
    const Phys &P = A.phys;
    const int NE = A.geo.NE;
    const size_t NK = (size_t)NE * K;
    const int ebase = xcd_remap(blockIdx.x, gridDim.x) * EPB;
    const int el = t / K;
    const int n = t - el * K;
    const int e = ebase + el;
    const bool act = (el < EPB) && (e < NE);
    const int ii[3] = {n % NP, (n / NP) % NP, DIM == 3 ? n / (NP * NP) : 0};
    R *visc = reinterpret_cast<R *>(A.visc);
    R *fvf = reinterpret_cast<R *>(A.fvf);
    const R gm1 = (R)P.gm1, gm1i = (R)P.gm1i;
    const ViscCoef<R> vcoef{(R)P.mu, (R)P.lam_h, P.sutherland != 0, (R)P.R_gas, (R)P.gamma, (R)P.PrInv};

    // every global load of this thread in flight together: its own node and
    // the neighbour trace nodes of its face jobs
    constexpr int NJ = EPB * 2 * DIM * NFP;
    constexpr int JT = (NJ + BLOCK - 1) / BLOCK;
    double ys[NV], wv[NV];
    double tv[JT][NV];
    if (act)
#pragma unroll
        for (int v = 0; v < NV; v++) ys[v] = A.y[v * NK + (size_t)e * K + n];
    double jn = 1.0, mown[GEN ? MC : 1];
#pragma unroll
    for (int c = 0; c < (GEN ? MC : 1); c++) mown[c] = 0.0;
    if constexpr (GEN && DIM == 3) {
        for (int i = t; i < EPB * 24; i += BLOCK)
            sCn[i / 24][i % 24] = (ebase + i / 24 < NE) ? A.geo.corner[(size_t)(ebase + i / 24) * 24 + i % 24] : 0.0;
        __syncthreads();
        if (act) hex_metrics(sCn[el], A.tab.x[ii[0]], A.tab.x[ii[1]], A.tab.x[ii[2]], mown, jn);
    } else if constexpr (GEN) {
        if (act) {
            jn = A.geo.jac[(size_t)e * K + n];
#pragma unroll
            for (int c = 0; c < MC; c++) mown[c] = A.geo.met[c * NK + (size_t)e * K + n];
        }
    }
#pragma unroll
    for (int k = 0; k < JT; k++) {
        const int j = t + k * BLOCK;
        const int ej = j / (2 * DIM * NFP);
        const int eo = ebase + ej;
        if (j < NJ && eo < NE) {
            const int rem = j - ej * (2 * DIM * NFP);
            const int f = rem / NFP, q = rem - f * NFP;
            const int r = f >> 1, side = f & 1;
            int en = neighbor_lane(A.geo, eo, r, side);
            int nn = line_node<DIM, NP>(r, q, side ? 0 : NP - 1);
            if (OPEN && boundary_of(A.geo, eo, r, side) != BC_PERIODIC) {
                // boundary point: this element's own face node
                en = eo;
                nn = line_node<DIM, NP>(r, q, side ? NP - 1 : 0);
            }
            if constexpr (GEN) {
                const size_t efo = (size_t)eo * (2 * DIM) + f;
                if ((A.geo.fface[efo] >> 1) & 7) {
                    en = eo;
                    nn = line_node<DIM, NP>(r, q, side ? NP - 1 : 0);
                } else {
                    const int gn = A.geo.fnb[efo * NFP + q];
                    en = gn / K;
                    nn = gn - en * K;
                }
            }
#pragma unroll
            for (int v = 0; v < NV; v++) tv[k][v] = A.y[v * NK + (size_t)en * K + nn];
        }
    }
    if (act) {
        if (n == K - 1)
#pragma unroll
            for (int v = 0; v < NV; v++) sUl[el][v] = ys[v];
        cons2entropy<DIM, !RED>(ys, P, wv);
        if (MIXED && n == 0)
#pragma unroll
            for (int v = V0; v < NV; v++) sWref[el][v] = wv[v];
    }
    if (MIXED) __syncthreads();
    if (act)
#pragma unroll
        for (int v = V0; v < NV; v++) sW[el][v - V0][n] = MIXED ? (R)(wv[v] - sWref[el][v]) : (R)wv[v];
    // neighbour traces of the entropy variables
#pragma unroll
    for (int k = 0; k < JT; k++) {
        const int j = t + k * BLOCK;
        const int ej = j / (2 * DIM * NFP);
        const int eo = ebase + ej;
        if (j < NJ && eo < NE) {
            const int rem = j - ej * (2 * DIM * NFP);
            const int f = rem / NFP, q = rem - f * NFP;
            double w[NV];
            cons2entropy<DIM, !RED>(tv[k], P, w);
            const int code = GEN ? A.geo.fface[(size_t)eo * (2 * DIM) + f] : 0;
            const int bt = GEN ? ((code >> 1) & 7) : OPEN ? boundary_of(A.geo, eo, f >> 1, f & 1) : BC_PERIODIC;
            if ((OPEN || GEN) && bt != BC_PERIODIC) {
                // the lifting flux itself (not a trace) for the surface part
                double fb[NV];
                if constexpr (RED) cons2entropy<DIM>(tv[k], P, w);
                lift_flux<DIM>(bt, w, A.geo.bcs + (GEN ? (code >> 4) : f) * 5, P, A.quirks != 0, fb);
#pragma unroll
                for (int v = V0; v < NV; v++) sWN[ej][f][v - V0][q] = (R)fb[v];
            } else {
#pragma unroll
                for (int v = V0; v < NV; v++) sWN[ej][f][v - V0][q] = MIXED ? (R)(w[v] - sWref[ej][v]) : (R)w[v];
            }
        }
    }
    __syncthreads();
    // every start load has been used by now; saying so (free here, before
    // any store) keeps the compiler's count from treating a load left unused
    // on some lane's path as pending, which would make it wait for this
    // thread's face-trace stores to complete further down.  (gfx9's s_waitcnt
    // immediate: vmcnt 0, expcnt 7, lgkmcnt 15.)
    __builtin_amdgcn_s_waitcnt(0x0F70);

    R gp[DIM][NV];
    R yr[NV];
#pragma unroll
    for (int v = 0; v < NV; v++) yr[v] = act ? (R)ys[v] : R(1);
    if constexpr (GEN) if (act) {
        // grad w = (sum_r (D-sum along r) adj row r) / J, then the face terms
        // f n / (w0 J) with each face point's normal (LiftingBR1.cpp:10-272)
        const R invJ = (R)(1.0 / jn), aface = (R)(1.0 / (A.tab.w[0] * jn)), half = 0.5;
        R sd[DIM][NV];
#pragma unroll
        for (int c = 0; c < DIM; c++) {
            const int a = ii[c];
            const int l = line_of<DIM, NP>(c, ii[0], ii[1], ii[2]);
#pragma unroll
            for (int v = V0; v < NV; v++) {
                R s = 0;
#pragma unroll
                for (int m = 0; m < NP; m++)
                    s = (m == 0) ? sW[el][v - V0][line_node<DIM, NP>(c, l, m)] * sD[a * NP + m]
                                 : s + sW[el][v - V0][line_node<DIM, NP>(c, l, m)] * sD[a * NP + m];
                sd[c][v] = s;
            }
        }
#pragma unroll
        for (int cc = 0; cc < DIM; cc++)
#pragma unroll
            for (int v = V0; v < NV; v++)
            {
                R a = sd[0][v] * (R)mown[cc];
#pragma unroll
                for (int c = 1; c < DIM; c++) a = a + sd[c][v] * (R)mown[DIM * c + cc];
                gp[cc][v] = a * invJ;
            }
#pragma unroll
        for (int c = 0; c < DIM; c++) {
            const int a = ii[c];
            if (a == 0 || a == NP - 1) {
                const int side = (a == NP - 1), f = 2 * c + side;
                const int l = line_of<DIM, NP>(c, ii[0], ii[1], ii[2]);
                const size_t ef = (size_t)e * (2 * DIM) + f;
                const int code = A.geo.fface[ef];
                R nv2[DIM];
#pragma unroll
                for (int d = 0; d < DIM; d++) nv2[d] = (R)A.geo.fnor[(ef * NFP + l) * DIM + d];
                const bool bnd = ((code >> 1) & 7) != BC_PERIODIC;
                const bool own = code & 1;
#pragma unroll
                for (int v = V0; v < NV; v++) {
                    R fv;
                    if (bnd) fv = sWN[el][f][v - V0][l];
                    else {
                        const R wo = sW[el][v - V0][n], wn = sWN[el][f][v - V0][l];
                        fv = own ? half * (wn - wo) : half * (wo - wn);
                    }
#pragma unroll
                    for (int cc = 0; cc < DIM; cc++) gp[cc][v] += aface * (fv * nv2[cc]);
                }
            }
        }
#pragma unroll
        for (int c = 0; c < DIM; c++) {
            if constexpr (RED) entgrad2velgrad<DIM, R>(yr, gm1, gp[c]);
            else entgrad2primgrad<DIM, R>(yr, gm1, gm1i, A.quirks != 0, gp[c]);
        }
        if (!RED && A.grad)
#pragma unroll
            for (int c = 0; c < DIM; c++)
#pragma unroll
                for (int v = 0; v < NV; v++) A.grad[(c * NV + v) * NK + (size_t)e * K + n] = (double)gp[c][v];
    }
    if constexpr (!GEN) if (act) {
        const R nrm[3] = {(R)A.geo.nrm[0], (R)A.geo.nrm[1], (R)A.geo.nrm[2]};
        const R invJ = (R)A.geo.invJ, aface = (R)A.geo.aface, half = 0.5;
        // volume part: grad_r w = sum_l D_{i_r l} w_l, times adj / J
        // (LiftingBR1.cpp:176-215)
#pragma unroll
        for (int c = 0; c < DIM; c++) {
            const int a = ii[c];
            const int l = line_of<DIM, NP>(c, ii[0], ii[1], ii[2]);
#pragma unroll
            for (int v = 0; v < NV; v++) {
                R s = 0;
#pragma unroll
                for (int m = 0; m < NP; m++)
                    s = (m == 0) ? sW[el][v][line_node<DIM, NP>(c, l, m)] * sD[a * NP + m]
                                 : s + sW[el][v][line_node<DIM, NP>(c, l, m)] * sD[a * NP + m];
                gp[c][v] = (s * nrm[c]) * invJ;
            }
            // surface part: +1/2 (w2 - w1) n / (w0 J) on both sides (LiftingBR1.cpp:37-65)
            if (a == 0 || a == NP - 1) {
                const int side = (a == NP - 1);
                if (OPEN && boundary_of(A.geo, e, c, side) != BC_PERIODIC) {
                    // f n_c / (w0 J) with the outward normal (LiftingBR1.cpp:311-407)
                    const R nc = side ? nrm[c] : -nrm[c];
#pragma unroll
                    for (int v = 0; v < NV; v++) gp[c][v] += aface * (sWN[el][2 * c + side][v][l] * nc);
                } else {
#pragma unroll
                    for (int v = 0; v < NV; v++) {
                        const R wo = sW[el][v][n];
                        const R wn = sWN[el][2 * c + side][v][l];
                        const R f = side ? half * (wn - wo) : half * (wo - wn);
                        gp[c][v] += aface * (f * nrm[c]);
                    }
                }
            }
        }
#pragma unroll
        for (int c = 0; c < DIM; c++) entgrad2primgrad<DIM, R>(yr, gm1, gm1i, A.quirks != 0, gp[c]);
        if (A.grad)
#pragma unroll
            for (int c = 0; c < DIM; c++)
#pragma unroll
                for (int v = 0; v < NV; v++) A.grad[(c * NV + v) * NK + (size_t)e * K + n] = (double)gp[c][v];
    }
    __syncthreads();   // sW/sWN are dead from here; sFV reuses their storage

    // this element's half of its face traces, which belongs to the face terms
    // +-(1/w0) (Fv.n own + neighbour)/2 and goes into the volume sums (k_rhs_l
    // adds the neighbour's half; a boundary side's flux is k_rhs_l's alone)
    R own[NV - 1];
#pragma unroll
    for (int v = 0; v < NV - 1; v++) own[v] = 0;
    if (act) {
        R fl[DIM + 1][DIM];
        // volume viscous flux uses the stale node K-1 state (DGSEMIntegrator.cpp:620)
        R sv[NV];
#pragma unroll
        for (int v = 0; v < NV; v++) sv[v] = A.quirks ? (R)sUl[el][v] : yr[v];
        viscous_flux<DIM, R>(sv, gp, gm1, gm1i, vcoef, fl);
#pragma unroll
        for (int r = 0; r < DIM; r++)
#pragma unroll
            for (int v = 1; v < NV; v++) {
                if constexpr (GEN) {
                    // contravariant: adj row r times the physical flux
                    R a = (R)mown[DIM * r] * fl[v - 1][0];
#pragma unroll
                    for (int c = 1; c < DIM; c++) a += (R)mown[DIM * r + c] * fl[v - 1][c];
                    sFV[el][r][v - 1][n] = a;
                } else {
                    sFV[el][r][v - 1][n] = (R)A.geo.nrm[r] * fl[v - 1][r];
                }
            }
        bool onface = false;
#pragma unroll
        for (int c = 0; c < DIM; c++) onface |= (ii[c] == 0 || ii[c] == NP - 1);
        if (onface) {
            if (A.quirks) viscous_flux<DIM, R>(yr, gp, gm1, gm1i, vcoef, fl);
#pragma unroll
            for (int c = 0; c < DIM; c++) {
                if (ii[c] == 0 || ii[c] == NP - 1) {
                    const int side = (ii[c] == NP - 1);
                    const int l = line_of<DIM, NP>(c, ii[0], ii[1], ii[2]);
                    R *dst = fvf + (((size_t)e * 2 * DIM + 2 * c + side) * (NV - 1)) * NFP;
                    if constexpr (GEN) {
                        // Fv.n with the face's normal (outward of its first element)
                        const size_t ef = (size_t)e * (2 * DIM) + 2 * c + side;
                        R nf[DIM];
#pragma unroll
                        for (int d = 0; d < DIM; d++) nf[d] = (R)A.geo.fnor[(ef * NFP + l) * DIM + d];
#pragma unroll
                        for (int v = 1; v < NV; v++) {
                            R a = fl[v - 1][0] * nf[0];
#pragma unroll
                            for (int d = 1; d < DIM; d++) a = a + fl[v - 1][d] * nf[d];
                            dst[(v - 1) * NFP + l] = a;
                            const int code = A.geo.fface[ef];
                            const R h = ((code >> 1) & 7) != BC_PERIODIC ? R(0) : (R)(0.5 / A.tab.w[0]);
                            own[v - 1] += ((code & 1) ? h : -h) * a;
                        }
                    } else {
                        R h = (R)(0.5 / A.tab.w[0]) * (R)A.geo.nrm[c];
                        if (OPEN && boundary_of(A.geo, e, c, side) != BC_PERIODIC) h = 0;
#pragma unroll
                        for (int v = 1; v < NV; v++) {
                            dst[(v - 1) * NFP + l] = fl[v - 1][c];
                            own[v - 1] += (side ? h : -h) * fl[v - 1][c];
                        }
                    }
                }
            }
        }
    }
    __syncthreads();
    if (act) {
        // sum_r sum_l Dhat_{i_r l} (adj Fv)^r_l  (DGSEMIntegrator.cpp:705-738)
        R acc[NV - 1];
#pragma unroll
        for (int v = 0; v < NV - 1; v++) acc[v] = 0;
#pragma unroll
        for (int r = 0; r < DIM; r++) {
            const int a = ii[r];
            const int l = line_of<DIM, NP>(r, ii[0], ii[1], ii[2]);
#pragma unroll
            for (int m = 0; m < NP; m++) {
                const int nm = line_node<DIM, NP>(r, l, m);
                const R dm = sDh[a * NP + m];
#pragma unroll
                for (int v = 0; v < NV - 1; v++) acc[v] += sFV[el][r][v][nm] * dm;
            }
        }
#pragma unroll
        for (int v = 0; v < NV - 1; v++) visc[v * NK + (size_t)e * K + n] = acc[v] + own[v];
    }
}

// State of a time loop run on the device (Simulation::Run's stepping,
// Simulation.cpp:893-907, 1007-1022): time, step size, the clipped step of
// the current step, done flag and step count.
struct LoopState {
    double t, dt, dt_real;
    int done, steps, bad;
};

} // namespace prandtl
