// k_rhs_l: the flux-differencing RHS of two- and three-dimensional meshes with
// one thread per tensor line (gfx950): Cartesian boxes, periodic or with
// boundary sides, quadrilateral and hexahedral meshes, axisymmetric meshes,
// and the tiles of the batched ensemble.  Restates DGSEMIntegrator.cpp:151-433,
// 435-549, 601-864, 972-1196, BdrFaceIntegrator.cpp:61-175, PerssonPeraire-
// Indicator.cpp:21-58, DGSEMOperator.cpp:60-80 and MFEM's RK3SSPSolver stage
// arithmetic.
//
//  - node phase: the workgroup's EPB elements are loaded (coalesced, one node
//    per thread and pass), and each node's rho, v, beta = rho/(2p) and wave
//    speed go to LDS;
//  - line phase: thread (element, direction r, line l) evaluates the two
//    surface points at its line's ends (both neighbouring elements compute a
//    face point, with the same operands, so no scatter is needed), its NP(NP-1)/2
//    symmetric volume pairs and, in blended elements, its NP-1 subcell
//    interfaces, and sums each node's terms in registers;
//  - the DIM partial sums of a node are added in LDS in direction order (DIM
//    barrier-separated passes, no atomics), then the assembly adds the viscous
//    volume term, scales by 1/J and does the RK stage combination, reading the
//    state again (from the cache).
//
// What shapes it:
//  - No flux goes through LDS.  Taking the pairs as jobs of a workgroup's
//    threads costs 5 writes and 10 reads of LDS per pair in 3-D and leaves
//    the sums to a part of the threads.
//  - The pairs of a line are straight-line code.  A line's smallest and
//    largest rho and beta bound the ratio of every pair, so the range of the log
//    means (log_means) is chosen once per line, with an unrolled loop per
//    range.  The choice depends on the line's own values, or between ranges
//    that agree bitwise, so results do not depend on the lanes that share a
//    wave, nor on the workgroup's size.
//  - Sums are kept in units of 1/J: a node's total is (visc - acc) / J, acc =
//    (1 - alpha) vol - alpha fv - surface / w0.  (1 - alpha) is put into the
//    metric vector, in which the fluxes are linear, so the sums start with
//    the surface terms and need no second set of registers.
//  - A mesh line's metric vectors are a polynomial of its coordinate (straight-
//    sided elements), formed from the element's corners: no metric is loaded.
//  - The indicator's transforms run on the line threads: NP values in
//    registers, NP^2 multiply-adds.
//
// Bound: at 3-D N = 3, 45 x 43 x 41 elements with Navier-Stokes terms, HBM: 0.96
// GB, 0.21 ms at the 4.55 TB/s of a large copy, in 0.22 ms.  At 3-D N = 7, 32^3
// elements, blended Navier-Stokes, FP64 issue and HBM together: 3,025 vector
// instructions per wave, 0.53 ms of issue, and 2.6 GB, 0.58 ms at the copy rate, in
// 0.99 ms at three waves per SIMD, which hide neither completely (two: 1.16 times
// slower).  Against the kernel that took pairs as jobs, per right-hand side:
// that case 3,475 -> 1,617 us (k_visc's 660 included); 2-D N = 3, 384^2
// blended 172 -> 70; Euler 16^3 N = 7 279 -> 95, 28^3 N = 4 207 -> 125, 9x8x7
// N = 6 39.8 -> 18.2; slip walls 40^3 N = 2 159 -> 97, 32x31x30 N = 3 133 ->
// 97; 13,600 blended quadrilaterals N = 3 28.4 -> 17; 16^3 hexahedra N = 3
// Navier-Stokes 52.5 -> 41; a 64-case ensemble, two steps, 969 -> 368.
#pragma once
#include "dg_device.h"

namespace prandtl {

// Elements per workgroup of the natural shape.  One or two dimensions: as many
// as a single wave holds (its barriers cost nothing, and small meshes spread
// over more CUs); 3-D: the best thread utilisation within 256 threads.
constexpr int lines_epb(int DIM, int TE)
{
    if (DIM < 3) return 64 / TE;
    int best = 1;
    double bu = 0.0;
    for (int e = 1; r64(e * TE) <= 256; e++) {
        const double u = (double)(e * TE) / r64(e * TE);
        if (u >= bu) { bu = u; best = e; }
    }
    return best;
}

// LDS slot of node (i, j, k) in a row.  The LDS serves a wave's 8-byte
// accesses 32 lanes at a time from 64 four-byte banks, so 32 lanes reading
// distinct doubles run in one pass when their slots are distinct mod 32.
//  - 3-D NP = 4: 16k + 4((j+k) mod 4) + ((i+k) mod 4).  In the planes i = m,
//    j = m and k = m (node m of every line of a direction) the slots are
//    distinct mod 16; elements lie 16 (mod 32) doubles apart and a half-wave
//    holds one direction's lines of two elements.
//  - 3-D NP = 8: 64k + 8((j+k) mod 8) + ((i+j+2k) mod 8); a half-wave holds 32
//    lines of one direction, distinct mod 32 in each plane.
//  Node-order accesses (32 consecutive nodes) are distinct mod 32 in both.
//  - others: node order, with one double of padding per x-row where NP = 6.
//    Their lines do not align with half-waves; counted over all line and
//    node accesses, two lanes share a bank (1.6 to 2.0 passes).
template <int DIM, int NP> __host__ __device__ constexpr int lines_slot(int i, int j, int k)
{
    if (DIM == 3 && NP == 4) return 16 * k + 4 * ((j + k) & 3) + ((i + k) & 3);
    if (DIM == 3 && NP == 8) return 64 * k + 8 * ((j + k) & 7) + ((i + j + 2 * k) & 7);
    const int n = (k * NP + j) * NP + i;
    return NP == 6 ? n + n / NP : n;
}
template <int DIM, int NP> __device__ __forceinline__ int lines_node_slot(int n)
{
    if (DIM == 1) return n;
    if (DIM == 2) return lines_slot<DIM, NP>(n % NP, n / NP, 0);
    return lines_slot<DIM, NP>(n % NP, (n / NP) % NP, n / (NP * NP));
}

template <int DIM, int NP, int FB = 0> struct LnCfg {
    static constexpr int NV = DIM + 2;
    static constexpr int K = npow(NP, DIM);
    static constexpr int NFP = npow(NP, DIM - 1);
    static constexpr int TE = DIM * NFP;
    static constexpr int EPB = FB ? FB / TE : lines_epb(DIM, TE);
    static constexpr int BLOCK = FB ? FB : r64(EPB * TE);
    static constexpr int NPASS = (EPB * K + BLOCK - 1) / BLOCK;
    // half-waves of one direction and two elements (lines_slot)
    static constexpr bool HALF = DIM == 3 && NP == 4 && EPB % 2 == 0 && BLOCK == EPB * TE;
    static constexpr int NPAIR = NP * (NP - 1) / 2;
    static constexpr int NR = NV + 1;   // rows of an element: rho, v, beta, lambda
    static constexpr int KP = NP == 6 ? K + K / NP : K;
    static constexpr int ES = NR * KP + (DIM == 3 && NP == 4 ? (NR * KP % 32 == 0 ? 16 : 0) : 0);
    static_assert(EPB >= 1, "a workgroup holds an element's lines");
    static constexpr int WAVES = 3;
};

// Whether the pair and Vandermonde tables are read from LDS (broadcasts)
// instead of scalar registers.  Where they exceed the scalar registers each
// use costs a v_readlane: 3-D N = 7 974 of 3,989 vector instructions per
// wave (1,720 -> 1,607 us per right-hand side at 32^3); blended 3-D N = 4
// 26.9 -> 22.8 us at 12^3, N = 3 102 -> 99 at 32x31x30.  Where they fit, the
// LDS reads cost more (2-D N = 3 slip-wall and mesh kernels 3-4% slower).
constexpr bool lines_ltab(int DIM, int NP, bool BLEND) { return NP >= 6 || (DIM == 3 && NP >= 4 && BLEND); }

// Which line a thread holds: element el of the workgroup, direction r, line l
// with the other indices la, lb (increasing direction), rem = r NFP + l; base
// and stride give its nodes' numbers, slots() their LDS slots.  NP = 8: a wave
// is one direction, so r is scalar.
template <int DIM, int NP, int FB> struct LinePos {
    using C = LnCfg<DIM, NP, FB>;
    int el, r, l, rem, la, lb, base, stride;
    __device__ __forceinline__ explicit LinePos(int t)
    {
        constexpr int NFP = C::NFP, TE = C::TE;
        if constexpr (C::HALF) {
            const int h = t >> 5;
            r = h % 3;
            el = 2 * (h / 3) + ((t >> 4) & 1);
            l = t & 15;
            rem = r * NFP + l;
        } else {
            el = C::EPB == 1 ? 0 : t / TE;
            rem = t - el * TE;
            r = rem / NFP;
            if constexpr (NFP == 64 && C::EPB == 1) r = __builtin_amdgcn_readfirstlane(r);
            l = rem - r * NFP;
        }
        la = DIM == 3 ? l % NP : l;
        lb = DIM == 3 ? l / NP : 0;
        base = r == 0 ? l * NP : (DIM == 3 && r == 1 ? lb * NP * NP + la : l);
        stride = r == 0 ? 1 : (r == 1 ? NP : NP * NP);
    }
    __device__ __forceinline__ void slots(int *ls) const
    {
#pragma unroll
        for (int m = 0; m < NP; m++) {
            if constexpr (DIM == 2) ls[m] = r == 0 ? lines_slot<DIM, NP>(m, la, 0) : lines_slot<DIM, NP>(la, m, 0);
            else ls[m] = lines_slot<DIM, NP>(r == 0 ? m : la, r == 1 ? m : (r == 0 ? la : lb), r == 2 ? m : lb);
        }
    }
};

// LDS of one tile (EPB elements).
template <int DIM, int NP, bool BLEND, int FB, bool GEN, bool AXI> struct LineSmem {
    using C = LnCfg<DIM, NP, FB>;
    static constexpr bool LTAB = lines_ltab(DIM, NP, BLEND);
    double Q[C::EPB * C::ES];                                   // rows; then the partial sums
    double X[BLEND ? C::EPB : 1][BLEND ? C::KP : 1];            // indicator: rho p and its transforms
    double E[BLEND ? C::EPB : 1][3][BLEND ? C::NFP : 1];        // modal energies per line
    double Al[C::EPB];
    double Red[(C::BLOCK + 63) / 64];
    double Cn[GEN ? C::EPB : 1][GEN ? (DIM == 3 ? 24 : 8) : 1];   // element corners
    double R[AXI ? C::EPB : 1][AXI ? C::KP : 1];                // r of the nodes
    double Pr[AXI ? C::EPB : 1][AXI ? C::KP : 1];               // p of the nodes
    double Xn[GEN ? NP : 1];                                    // LGL nodes
    double D2[LTAB ? C::NPAIR : 1][2];                       // 2 D_ab, 2 D_ba of each pair
    double V1[LTAB && BLEND ? NP * NP : 1];                  // inverse 1-D Vandermonde
};

// What a two-point flux with dissipation needs of a node beyond (rho, v,
// beta), formed from these alone.
template <int DIM> __device__ __forceinline__ void face_quants(NodeQ<DIM> &q, const Phys &P)
{
    double vsq = 0.0;
#pragma unroll
    for (int d = 0; d < DIM; d++) vsq = (d == 0) ? q.v[d] * q.v[d] : fma(q.v[d], q.v[d], vsq);
    q.ibeta = rcp_nr(q.beta);
    q.lam = sqrt(vsq) + sqrt(0.5 * P.gamma * q.ibeta);
}

// ComputeViscousFlux left velocities in the momentum slots of a face point's
// state (DGSEMIntegrator.cpp:471-481): the quantities of that state.
template <int DIM> __device__ __forceinline__ void alias_quants(NodeQ<DIM> &q, const Phys &P)
{
    const double ri = rcp_nr(q.rho);
    double p = 0.5 * q.rho * rcp_nr(q.beta), v0 = 0.0, v1 = 0.0;
#pragma unroll
    for (int d = 0; d < DIM; d++) {
        v0 = (d == 0) ? q.v[d] * q.v[d] : v0 + q.v[d] * q.v[d];
        q.v[d] *= ri;
        v1 = (d == 0) ? q.v[d] * q.v[d] : v1 + q.v[d] * q.v[d];
    }
    p += P.gm1 * (0.5 * q.rho) * (v0 - v1);
    q.beta = 0.5 * q.rho * rcp_nr(p);
    face_quants<DIM>(q, P);
}

// Metric vector (adjugate row rr) along a line of direction rr of a straight-
// sided element: a polynomial of the line's coordinate xi with coefficients
// m[0] + xi m[1] + xi^2 m[2] (quadrilaterals: linear).  c: the element's
// corners in vertex order; ca, cb: the line's other two coordinates, in
// increasing order of direction.
template <int DIM>
__device__ __forceinline__ void line_metric(const double *c, int rr, double ca, double cb, double (*m)[DIM])
{
    if constexpr (DIM == 2) {
        // the derivative along the other direction, at the line's two ends
        const int i0 = rr == 0 ? 3 : 1, i1 = 2, j1 = rr == 0 ? 1 : 3;
        const double ax = c[2 * i0] - c[0], ay = c[2 * i0 + 1] - c[1];
        const double bx = c[2 * i1] - c[2 * j1] - ax, by = c[2 * i1 + 1] - c[2 * j1 + 1] - ay;
        const double s = rr == 0 ? 1.0 : -1.0;
        m[0][0] = s * ay; m[0][1] = -s * ax;
        m[1][0] = s * by; m[1][1] = -s * bx;
    } else {
        // x_s (linear in xi at coordinate t) cross x_t (at coordinate s), with
        // (s, t) the two directions after rr in cyclic order
        const int s = rr == 2 ? 0 : rr + 1, t = rr == 0 ? 2 : rr - 1;
        const double cs = rr == 1 ? cb : ca, ct = rr == 1 ? ca : cb;
        auto corner = [&](int br, int bs, int bt) {
            int b[3];
#pragma unroll
            for (int d = 0; d < 3; d++) b[d] = d == rr ? br : d == s ? bs : bt;
            return c + 3 * (4 * b[2] + (b[1] ? 3 - b[0] : b[0]));
        };
        (void)t;
        double A[2][3], B[2][3];
#pragma unroll
        for (int br = 0; br < 2; br++) {
            const double *p00 = corner(br, 0, 0), *p10 = corner(br, 1, 0), *p01 = corner(br, 0, 1), *p11 = corner(br, 1, 1);
#pragma unroll
            for (int d = 0; d < 3; d++) {
                A[br][d] = (1.0 - ct) * (p10[d] - p00[d]) + ct * (p11[d] - p01[d]);
                B[br][d] = (1.0 - cs) * (p01[d] - p00[d]) + cs * (p11[d] - p10[d]);
            }
        }
#pragma unroll
        for (int d = 0; d < 3; d++) { A[1][d] -= A[0][d]; B[1][d] -= B[0][d]; }
#pragma unroll
        for (int d = 0; d < 3; d++) {
            const int u = (d + 1) % 3, v = (d + 2) % 3;
            m[0][d] = A[0][u] * B[0][v] - A[0][v] * B[0][u];
            m[1][d] = (A[0][u] * B[1][v] - A[0][v] * B[1][u]) + (A[1][u] * B[0][v] - A[1][v] * B[0][u]);
            m[2][d] = A[1][u] * B[1][v] - A[1][v] * B[1][u];
        }
    }
}

// One tile: elements [tile*EPB, tile*EPB + EPB) of the case A describes; slot
// indexes the tile's running wave-speed maximum.
// BLEND: modal indicator + subcell FV blending.  QNS3: the reference's NS-3D
// zeta-partner defect (faithful NS in 3-D).  VT: element type of k_visc's
// outputs (float in the mixed form).  FB: forced workgroup size.  OPEN:
// boundary sides on a Cartesian box.  GEN: quadrilateral or hexahedral mesh.
// AXI (with GEN, Euler): axisymmetric, A.y the weighted state r U.
// tid: the thread's index as the caller sees it (a loop over tiles passes one
// the compiler cannot hoist out of the loop).
template <int DIM, int NP, bool BLEND, bool QNS3, typename VT, int FB, bool OPEN = false, bool GEN = false,
          bool AXI = false>
__device__ __forceinline__ void line_body(const KArgs &A, const int tile, const int slot,
                                          LineSmem<DIM, NP, BLEND, FB, GEN, AXI> &S, const int tid = -1)
{
    using C = LnCfg<DIM, NP, FB>;
    constexpr int NV = C::NV, K = C::K, NFP = C::NFP, TE = C::TE, EPB = C::EPB, BLOCK = C::BLOCK, NPASS = C::NPASS;
    constexpr int KP = C::KP, ES = C::ES;
    constexpr bool LTAB = lines_ltab(DIM, NP, BLEND);
    static_assert(DIM > 1, "1-D right-hand sides run node threads");
    static_assert(!AXI || (GEN && DIM == 2), "axisymmetric meshes are quadrilateral meshes");
    auto sQ = [&](int e2, int row, int s) -> double & { return S.Q[e2 * ES + row * KP + s]; };

    if (A.skip && *A.skip) return;   // uniform: before any barrier
    const int t = tid < 0 ? (int)threadIdx.x : tid;
    const int ebase = tile * EPB;
    const int NE = A.geo.NE;
    const size_t NK = (size_t)NE * K;
    const Phys &P = A.phys;
    const bool quirk3d = A.quirks != 0;
    const double lam_old = (t == 0) ? A.lam[slot] : 0.0;

    const LinePos<DIM, NP, FB> L(t);
    const int el = L.el, r = L.r, l = L.l, rem = L.rem, la = L.la, lb = L.lb, base = L.base, stride = L.stride;
    const int e = ebase + el;
    const bool lact = (el < EPB) && (rem < TE) && (e < NE);
    int ls[NP];
    L.slots(ls);

    // ---- start loads: the nodes first, then the traces at the line's ends.
    // Loads complete in issue order, so the node phase waits for its own
    // loads while the traces are in flight; every load is on every path (one
    // skipped on some path would make that wait a wait for everything):
    // lanes without an element load from index 0 and discard the value.
    const int nact = (NE - ebase) < EPB ? (NE - ebase) * K : EPB * K;
    int gn[2] = {0, 0}, code[2] = {0, 0};   // GEN: end points' neighbour nodes and face codes
    if constexpr (GEN) {
#pragma unroll
        for (int side = 0; side < 2; side++) {
            const size_t ef = lact ? (size_t)e * (2 * DIM) + 2 * r + side : 0;
            code[side] = A.geo.fface[ef];
            gn[side] = A.geo.fnb[ef * NFP + (lact ? l : 0)];
        }
    }
    double ysp[NPASS][NV];
    AxNode xn[AXI ? NPASS : 1], xt[AXI ? 2 : 1];
    size_t gt[2] = {0, 0};
#pragma unroll
    for (int p = 0; p < NPASS; p++) {
        const int i = t + p * BLOCK;
        const size_t gi = (i < nact) ? (size_t)ebase * K + i : 0;
        if constexpr (AXI) {
            xn[p] = axis_load(A.y, A.geo, NK, gi);
        } else {
#pragma unroll
            for (int v = 0; v < NV; v++) {
                const double y = A.y[v * NK + gi];
                ysp[p][v] = (i < nact) ? y : 1.0;
            }
        }
    }
    double pt[2][NV];       // neighbour states; on a boundary side this element's own face node
    int bt[2] = {BC_PERIODIC, BC_PERIODIC};
    double nv[GEN ? 2 : 1][DIM];   // GEN: the end points' normals, outward of the face's first element
    VT ftn[2][NV - 1];
#pragma unroll
    for (int side = 0; side < 2; side++) {
        size_t g = 0;
        int en = 0;
        if constexpr (GEN) {
            bt[side] = lact ? (code[side] >> 1) & 7 : BC_PERIODIC;
            if (lact) g = bt[side] != BC_PERIODIC ? (size_t)e * K + base + (side ? (NP - 1) * stride : 0) : (size_t)gn[side];
            const size_t ef = lact ? (size_t)e * (2 * DIM) + 2 * r + side : 0;
#pragma unroll
            for (int d = 0; d < DIM; d++) nv[side][d] = A.geo.fnor[(ef * NFP + (lact ? l : 0)) * DIM + d];
        } else {
            en = lact ? neighbor_lane(A.geo, e, r, side) : 0;
            int nn = base + (side ? 0 : (NP - 1) * stride);
            if (OPEN && lact) {
                bt[side] = boundary_of(A.geo, e, r, side);
                if (bt[side] != BC_PERIODIC) { en = e; nn = base + (side ? (NP - 1) * stride : 0); }
            }
            g = lact ? (size_t)en * K + nn : 0;
        }
        if constexpr (AXI) {
            xt[side] = axis_load(A.y, A.geo, NK, g);
            gt[side] = g;
        } else {
#pragma unroll
            for (int v = 0; v < NV; v++) {
                const double y = A.y[v * NK + g];
                pt[side][v] = lact ? y : 1.0;
            }
        }
        if constexpr (!AXI) {
            // the neighbour's viscous face trace (this element's own is in
            // k_visc's volume term); without viscous terms it is read from
            // the state array and discarded.  On a boundary side: this
            // element's own trace
            const bool vact = A.parabolic && lact;
            const VT *fv = A.parabolic ? static_cast<const VT *>(A.fvf) : reinterpret_cast<const VT *>(A.y);
            size_t on = 0;
            if (vact) {
                const size_t ef = (size_t)e * 2 * DIM + 2 * r + side;
                if constexpr (GEN) {
                    if (bt[side] == BC_PERIODIC) {
                        const int nf = A.geo.fnf[ef];
                        const size_t fid = (size_t)(nf >> 1);
                        int l2;
                        if constexpr (DIM == 2) l2 = (nf & 1) ? NP - 1 - l : l;
                        else l2 = face_point_3<NP>(gn[side] - (int)(fid / 6) * K, (int)(fid % 6) >> 1);
                        on = fid * (NV - 1) * NFP + l2;
                    } else {
                        on = ef * (NV - 1) * NFP + l;
                    }
                } else {
                    const bool bnd = OPEN && bt[side] != BC_PERIODIC;
                    on = (bnd ? ef : (size_t)en * 2 * DIM + 2 * r + 1 - side) * (NV - 1) * NFP + l;
                }
            }
#pragma unroll
            for (int v = 0; v < NV - 1; v++) {
                const VT b = fv[on + v * NFP];
                ftn[side][v] = vact ? b : VT(0);
            }
        }
    }
    if constexpr (LTAB) {
        static_assert(NP * NP <= BLOCK, "one table entry per thread");
        if (t < NP * NP) {
            const int a = t / NP, b = t - a * NP;
            const double d = A.tab.Dh2[a * MAXNP + b];
            const double w = BLEND ? A.tab.V1i[a * MAXNP + b] : 0.0;
            if (a < b) S.D2[pair_index<NP>(a, b)][0] = d;
            if (b < a) S.D2[pair_index<NP>(b, a)][1] = d;
            if (BLEND) S.V1[t] = w;
        }
    }
    auto dpair = [&](int a, int b, int k) {
        if constexpr (LTAB) return S.D2[pair_index<NP>(a, b)][k];
        else return k ? A.tab.Dh2[b * MAXNP + a] : A.tab.Dh2[a * MAXNP + b];
    };
    auto v1i = [&](int a, int m) {
        if constexpr (LTAB) return S.V1[a * NP + m];
        else return A.tab.V1i[a * MAXNP + m];
    };
    if constexpr (GEN) {
        constexpr int NC = DIM == 3 ? 24 : 8;
        for (int i = t; i < EPB * NC; i += BLOCK)
            S.Cn[i / NC][i % NC] = (ebase + i / NC < NE) ? A.geo.corner[(size_t)ebase * NC + i] : 0.0;
        if (t < NP) S.Xn[t] = A.tab.x[t];
    }

    // ---- node phase ----
    double lam = 0.0;
#pragma unroll
    for (int p = 0; p < NPASS; p++) {
        const int i = t + p * BLOCK;
        if (i >= nact) continue;
        const int e2 = EPB == 1 ? 0 : i / K, n = i - e2 * K;
        const int s = lines_node_slot<DIM, NP>(n);
        if constexpr (AXI) axis_state(A.y, A.geo, K, NK, (size_t)ebase * K + i, xn[p], ysp[p]);
        const NodeQ<DIM> q = node_quants<DIM>(ysp[p], P);
        sQ(e2, 0, s) = q.rho;
#pragma unroll
        for (int d = 0; d < DIM; d++) sQ(e2, 1 + d, s) = q.v[d];
        sQ(e2, NV - 1, s) = q.beta;
        sQ(e2, NV, s) = q.lam;
        if constexpr (BLEND) {
            double vsq = 0.0;
#pragma unroll
            for (int d = 0; d < DIM; d++) vsq = (d == 0) ? q.v[d] * q.v[d] : vsq + q.v[d] * q.v[d];
            S.X[e2][s] = q.rho * (P.gm1 * (ysp[p][NV - 1] - 0.5 * q.rho * vsq));   // rho p
        }
        if constexpr (AXI) {
            // PressureFromConservative (DGSEMIntegrator.cpp:1306-1315)
            const double ke = 0.5 * ((ysp[p][1] * ysp[p][1] + ysp[p][2] * ysp[p][2]) / ysp[p][0]);
            S.Pr[e2][s] = P.gm1 * (ysp[p][3] - ke);
            S.R[e2][s] = A.geo.rnode[(size_t)ebase * K + i];
        }
        const double lq = (q.lam == q.lam) ? q.lam : 0.0;
        lam = (lam < lq) ? lq : lam;
    }
    __syncthreads();
    auto node = [&](int m) {
        NodeQ<DIM> q;
        q.rho = sQ(el, 0, ls[m]);
#pragma unroll
        for (int d = 0; d < DIM; d++) q.v[d] = sQ(el, 1 + d, ls[m]);
        q.beta = sQ(el, NV - 1, ls[m]);
        return q;
    };
    auto face_node = [&](int m) {
        NodeQ<DIM> q = node(m);
        q.lam = sQ(el, NV, ls[m]);
        q.ibeta = rcp_nr(q.beta);
        return q;
    };

    // the line's metric vector on a box
    const double nr = GEN ? 0.0 : lane_pick3(A.geo.nrm[0], A.geo.nrm[1], A.geo.nrm[2], r);
    double nvec[DIM];
#pragma unroll
    for (int d = 0; d < DIM; d++) nvec[d] = (d == r) ? nr : 0.0;

    // ---- surface points of the line's ends: the first terms of the end
    // nodes' sums.  A point's flux is toward +e_r (boxes) or out of the face's
    // first element, the same on both its sides: (rho, v, beta, lambda) of
    // either node come from the same formulas on both
    double acc[NP][NV];
#pragma unroll
    for (int a = 0; a < NP; a++)
#pragma unroll
        for (int v = 0; v < NV; v++) acc[a][v] = 0.0;
    if (lact) {
        const double iw0 = 1.0 / A.tab.w[0];
#pragma unroll
        for (int side = 0; side < 2; side++) {
            double *pn = pt[side];
            const int mo = side ? NP - 1 : 0;
            if constexpr (AXI) axis_state(A.y, A.geo, K, NK, gt[side], xt[side], pn);
            double F[NV];
            if ((OPEN || GEN) && bt[side] != BC_PERIODIC) {
                // boundary point: F_b for the outward normal at the interior
                // node (BdrFaceIntegrator.cpp:61-123, DGSEMNonlinearForm.cpp:
                // 776-826); its wave speed joins the running maximum
                // (DGSEMOperator.cpp:585-589)
                double bs[5], nn[DIM], lb;
                if constexpr (GEN) {
                    const int at = code[side] >> 4;
#pragma unroll
                    for (int v = 0; v < 5; v++) bs[v] = A.geo.bcs[at * 5 + v];
                    if (A.geo.bfn && A.geo.bfn[at * 16] != 0.0) {
                        // the attribute's time-dependent outer state at this
                        // point: "below" where n . x - offset - speed t < 0
                        // (SpecifiedStateBdrFaceIntegrator.cpp:24-34), evaluated
                        // left to right without contraction
                        const double *fn = A.geo.bfn + at * 16;
                        const double *xp = A.geo.fxy + (((size_t)e * (2 * DIM) + 2 * r + side) * NFP + l) * 2;
                        const double tt = (A.tp ? *A.tp : 0.0) + A.tc * step_dt(A);
                        double sd = __dmul_rn(fn[1], xp[0]);
                        sd = __dadd_rn(sd, __dmul_rn(fn[2], xp[1]));
                        sd = __dadd_rn(sd, __dmul_rn(fn[3], 0.0));
                        sd = __dsub_rn(sd, fn[4]);
                        sd = __dsub_rn(sd, __dmul_rn(fn[5], tt));
#pragma unroll
                        for (int v = 0; v < 5; v++) bs[v] = (sd < 0.0) ? fn[6 + v] : fn[11 + v];
                    }
#pragma unroll
                    for (int d = 0; d < DIM; d++) nn[d] = nv[side][d];
                    lb = boundary_flux_vn<DIM>(bt[side], nn, pn, bs, P, quirk3d, F);
                } else {
#pragma unroll
                    for (int v = 0; v < 5; v++) bs[v] = A.geo.bcs[(2 * r + side) * 5 + v];
#pragma unroll
                    for (int d = 0; d < DIM; d++) nn[d] = side ? nvec[d] : -nvec[d];
                    lb = boundary_flux<DIM>(bt[side], r, side ? nr : -nr, nr, pn, bs, P, quirk3d, F);
                }
                lam = (lam < lb) ? lb : lam;
                if constexpr (AXI) {
                    // dU_face1 *= r (BdrFaceIntegrator.cpp:109-111)
                    const double rf = S.R[el][ls[mo]];
#pragma unroll
                    for (int v = 0; v < NV; v++) F[v] *= rf;
                }
                if constexpr (!AXI) {
                    if (A.parabolic && (bt[side] == BC_OUTFLOW || bt[side] == BC_NOSLIP)) {
                        // - Fv.n of the interior state and gradients; inflow
                        // and specified states have zero gradients, so no
                        // viscous flux (BdrFaceIntegrator.cpp:141-175); the
                        // no-slip wall's energy term is V.(Fv.n)_mom + qn |n|
                        double fn[NV], n2 = nn[0] * nn[0];
#pragma unroll
                        for (int d = 1; d < DIM; d++) n2 = n2 + nn[d] * nn[d];
#pragma unroll
                        for (int v = 1; v < NV; v++) fn[v] = GEN ? (double)ftn[side][v - 1] : (double)ftn[side][v - 1] * (side ? nr : -nr);
                        if (bt[side] == BC_NOSLIP) {
                            double en = bs[0] * fn[1];
#pragma unroll
                            for (int d = 1; d < DIM; d++) en = en + bs[d] * fn[1 + d];
                            fn[NV - 1] = en + bs[3] * sqrt(n2);
                        }
#pragma unroll
                        for (int v = 1; v < NV; v++) F[v] -= fn[v];
                    }
                }
#pragma unroll
                for (int v = 0; v < NV; v++) acc[mo][v] = iw0 * F[v];
                continue;
            }
            NodeQ<DIM> qo = face_node(mo), qn = node_quants<DIM>(pn, P);
            qn.ibeta = rcp_nr(qn.beta);
            if constexpr (!AXI) {
                if (A.parabolic && A.quirks) {
                    alias_quants<DIM>(qo, P);
                    alias_quants<DIM>(qn, P);
                }
            }
            // the face's first side: the low element on a box
            const bool own = GEN ? (code[side] & 1) != 0 : side != 0;
            NodeQ<DIM> q1, q2;
            q1.rho = own ? qo.rho : qn.rho; q2.rho = own ? qn.rho : qo.rho;
            q1.beta = own ? qo.beta : qn.beta; q2.beta = own ? qn.beta : qo.beta;
            q1.ibeta = own ? qo.ibeta : qn.ibeta; q2.ibeta = own ? qn.ibeta : qo.ibeta;
            q1.lam = own ? qo.lam : qn.lam; q2.lam = own ? qn.lam : qo.lam;
#pragma unroll
            for (int d = 0; d < DIM; d++) { q1.v[d] = own ? qo.v[d] : qn.v[d]; q2.v[d] = own ? qn.v[d] : qo.v[d]; }
            if constexpr (GEN) {
                ec_flux<DIM, true, DIM == 3>(nv[side], normal_length<DIM>(nv[side], A.geo.nsc, A.geo.insc), q1, q2, P, quirk3d, F);
            } else {
                if (A.ec) ec_flux<DIM, false>(nvec, nr, q1, q2, P, false, F);
                else ec_flux<DIM, true, DIM == 3>(nvec, nr, q1, q2, P, quirk3d, F);
            }
            if constexpr (AXI) {
                // flux_num *= r (DGSEMIntegrator.cpp:190-205), the r of the
                // first element's node on both sides
                const double rl = S.R[el][ls[mo]], rg = A.geo.rnode[gn[side]];
                const double rf = own ? rl : rg;
#pragma unroll
                for (int v = 0; v < NV; v++) F[v] *= rf;
            }
            if constexpr (!AXI) {
                if (A.parabolic) {
                    // the neighbour's half of the mean of the two sides' traces
                    // Fv.n (boxes: per unit normal)
                    const double hn = GEN ? 0.5 : 0.5 * nr;
#pragma unroll
                    for (int v = 1; v < NV; v++) F[v] -= (double)ftn[side][v - 1] * hn;
                }
            }
            const double sg = own ? iw0 : -iw0;
#pragma unroll
            for (int v = 0; v < NV; v++) acc[mo][v] = sg * F[v];
        }
    }

    // ---- modal indicator and blending coefficient ----
    double alpha_e = 0.0;
    if constexpr (BLEND) {
        // modes = V^-1 (rho p), one direction at a time on that direction's
        // line threads (V^-1 = kron of 1-D inverses); after the last the
        // thread holds its line's modes and sums their squares: over the
        // modes of degree <= N-2 in every direction, over the others of
        // degree <= N-1, and over the rest.  The energies of
        // PerssonPeraireIndicator.cpp:38-52 are the first, the first two and
        // all three, and its 1 - m1/m and 1 - m2/m1 are the third over all
        // and the second over the first two, without the cancellation, which
        // alpha's steep logistic magnifies
#pragma unroll
        for (int rr = 0; rr < DIM; rr++) {
            if (lact && r == rr) {
                double q[NP], md[NP];
#pragma unroll
                for (int m = 0; m < NP; m++) q[m] = S.X[el][ls[m]];
#pragma unroll
                for (int a = 0; a < NP; a++) {
                    double s = 0.0;
#pragma unroll
                    for (int m = 0; m < NP; m++) s = (m == 0) ? v1i(a, 0) * q[0] : fma(v1i(a, m), q[m], s);
                    md[a] = s;
                }
                if (rr < DIM - 1) {
#pragma unroll
                    for (int m = 0; m < NP; m++) S.X[el][ls[m]] = md[m];
                } else {
                    double lo = 0.0;
#pragma unroll
                    for (int a = 0; a < NP - 2; a++) lo = fma(md[a], md[a], lo);
                    const double mid = md[NP - 2] * md[NP - 2], top = md[NP - 1] * md[NP - 1];
                    const bool in1 = la <= NP - 2 && lb <= NP - 2;
                    const bool in2 = NP > 2 && la <= NP - 3 && (DIM < 3 || lb <= NP - 3);
                    S.E[el][0][l] = in1 ? top : lo + mid + top;
                    S.E[el][1][l] = in2 ? mid : (in1 ? lo + mid : 0.0);
                    S.E[el][2][l] = in2 ? lo : 0.0;
                }
            }
            __syncthreads();
        }
        if constexpr (DIM == 3) {
            // rows of NP partial sums, then (below) the NP row sums
            if (lact && rem < 3 * NP) {
                const int c = rem / NP, row = rem - c * NP;
                double s = 0.0;
#pragma unroll
                for (int m = 0; m < NP; m++) s += S.E[el][c][row * NP + m];
                S.X[el][rem] = s;
            }
            __syncthreads();
        }
        if (lact && rem == 0) {
            double m3[3];
#pragma unroll
            for (int c = 0; c < 3; c++) {
                m3[c] = 0.0;
                if constexpr (DIM == 3) {
#pragma unroll
                    for (int m = 0; m < NP; m++) m3[c] += S.X[el][c * NP + m];
                } else {
#pragma unroll
                    for (int m = 0; m < NFP; m++) m3[c] += S.E[el][c][m];
                }
            }
            const double m1 = m3[2] + m3[1];
            double eta = m3[0] / (m1 + m3[0]);
            const double eta2 = m3[1] / m1;
            eta = (eta < eta2) ? eta2 : eta;
            // DGSEMOperator.cpp:67-77, sharpness 9.21024 (DGSEMOperator.hpp:50)
            double al = 1.0 / (1.0 + exp(-9.21024 * (eta - P.thresh) / P.thresh));
            if (al < P.alpha_min) al = 0.0;
            else if (al > 1.0 - P.alpha_min) al = 1.0;
            al = (P.alpha_max < al) ? P.alpha_max : al;
            S.Al[el] = al;
            A.alpha[e] = al;
            A.eta[e] = eta;
        }
        __syncthreads();
        if (lact) alpha_e = S.Al[el];
    }

    // ---- volume pairs ----
    // (1 - alpha) goes into the metric vector, in which the fluxes are linear
    if (lact) {
        const double om = BLEND ? 1.0 - alpha_e : 1.0;
        constexpr int MO = DIM == 3 ? 3 : 2;   // coefficients of a mesh line's metric polynomial
        double mc[GEN ? MO : 1][DIM];
        if constexpr (GEN) {
            line_metric<DIM>(S.Cn[el], r, DIM == 3 ? S.Xn[la] : 0.0, DIM == 3 ? S.Xn[lb] : 0.0, mc);
#pragma unroll
            for (int o = 0; o < MO; o++)
#pragma unroll
                for (int d = 0; d < DIM; d++) mc[o][d] *= om;
        }
#pragma unroll
        for (int d = 0; d < DIM; d++) nvec[d] *= om;
        // the mean of two nodes' metric vectors (AXI: times the r at the
        // pair's midpoint, DGSEMIntegrator.cpp:272-292)
        auto mean_metric = [&](int a, int b, double *n) {
            if constexpr (GEN) {
                const double x1 = 0.5 * (A.tab.x[a] + A.tab.x[b]);
                const double x2 = 0.5 * (A.tab.x[a] * A.tab.x[a] + A.tab.x[b] * A.tab.x[b]);
                const double rh = AXI ? 0.5 * (S.R[el][ls[a]] + S.R[el][ls[b]]) : 1.0;
#pragma unroll
                for (int d = 0; d < DIM; d++) {
                    n[d] = fma(mc[1][d], x1, mc[0][d]);
                    if constexpr (DIM == 3) n[d] = fma(mc[2][d], x2, n[d]);
                    if constexpr (AXI) n[d] *= rh;
                }
            } else {
#pragma unroll
                for (int d = 0; d < DIM; d++) n[d] = nvec[d];
            }
        };
        auto pairs = [&](auto range) {
            constexpr int RANGE = decltype(range)::value;
            const bool zq = QNS3 && r == 2;
#pragma unroll
            for (int a = 0; a < NP; a++) {
                const NodeQ<DIM> qa = node(a);
#pragma unroll
                for (int b = a + 1; b < NP; b++) {
                    // (read node b here: kept from pair to pair, a line's
                    // nodes would need 2 NP NV registers more)
                    asm volatile("" ::: "memory");
                    const NodeQ<DIM> qb = node(b);
                    double F[NV], n[DIM];
                    mean_metric(a, b, n);
                    if constexpr (RANGE == LM_PAIR) ec_flux<DIM, false>(n, 0.0, qa, qb, P, false, F);
                    else ec_flux_r<DIM, false, RANGE>(n, 0.0, qa, qb, P, false, F);
                    const double dab = dpair(a, b, 0), dba = dpair(a, b, 1);
#pragma unroll
                    for (int v = 0; v < NV; v++) {
                        acc[a][v] = fma(dab, F[v], acc[a][v]);
                        if (!zq) acc[b][v] = fma(dba, F[v], acc[b][v]);
                        // (not to be moved past the second flux's branches,
                        // which would keep every F)
                        if constexpr (QNS3 || RANGE == LM_PAIR) asm volatile("" : "+v"(acc[a][v]), "+v"(acc[b][v]));
                    }
                }
                if constexpr (QNS3) {
                    if (zq && a < NP - 1 && lb < NP - 1) {
                        // zeta partners a < b of node b: the eta flux of node
                        // a with node (i, NP-1, a) of its eta line; 0 on the
                        // eta line's last node (DGSEMIntegrator.cpp:702)
                        const int se = lines_slot<DIM, NP>(la, NP - 1, a);
                        NodeQ<DIM> qe;
                        qe.rho = sQ(el, 0, se);
#pragma unroll
                        for (int d = 0; d < DIM; d++) qe.v[d] = sQ(el, 1 + d, se);
                        qe.beta = sQ(el, NV - 1, se);
                        double n1[DIM];
                        if constexpr (GEN) {
                            double m1[MO][DIM];
                            line_metric<DIM>(S.Cn[el], 1, S.Xn[la], A.tab.x[a], m1);
                            const double xa = S.Xn[lb], xe = A.tab.x[NP - 1];
#pragma unroll
                            for (int d = 0; d < DIM; d++)
                                n1[d] = om * (m1[0][d] + 0.5 * (xa + xe) * m1[1][d] + 0.5 * (xa * xa + xe * xe) * m1[MO - 1][d]);
                        } else {
#pragma unroll
                            for (int d = 0; d < DIM; d++) n1[d] = d == 1 ? om * A.geo.nrm[1] : 0.0;
                        }
                        double g[NV];
                        if constexpr (RANGE == LM_PAIR) ec_flux<DIM, false>(n1, 0.0, qa, qe, P, false, g);
                        else ec_flux_r<DIM, false, RANGE>(n1, 0.0, qa, qe, P, false, g);
#pragma unroll
                        for (int b = a + 1; b < NP; b++)
#pragma unroll
                            for (int v = 0; v < NV; v++) {
                                acc[b][v] = fma(dpair(a, b, 1), g[v], acc[b][v]);
                                asm volatile("" : "+v"(acc[b][v]));
                            }
                    }
                }
            }
        };
        if constexpr (QNS3 && GEN) {
            // the range pair by pair: the second flux per node and its metrics
            // leave no registers for separate loops
            pairs(std::integral_constant<int, LM_PAIR>{});
        } else {
            double rlo = sQ(el, 0, ls[0]), rhi = rlo, blo = sQ(el, NV - 1, ls[0]), bhi = blo;
#pragma unroll
            for (int m = 1; m < NP; m++) {
                const double a = sQ(el, 0, ls[m]), b = sQ(el, NV - 1, ls[m]);
                rlo = fmin(rlo, a); rhi = fmax(rhi, a);
                blo = fmin(blo, b); bhi = fmax(bhi, b);
            }
            if constexpr (QNS3) {
                // and the zeta partners' second nodes
                if (r == 2 && lb < NP - 1)
#pragma unroll
                    for (int m = 0; m < NP - 1; m++) {
                        const int se = lines_slot<DIM, NP>(la, NP - 1, m);
                        const double a = sQ(el, 0, se), b = sQ(el, NV - 1, se);
                        rlo = fmin(rlo, a); rhi = fmax(rhi, a);
                        blo = fmin(blo, b); bhi = fmax(bhi, b);
                    }
            }
            // a pair's ratio is at most that of the line's extremes (positive
            // values; others fail both tests, but for a NaN, which fmin and
            // fmax drop and which makes its pairs' fluxes NaN in any range).
            // SHORT, where a line's values differ by at most 2%, in 3-D only: in
            // 2-D more waves hold lines of both kinds, and would run two loops,
            // as would the faithful NS-3D form on coarse meshes, whose loops are
            // long (N = 6, 210 elements 32 us without, 40 with)
            const double dr = rhi - rlo, rs = rhi + rlo, db = bhi - blo, bs = bhi + blo;
            if (DIM == 3 && !QNS3 && ((dr < 0.01 * rs) & (db < 0.01 * bs))) pairs(std::integral_constant<int, LM_SHORT>{});
            else if constexpr (NP >= 7) pairs(std::integral_constant<int, LM_PAIR>{});   // (registers)
            else if (__any(lm_outside(rlo, rhi) | lm_outside(blo, bhi))) pairs(std::integral_constant<int, LM_ANY>{});
            else pairs(std::integral_constant<int, LM_MID>{});
        }

        if constexpr (BLEND) {
            if (alpha_e > 0.0) {
                // blended element: subcell FV fluxes G along the line, 0 at the
                // element boundary (DGSEMIntegrator.cpp:972-1196)
                NodeQ<DIM> qa = face_node(0);
#pragma unroll
                for (int i = 0; i < NP - 1; i++) {
                    const NodeQ<DIM> qb = face_node(i + 1);
                    double ns[DIM], nd;
                    if constexpr (GEN) {
                        const double *sn = A.geo.subn + ((((size_t)e * DIM + r) * NFP + l) * (NP - 1) + i) * DIM;
#pragma unroll
                        for (int d = 0; d < DIM; d++) ns[d] = sn[d];
                        nd = normal_length<DIM>(ns, A.geo.nsc, A.geo.insc);
                        if constexpr (AXI) {
                            // flux_num *= mid_r (DGSEMIntegrator.cpp:1030-1032, 1110-1112)
                            const double rh = 0.5 * (S.R[el][ls[i]] + S.R[el][ls[i + 1]]);
                            nd *= rh;
#pragma unroll
                            for (int d = 0; d < DIM; d++) ns[d] *= rh;
                        }
                    } else {
                        nd = lane_pick3(A.tab.subn[0][i], A.tab.subn[1][i], A.tab.subn[2][i], r);
#pragma unroll
                        for (int d = 0; d < DIM; d++) ns[d] = d == r ? nd : 0.0;
                    }
                    double G[NV];
                    ec_flux<DIM, true>(ns, nd, qa, qb, P, quirk3d, G);
                    const double fa = alpha_e * rcp_nr(A.tab.w[i]), fb = alpha_e * rcp_nr(A.tab.w[i + 1]);
#pragma unroll
                    for (int v = 0; v < NV; v++) {
                        acc[i][v] = fma(fa, G[v], acc[i][v]);
                        acc[i + 1][v] = fma(-fb, G[v], acc[i + 1][v]);
                        asm volatile("" : "+v"(acc[i][v]), "+v"(acc[i + 1][v]));
                    }
                    qa = qb;
                }
            }
        }
    }

    // every start load has been used by now; saying so (free here) keeps a
    // load left unused on some lane's path from being waited for below
    // (gfx9's s_waitcnt immediate: vmcnt 0, expcnt 7, lgkmcnt 15)
    __builtin_amdgcn_s_waitcnt(0x0F70);

    // ---- the assembly's inputs, in flight during the direction sums where
    // the registers allow it
    constexpr bool PRE = NPASS <= 2;
    const double dt = step_dt(A);
    double yv[PRE ? NPASS : 1][NV], u0v[PRE ? NPASS : 1][NV], vs[PRE ? NPASS : 1][NV - 1], jn[PRE ? NPASS : 1];
    auto inputs = [&](int i, double *y, double *u0, double *vi, double &j) {
        const size_t gi = (size_t)ebase * K + i;
        const bool in = i < nact;
        j = (GEN && in) ? A.geo.jac[gi] : 1.0;
#pragma unroll
        for (int v = 0; v < NV; v++) {
            y[v] = (A.mode != 0 && in) ? A.y[v * NK + gi] : 0.0;
            u0[v] = (A.mode == 2 && in) ? A.u0[v * NK + gi] : 0.0;
            if (v > 0) vi[v - 1] = (A.parabolic && in) ? (double)static_cast<const VT *>(A.visc)[(v - 1) * NK + gi] : 0.0;
        }
    };
    if constexpr (PRE) {
#pragma unroll
        for (int p = 0; p < NPASS; p++) inputs(t + p * BLOCK, yv[p], u0v[p], vs[p], jn[p]);
    }
    __syncthreads();   // the partial sums take the rows' place

    // ---- node sums over the directions, in direction order ----
#pragma unroll
    for (int rr = 0; rr < DIM; rr++) {
        if (lact && r == rr) {
#pragma unroll
            for (int a = 0; a < NP; a++)
#pragma unroll
                for (int v = 0; v < NV; v++) sQ(el, v, ls[a]) = (rr == 0) ? acc[a][v] : sQ(el, v, ls[a]) + acc[a][v];
        }
        __syncthreads();
    }

    // ---- viscous volume term, stage update, store ----
#pragma unroll
    for (int p = 0; p < NPASS; p++) {
        const int i = t + p * BLOCK;
        if (i >= nact) continue;
        const int e2 = EPB == 1 ? 0 : i / K, n = i - e2 * K;
        const int s = lines_node_slot<DIM, NP>(n);
        const size_t gi = (size_t)ebase * K + i;
        constexpr int Z = 0;
        const int pp = PRE ? p : Z;
        if constexpr (!PRE) inputs(i, yv[0], u0v[0], vs[0], jn[0]);
        const double iJ = GEN ? rcp_nr(jn[pp]) : A.geo.invJ;
#pragma unroll
        for (int v = 0; v < NV; v++) {
            double tot = -sQ(e2, v, s);
            if (v > 0) tot += vs[pp][v - 1];
            tot *= iJ;
            if constexpr (AXI) {
                if (v == 2) {
                    tot += S.Pr[e2][s];   // pressure source (DGSEMIntegrator.cpp:411-426)
                    // ZeroAxisRadialMom (DGSEMOperator.cpp:521-533)
                    const int ax = A.geo.axm[gi];
                    if (ax >= 0 && (ax & 1)) tot = 0.0;
                }
            }
            double o = tot;
            if (A.mode != 0) {
                o = fma(dt, tot, yv[pp][v]);
                if (A.mode == 2) o = fma(A.c1, o, A.c0 * u0v[pp][v]);
            }
            A.out[v * NK + gi] = o;
        }
    }
    block_lam_max<BLOCK>(lam, lam_old, A.lam, S.Red, slot);
}

// Waves per SIMD to ask the register allocator for: 4 on 3-D boxes where 128
// registers suffice but for a few spills (N = 3: 14; N = 2 blended: none), else
// 3 (168).  45 x 43 x 41 N = 3 Navier-Stokes 228 -> 210 us per launch, mixed 251
// -> 224, 40 x 41 x 39 blended Euler 209 -> 193, N = 2 108 -> 101; 16^3 the same
// (its waves are 3 per SIMD).  2-D lines gain nothing from it (0.97 to 1.02).
constexpr int lines_waves(int DIM, int NP, bool BLEND, bool QNS3, bool OPEN, bool GEN)
{
    return DIM == 3 && (NP == 4 || (NP == 3 && BLEND)) && !QNS3 && !OPEN && !GEN ? 4 : 3;
}

template <int DIM, int NP, bool BLEND, bool QNS3, typename VT, int FB, bool OPEN = false, bool GEN = false,
          bool AXI = false>
__global__ void __launch_bounds__((LnCfg<DIM, NP, FB>::BLOCK))
__attribute__((amdgpu_waves_per_eu((lines_waves(DIM, NP, BLEND, QNS3, OPEN, GEN))))) k_rhs_l(const KArgs A)
{
    __shared__ LineSmem<DIM, NP, BLEND, FB, GEN, AXI> S;
    line_body<DIM, NP, BLEND, QNS3, VT, FB, OPEN, GEN, AXI>(A, xcd_remap(blockIdx.x, gridDim.x), blockIdx.x, S);
}

} // namespace prandtl
