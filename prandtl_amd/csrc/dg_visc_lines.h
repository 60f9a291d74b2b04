// k_visc_l: the viscous kernel of Cartesian boxes (periodic or with boundary
// sides), corrected mode, with one thread per tensor line (gfx950).  Same
// operator as k_visc there (LiftingBR1.cpp:10-66,156-219,311-407;
// DGSEMOperator.cpp:82-159; NavierStokesFlux.cpp:12-58;
// DGSEMIntegrator.cpp:435-549,617-641,705-738).
//
//  - What the viscous flux needs of the entropy-variable gradients are those
//    of beta v and -beta (beta = rho/p): grad v = T (grad(beta v) - v grad beta)
//    and grad T = -T^2 grad beta with T = p/rho.  The first entropy variable's
//    gradient cancels (EntropyGrad2PrimGrad forms the density gradient from it
//    and the heat flux takes it out again), so no logarithm is evaluated.
//    (Not in faithful mode, whose volume flux mixes two nodes' states, and not
//    for prandtl's gradient output: k_visc serves both.)
//  - node phase: v, T and beta of the workgroup's nodes into LDS;
//  - gradient phase: thread (element, direction r, line l) forms the line's
//    derivatives from registers, with the face jumps at its two ends, as
//    d_r v and d_r T;
//  - the direction threads exchange only what the stress needs, the sums
//    d_r v_c + d_c v_r and the divergence, through LDS rows that are added to
//    in direction order;
//  - flux phase: the line's flux along r stays in the thread's registers for
//    the D^ sums; the ends are the element's face traces, written for the
//    neighbours.  This element's half of each trace goes into the volume term
//    (D^ = D + E, E the boundary terms: half of E here, and k_rhs_l adds the
//    neighbour's half);
//  - the directions' sums are added in LDS in direction order.
//  A thread's components are ordered with its own direction first (r, r+1,
//  r+2 cyclically), so registers are indexed by constants and only LDS rows
//  and global offsets depend on r.
//  D is applied in even-odd form (half the multiply-adds, and few enough
//  entries for scalar registers), D^ as D and its boundary terms.
//
// Bound: HBM on large meshes: 0.72 GB, 0.16 ms at the 4.55 TB/s of a large copy,
// in 0.17 ms at 3-D N = 3 45 x 43 x 41; 2.2 GB, 0.48 ms, in 0.55 at N = 7 32^3 (0.22
// ms of vector issue, 0.16 ms of LDS).  At 16^3, all resident at once at three to
// four waves per SIMD, latency.  Against k_visc, which read a line's nodes once per node
// (240 LDS reads per node at N = 7, 80 here) and took four logarithms per node
// and face point, per launch: 3-D N = 3 16^3 17.2 -> 12.2 us, 45 x 43 x 41 208
// -> 170, N = 7 32^3 686 -> 540; mixed N = 3 16^3 15.6 (on the FP32 matrix
// cores) -> 9.5.  With one trace per face point instead of two to read, k_rhs_l
// takes 16.6 instead of 17.6, 242 instead of 250 and 980 instead of 1031.
// Error against long double, relative L2 of a right-hand side of a fine mesh, next
// to k_visc's: N = 4, 5 and 7 0.82 to 0.97 times; mixed, against FP64, 0.85 to 0.97 times.
//
// MIXED: the mixed-precision form, as k_visc's: v, T and the entropy variables,
// shifted by their value at the element's node 0, are formed in FP64 and
// rounded; the rest is FP32, the outputs included.
#pragma once
#include "dg_lines.h"

namespace prandtl {

template <int DIM, int NP, int FB> struct VlCfg : LnCfg<DIM, NP, FB> {
    using L = LnCfg<DIM, NP, FB>;
    static constexpr int NL = DIM + 1;              // flux components: momentum, energy
    static constexpr int NG = DIM == 3 ? 4 : 2;     // exchange rows: off-diagonal sums, divergence
    // rows of an element: v, T, then beta (mixed: the shifted entropy
    // variables), whose place the exchange rows take; the output sums start at row 0
    static constexpr int NR = DIM + 1 + (NG > NL ? NG : NL);
    static constexpr int ES = NR * L::KP + (DIM == 3 && NP == 4 ? (NR * L::KP % 32 == 0 ? 16 : 0) : 0);
};

// y = D x along a line, D in even-odd form (EvenOdd).  The even parts are taken
// of x - x_0, which has the same derivative: rounded sums of the values themselves
// would lose what their differences hold (the right-hand side's error grew by
// 54% at N = 4, 18% at N = 5 and 10% at N = 7 against sums over plain rows of D).
// In FP32 (the mixed form, whose values are shifted already) by plain rows.
template <int NP, typename R> __device__ __forceinline__ void line_deriv(const VArgs &A, const R *x, R *y)
{
    if constexpr (std::is_same<R, float>::value) {
#pragma unroll
        for (int a = 0; a < NP; a++)
#pragma unroll
            for (int m = 0; m < NP; m++) {
                const float d = (float)A.tab.D[a * MAXNP + m];
                y[a] = m == 0 ? d * x[0] : fmaf(d, x[m], y[a]);
            }
    } else {
        constexpr int H = NP / 2;
        const EvenOdd &M = A.eD;
        double p[H], q[H];
        const double xs = x[0];
#pragma unroll
        for (int m = 0; m < H; m++) {
            const double od = x[m] - x[NP - 1 - m];
            const double ev = m == 0 ? -od : (x[m] - xs) + (x[NP - 1 - m] - xs);
#pragma unroll
            for (int a = 0; a < H; a++) {
                p[a] = m == 0 ? M.e[4 * a] * ev : fma(M.e[4 * a + m], ev, p[a]);
                q[a] = m == 0 ? M.o[4 * a] * od : fma(M.o[4 * a + m], od, q[a]);
            }
            if constexpr (NP & 1) y[H] = m == 0 ? M.r[0] * od : fma(M.r[m], od, y[H]);
        }
#pragma unroll
        for (int a = 0; a < H; a++) {
            if constexpr (NP & 1) p[a] = fma(M.c[a], x[H] - xs, p[a]);
            y[a] = q[a] + p[a];
            y[NP - 1 - a] = q[a] - p[a];
        }
    }
}

template <int DIM, int NP, bool MIXED, int FB, bool OPEN>
__global__ void __launch_bounds__((VlCfg<DIM, NP, FB>::BLOCK))
__attribute__((amdgpu_waves_per_eu((VlCfg<DIM, NP, FB>::WAVES)))) k_visc_l(const VArgs A)
{
    using C = VlCfg<DIM, NP, FB>;
    using R = typename std::conditional<MIXED, float, double>::type;
    constexpr int NV = DIM + 2, NL = C::NL, K = C::K, NFP = C::NFP, TE = C::TE, EPB = C::EPB, BLOCK = C::BLOCK;
    constexpr int NPASS = C::NPASS, KP = C::KP, ES = C::ES;
    __shared__ R sQ[EPB * ES];
    __shared__ double sRef[MIXED ? EPB : 1][NL];
    if (A.skip && *A.skip) return;   // uniform: before any barrier
    const int t = threadIdx.x;
    const int ebase = xcd_remap(blockIdx.x, gridDim.x) * EPB;
    const int NE = A.geo.NE;
    const size_t NK = (size_t)NE * K;
    const Phys &P = A.phys;
    const LinePos<DIM, NP, FB> L(t);
    // (threads past the lines of a workgroup count on beyond DIM)
    const int el = L.el, r = L.r < DIM ? L.r : 0, l = L.l;
    const int e = ebase + el;
    const bool lact = (el < EPB) && (L.rem < TE) && (e < NE);
    int ls[NP];
    L.slots(ls);
    // component c of this thread: direction dc[c] = (r + c) mod DIM; its LDS row
    int dc[DIM], rv[DIM];
#pragma unroll
    for (int c = 0; c < DIM; c++) {
        dc[c] = r + c < DIM ? r + c : r + c - DIM;
        rv[c] = el * ES + dc[c] * KP;
    }
    const int rT = el * ES + DIM * KP, rB = el * ES + (DIM + 1) * KP;

    // ---- start loads: nodes, then the neighbour states at the line's ends
    const int nact = (NE - ebase) < EPB ? (NE - ebase) * K : EPB * K;
    double ys[NPASS][NV];
#pragma unroll
    for (int p = 0; p < NPASS; p++) {
        const int i = t + p * BLOCK;
        const size_t gi = (i < nact) ? (size_t)ebase * K + i : 0;
#pragma unroll
        for (int v = 0; v < NV; v++) ys[p][v] = A.y[v * NK + gi];
    }
    double pt[2][NV];   // in this thread's component order; a boundary side: this element's own face node
    int bt[2] = {BC_PERIODIC, BC_PERIODIC};
#pragma unroll
    for (int side = 0; side < 2; side++) {
        int en = lact ? neighbor_lane(A.geo, e, r, side) : 0;
        int nn = L.base + (side ? 0 : (NP - 1) * L.stride);
        if (OPEN && lact) {
            bt[side] = boundary_of(A.geo, e, r, side);
            if (bt[side] != BC_PERIODIC) { en = e; nn = L.base + (side ? (NP - 1) * L.stride : 0); }
        }
        const size_t g = lact ? (size_t)en * K + nn : 0;
        pt[side][0] = A.y[g];
#pragma unroll
        for (int c = 0; c < DIM; c++) pt[side][1 + c] = A.y[(size_t)(1 + dc[c]) * NK + g];
        pt[side][NV - 1] = A.y[(size_t)(NV - 1) * NK + g];
    }

    // v, T = p/rho and beta = rho/p of a state
    auto quants = [&](const double *s, double *v, double &T, double &b) {
        const double ri = rcp_nr(s[0]);
        double vsq = 0.0;
#pragma unroll
        for (int d = 0; d < DIM; d++) {
            v[d] = s[1 + d] * ri;
            vsq = (d == 0) ? v[d] * v[d] : fma(v[d], v[d], vsq);
        }
        const double p = P.gm1 * (s[NV - 1] - 0.5 * s[0] * vsq);
        T = p * ri;
        b = s[0] * rcp_nr(p);
    };

    // ---- node phase ----
    double wv[MIXED ? NPASS : 1][NL];
#pragma unroll
    for (int p = 0; p < NPASS; p++) {
        const int i = t + p * BLOCK;
        if (i >= nact) continue;
        const int e2 = EPB == 1 ? 0 : i / K, n = i - e2 * K;
        R *q = sQ + e2 * ES + lines_node_slot<DIM, NP>(n);
        double v[DIM], T, b;
        quants(ys[p], v, T, b);
#pragma unroll
        for (int d = 0; d < DIM; d++) q[d * KP] = (R)v[d];
        q[DIM * KP] = (R)T;
        if constexpr (MIXED) {
#pragma unroll
            for (int d = 0; d < DIM; d++) wv[p][d] = b * v[d];
            wv[p][DIM] = b;
            if (n == 0)
#pragma unroll
                for (int d = 0; d < NL; d++) sRef[e2][d] = wv[p][d];
        } else {
            q[(DIM + 1) * KP] = b;
        }
    }
    __syncthreads();
    if constexpr (MIXED) {
#pragma unroll
        for (int p = 0; p < NPASS; p++) {
            const int i = t + p * BLOCK;
            if (i >= nact) continue;
            const int e2 = EPB == 1 ? 0 : i / K, n = i - e2 * K;
            R *q = sQ + e2 * ES + lines_node_slot<DIM, NP>(n);
#pragma unroll
            for (int d = 0; d < NL; d++) q[(DIM + 1 + d) * KP] = (R)(wv[p][d] - sRef[e2][d]);
        }
        __syncthreads();
    }

    // ---- gradient phase: dv[a][c] = d_r v_c and dT[a] = d_r T of the line's nodes
    const R half = 0.5, iw0 = (R)A.iw0;
    const R nr = (R)lane_pick3(A.geo.nrm[0], A.geo.nrm[1], A.geo.nrm[2], r);
    R dv[NP][DIM], dT[NP];
    if (lact) {
        const R sc = nr * (R)A.geo.invJ;
        // jump[side][c] / w0: what the end points' derivatives gain, of beta
        // v_c and (c = DIM) of beta; xn: the neighbour's values, or on a
        // boundary side the lifting flux
        R xn[2][NL];
#pragma unroll
        for (int side = 0; side < 2; side++) {
            if (OPEN && bt[side] != BC_PERIODIC) {
                // f n_r / (w0 J) with the outward normal (LiftingBR1.cpp:311-407)
                double w[NV], fb[NV], o[5], s[NV];
                const double *bo = A.geo.bcs + (2 * r + side) * 5;
#pragma unroll
                for (int v = 0; v < 5; v++) o[v] = bo[v];
                // the state in the order of the directions
                s[0] = pt[side][0];
                s[NV - 1] = pt[side][NV - 1];
#pragma unroll
                for (int d = 0; d < DIM; d++) {
                    double x = pt[side][1];
#pragma unroll
                    for (int c = 1; c < DIM; c++) x = dc[c] == d ? pt[side][1 + c] : x;
                    s[1 + d] = x;
                }
                cons2entropy<DIM>(s, P, w);
                lift_flux<DIM>(bt[side], w, o, P, false, fb);
                const double sg = side ? 1.0 : -1.0;
#pragma unroll
                for (int c = 0; c < DIM; c++) {
                    double x = fb[1];
#pragma unroll
                    for (int d = 1; d < DIM; d++) x = dc[c] == d ? fb[1 + d] : x;
                    xn[side][c] = (R)(sg * x);
                }
                xn[side][DIM] = (R)(-sg * fb[NV - 1]);
            } else {
                double v[DIM], T, b;
                quants(pt[side], v, T, b);
#pragma unroll
                for (int c = 0; c < DIM; c++) xn[side][c] = MIXED ? (R)(b * v[c] - sRef[el][dc[c]]) : (R)(b * v[c]);
                xn[side][DIM] = MIXED ? (R)(b - sRef[el][DIM]) : (R)b;
            }
        }
        R x[NP], db[NP];
        // sum_m D_am x_m plus the jumps at the ends, scaled by n_r / J
        auto deriv = [&](int c, R *y) {
            line_deriv<NP, R>(A, x, y);
            const R jl = (OPEN && bt[0] != BC_PERIODIC) ? xn[0][c] : half * (x[0] - xn[0][c]);
            const R jh = (OPEN && bt[1] != BC_PERIODIC) ? xn[1][c] : half * (xn[1][c] - x[NP - 1]);
            y[0] = fma(iw0, jl, y[0]);
            y[NP - 1] = fma(iw0, jh, y[NP - 1]);
#pragma unroll
            for (int a = 0; a < NP; a++) y[a] = y[a] * sc;
        };
#pragma unroll
        for (int m = 0; m < NP; m++) x[m] = sQ[rB + (MIXED ? DIM * KP : 0) + ls[m]];
        deriv(DIM, db);
#pragma unroll
        for (int c = 0; c < DIM; c++) {
            R v[NP], y[NP];
            // (beta is read again for each component: kept, NP = 8 spills)
            asm volatile("" ::: "memory");
#pragma unroll
            for (int m = 0; m < NP; m++) {
                v[m] = sQ[rv[c] + ls[m]];
                if constexpr (MIXED) x[m] = sQ[rv[c] + (DIM + 1) * KP + ls[m]];
                else x[m] = sQ[rB + ls[m]] * v[m];
            }
            deriv(c, y);
#pragma unroll
            for (int a = 0; a < NP; a++) dv[a][c] = fma(-v[a], db[a], y[a]);
        }
#pragma unroll
        for (int a = 0; a < NP; a++) {
            const R T = sQ[rT + ls[a]];
#pragma unroll
            for (int c = 0; c < DIM; c++) dv[a][c] *= T;
            dT[a] = -(T * T) * db[a];
        }
    }
    __syncthreads();   // beta's row is dead: the exchange rows take its place

    // ---- the sums d_i v_j + d_j v_i (3-D: in the row of the third
    // direction) and the divergence, in direction order
    auto row_of = [](int i, int j) { return DIM == 3 ? 3 - i - j : 0; };
    const int rD = rB + (C::NG - 1) * KP;
#pragma unroll
    for (int rr = 0; rr < DIM; rr++) {
        if (lact && r == rr) {
#pragma unroll
            for (int a = 0; a < NP; a++) {
                R &dg = sQ[rD + ls[a]];
                dg = rr == 0 ? dv[a][0] : dg + dv[a][0];
#pragma unroll
                for (int c = 1; c < DIM; c++) {
                    const int d = (rr + c) % DIM;
                    R &od = sQ[rB + row_of(rr, d) * KP + ls[a]];
                    od = d > rr ? dv[a][c] : od + dv[a][c];
                }
            }
        }
        __syncthreads();
    }

    // ---- the line's flux along r (per unit normal), traces, D^ sums ----
    R f[NL][NP];
    if (lact) {
        const R mu_bulk = R(2) / R(3), two = 2;
        const R gm1i = (R)P.gm1i;
        int ro[DIM];
#pragma unroll
        for (int c = 1; c < DIM; c++) ro[c] = rB + (DIM == 3 ? dc[3 - c] : 0) * KP;   // row of (r, dc[c])
#pragma unroll
        for (int a = 0; a < NP; a++) {
            // (node by node: reads hoisted over all nodes spill at NP = 8)
            if constexpr (NP >= 7) asm volatile("" ::: "memory");
            R mu = (R)P.mu, lam_h = (R)P.lam_h;
            if (P.sutherland) {
                // mu(T) from p / (rho R) = T / R
                mu = sutherland_mu<R>(R(1), sQ[rT + ls[a]], (R)P.R_gas);
                lam_h = mu * (R)P.gamma * (R)P.PrInv;
            }
            f[0][a] = mu * (two * dv[a][0] - mu_bulk * sQ[rD + ls[a]]);
#pragma unroll
            for (int c = 1; c < DIM; c++) f[c][a] = mu * sQ[ro[c] + ls[a]];
            R en = lam_h * (gm1i * dT[a]);
#pragma unroll
            for (int c = 0; c < DIM; c++) en = fma(sQ[rv[c] + ls[a]], f[c][a], en);
            f[DIM][a] = en;
        }
        R *fvf = reinterpret_cast<R *>(A.fvf) + ((size_t)e * 2 * DIM + 2 * r) * NL * NFP + l;
#pragma unroll
        for (int side = 0; side < 2; side++)
#pragma unroll
            for (int c = 0; c < NL; c++)
                fvf[(side * NL + (c < DIM ? dc[c < DIM ? c : 0] : DIM)) * NFP] = f[c][side ? NP - 1 : 0];
        // half of E; on a boundary side, whose flux is k_rhs_l's alone, the whole
        const R edge[2] = {(OPEN && bt[0] != BC_PERIODIC) ? iw0 : half * iw0, (OPEN && bt[1] != BC_PERIODIC) ? iw0 : half * iw0};
#pragma unroll
        for (int c = 0; c < NL; c++) {
            R x[NP];
#pragma unroll
            for (int a = 0; a < NP; a++) x[a] = nr * f[c][a];
            line_deriv<NP, R>(A, x, f[c]);
            f[c][0] = fma(edge[0], x[0], f[c][0]);
            f[c][NP - 1] = fma(-edge[1], x[NP - 1], f[c][NP - 1]);
        }
    }
    __syncthreads();   // the output sums take the rows' place

    // ---- sum over the directions, in direction order ----
#pragma unroll
    for (int rr = 0; rr < DIM; rr++) {
        if (lact && r == rr) {
#pragma unroll
            for (int a = 0; a < NP; a++)
#pragma unroll
                for (int c = 0; c < NL; c++) {
                    const int row = c < DIM ? (rr + c) % DIM : DIM;
                    R &o = sQ[el * ES + row * KP + ls[a]];
                    o = rr == 0 ? f[c][a] : o + f[c][a];
                }
        }
        __syncthreads();
    }
    R *visc = reinterpret_cast<R *>(A.visc);
#pragma unroll
    for (int p = 0; p < NPASS; p++) {
        const int i = t + p * BLOCK;
        if (i >= nact) continue;
        const int e2 = EPB == 1 ? 0 : i / K, n = i - e2 * K;
        const int s = e2 * ES + lines_node_slot<DIM, NP>(n);
#pragma unroll
        for (int v = 0; v < NL; v++) visc[v * NK + (size_t)ebase * K + i] = sQ[s + v * KP];
    }
}

} // namespace prandtl
