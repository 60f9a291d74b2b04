// k_rhs_p: the flux-differencing RHS of k_rhs_l (dg_lines.h) with one thread
// per node and direction, for meshes too small to fill the chip with line
// threads (gfx950).  Thread (element, direction r, node) evaluates its node's
// NP - 1 pairs along r, its face point and its two subcell interfaces: every
// pair is evaluated twice, once per node, but a thread's chain is NP - 1
// fluxes instead of NP (NP-1) / 2, one face point instead of two and NP instead
// of NP^2 terms of the indicator's transforms.  A node's terms are the same
// operations in the same order as k_rhs_l's, so the results are equal bit for
// bit, whichever of the two a mesh's size selects (points_ok).
//
// Bound: the chain of dependent FP64 operations between the launch and the
// store, with at most a few waves per SIMD.  In 1-D, against a kernel that took
// pairs and interfaces as jobs through LDS, per stage: N = 3 128 elements 8.8 ->
// 8.4 us, 200,000 49 -> 34; N = 7 185 -> 83.
#pragma once
#include "dg_lines.h"

namespace prandtl {

// Elements per workgroup: the fewest whose threads fill 78% of their waves.
constexpr int points_epb(int TN)
{
    int e = TN >= 64 ? 1 : 64 / TN;
    while (e * TN * 100 < 78 * r64(e * TN) && r64((e + 1) * TN) <= 256) e++;
    return e;
}

template <int DIM, int NP, int FB = 0> struct PtCfg {
    static constexpr int NV = DIM + 2;
    static constexpr int K = npow(NP, DIM);
    static constexpr int NFP = npow(NP, DIM - 1);
    static constexpr int TN = DIM * K;
    static constexpr int EPB = FB ? FB / TN : points_epb(TN);
    static constexpr int BLOCK = FB ? FB : r64(EPB * TN);
    static constexpr int NR = NV + 1;   // rows: rho, v, beta, lambda
    static constexpr int KP = LnCfg<DIM, NP, 0>::KP;
    static constexpr int ES = NR * KP;
};

// Whether a workgroup of one element's node threads can be launched.
constexpr bool points_built(int DIM, int NP) { return DIM * npow(NP, DIM) <= 1024; }

// LDS of one tile (EPB elements).
template <int DIM, int NP, bool BLEND, int FB, bool GEN, bool AXI> struct PointSmem {
    using C = PtCfg<DIM, NP, FB>;
    double Q[C::EPB * C::ES];                                   // rows; then the partial sums
    double X[2][BLEND ? C::EPB : 1][BLEND ? C::KP : 1];         // indicator: rho p and its transforms, in turn
    double E[BLEND ? C::EPB : 1][3][BLEND ? C::NFP : 1];        // modal energies per line
    double Al[C::EPB];
    double Red[C::BLOCK / 64];
    double Cn[GEN ? C::EPB : 1][GEN ? (DIM == 3 ? 24 : 8) : 1];   // element corners
    double Xn[NP], W[NP];                                       // LGL nodes and weights
    double D2[NP * NP];                                         // 2 D + E
    double V1[BLEND ? NP * NP : 1];                             // inverse 1-D Vandermonde
    double R[AXI ? C::EPB : 1][AXI ? C::KP : 1];                // r of the nodes
    double Pr[AXI ? C::EPB : 1][AXI ? C::KP : 1];               // p of the nodes
};

// One tile, as line_body: the same template parameters and arguments.
template <int DIM, int NP, bool BLEND, bool QNS3, typename VT, int FB, bool OPEN = false, bool GEN = false,
          bool AXI = false>
__device__ __forceinline__ void point_body(const KArgs &A, const int tile, const int slot,
                                           PointSmem<DIM, NP, BLEND, FB, GEN, AXI> &S)
{
    using C = PtCfg<DIM, NP, FB>;
    constexpr int NV = C::NV, K = C::K, NFP = C::NFP, TN = C::TN, EPB = C::EPB, BLOCK = C::BLOCK, KP = C::KP, ES = C::ES;
    constexpr bool VISC = DIM > 1 && !AXI;   // built with viscous terms
    static_assert(!AXI || (GEN && DIM == 2), "axisymmetric meshes are quadrilateral meshes");
    auto sQ = [&](int e2, int row, int s) -> double & { return S.Q[e2 * ES + row * KP + s]; };

    if (A.skip && *A.skip) return;   // uniform: before any barrier
    const int t = threadIdx.x;
    const int ebase = tile * EPB;
    const int NE = A.geo.NE;
    const size_t NK = (size_t)NE * K;
    const Phys &P = A.phys;
    const bool quirk3d = A.quirks != 0;
    const double lam_old = (t == 0) ? A.lam[slot] : 0.0;

    // this thread's node: node m of line l of direction r (the lines' ends in
    // consecutive lanes)
    const int el = EPB == 1 ? 0 : t / TN, rem = t - el * TN;
    const int e = ebase + el;
    const bool lact = (el < EPB) && (rem < TN) && (e < NE);
    const int r = lact ? rem / K : 0;
    const int ml = rem - r * K;
    const int m = lact ? ml / NFP : 0, l = lact ? ml - m * NFP : 0;
    const int la = DIM == 3 ? l % NP : l, lb = DIM == 3 ? l / NP : 0;
    const int base = r == 0 ? l * NP : (DIM == 3 && r == 1 ? lb * NP * NP + la : l);
    const int stride = r == 0 ? 1 : (r == 1 ? NP : NP * NP);
    const bool end = lact && (m == 0 || m == NP - 1);
    const int side = m == 0 ? 0 : 1;
    // LDS slot of node q of the line
    auto slot_of = [&](int q) {
        if constexpr (DIM == 1) return q;
        else if constexpr (DIM == 2) return r == 0 ? lines_slot<DIM, NP>(q, la, 0) : lines_slot<DIM, NP>(la, q, 0);
        else return lines_slot<DIM, NP>(r == 0 ? q : la, r == 1 ? q : (r == 0 ? la : lb), r == 2 ? q : lb);
    };
    int ls[NP];
#pragma unroll
    for (int q = 0; q < NP; q++) ls[q] = slot_of(q);
    const int lo = slot_of(m);

    // ---- start loads ----
    const int nact = (NE - ebase) < EPB ? (NE - ebase) * K : EPB * K;
    const size_t ef = lact ? (size_t)e * (2 * DIM) + 2 * r + side : 0;
    int gn = 0, code = 0;
    if constexpr (GEN) {
        code = A.geo.fface[ef];
        gn = A.geo.fnb[ef * NFP + l];
    }
    double ys[NV];
    const size_t gi = (t < nact) ? (size_t)ebase * K + t : 0;
    AxNode xo, xn;   // AXI: what the recoveries of the node and its neighbour load
    size_t gt = 0;
    if constexpr (AXI) {
        xo = axis_load(A.y, A.geo, NK, gi);
    } else {
#pragma unroll
        for (int v = 0; v < NV; v++) {
            const double y = A.y[v * NK + gi];
            ys[v] = (t < nact) ? y : 1.0;
        }
    }
    double pn[NV], nv[DIM];   // the neighbour's state, normal and viscous trace (lanes at a line's end)
    VT ftn[NV - 1];
    int bt = BC_PERIODIC;
    {
        size_t g = 0;
        int en = 0;
        if constexpr (GEN) {
            bt = end ? (code >> 1) & 7 : BC_PERIODIC;
            if (end) g = bt != BC_PERIODIC ? (size_t)e * K + base + m * stride : (size_t)gn;
#pragma unroll
            for (int d = 0; d < DIM; d++) nv[d] = A.geo.fnor[(ef * NFP + l) * DIM + d];
        } else {
            en = end ? neighbor_lane(A.geo, e, r, side) : 0;
            int nn = base + (side ? 0 : (NP - 1) * stride);
            if (OPEN && end) {
                bt = boundary_of(A.geo, e, r, side);
                if (bt != BC_PERIODIC) { en = e; nn = base + m * stride; }
            }
            g = end ? (size_t)en * K + nn : 0;
        }
        if constexpr (AXI) {
            xn = axis_load(A.y, A.geo, NK, g);
            gt = g;
        } else {
#pragma unroll
            for (int v = 0; v < NV; v++) {
                const double y = A.y[v * NK + g];
                pn[v] = end ? y : 1.0;
            }
        }
        const bool vact = VISC && A.parabolic && end;
        const VT *fv = VISC && A.parabolic ? static_cast<const VT *>(A.fvf) : reinterpret_cast<const VT *>(A.y);
        size_t on = 0;
        if (vact) {
            if constexpr (GEN) {
                if (bt == BC_PERIODIC) {
                    const int nf = A.geo.fnf[ef];
                    const size_t fid = (size_t)(nf >> 1);
                    int l2;
                    if constexpr (DIM == 2) l2 = (nf & 1) ? NP - 1 - l : l;
                    else l2 = face_point_3<NP>(gn - (int)(fid / 6) * K, (int)(fid % 6) >> 1);
                    on = fid * (NV - 1) * NFP + l2;
                } else {
                    on = ef * (NV - 1) * NFP + l;
                }
            } else {
                const bool bnd = OPEN && bt != BC_PERIODIC;
                on = (bnd ? ef : (size_t)en * 2 * DIM + 2 * r + 1 - side) * (NV - 1) * NFP + l;
            }
        }
#pragma unroll
        for (int v = 0; v < NV - 1; v++) {
            const VT b = fv[on + v * NFP];
            ftn[v] = vact ? b : VT(0);
        }
    }
    for (int i = t; i < NP * NP; i += BLOCK) {
        S.D2[i] = A.tab.Dh2[(i / NP) * MAXNP + i % NP];
        if constexpr (BLEND) S.V1[i] = A.tab.V1i[(i / NP) * MAXNP + i % NP];
    }
    if (t < NP) { S.Xn[t] = A.tab.x[t]; S.W[t] = A.tab.w[t]; }
    if constexpr (GEN) {
        constexpr int NC = DIM == 3 ? 24 : 8;
        for (int i = t; i < EPB * NC; i += BLOCK)
            S.Cn[i / NC][i % NC] = (ebase + i / NC < NE) ? A.geo.corner[(size_t)ebase * NC + i] : 0.0;
    }

    // ---- node phase ----
    double lam = 0.0;
    const int e2 = EPB == 1 ? 0 : t / K, n2 = t - e2 * K;
    const int sn = t < nact ? lines_node_slot<DIM, NP>(n2) : 0;
    if (t < nact) {
        if constexpr (AXI) axis_state(A.y, A.geo, K, NK, gi, xo, ys);
        const NodeQ<DIM> q = node_quants<DIM>(ys, P);
        sQ(e2, 0, sn) = q.rho;
#pragma unroll
        for (int d = 0; d < DIM; d++) sQ(e2, 1 + d, sn) = q.v[d];
        sQ(e2, NV - 1, sn) = q.beta;
        sQ(e2, NV, sn) = q.lam;
        if constexpr (BLEND) {
            double vsq = 0.0;
#pragma unroll
            for (int d = 0; d < DIM; d++) vsq = (d == 0) ? q.v[d] * q.v[d] : vsq + q.v[d] * q.v[d];
            S.X[0][e2][sn] = q.rho * (P.gm1 * (ys[NV - 1] - 0.5 * q.rho * vsq));   // rho p
        }
        if constexpr (AXI) {
            // PressureFromConservative (DGSEMIntegrator.cpp:1306-1315)
            const double ke = 0.5 * ((ys[1] * ys[1] + ys[2] * ys[2]) / ys[0]);
            S.Pr[e2][sn] = P.gm1 * (ys[3] - ke);
            S.R[e2][sn] = A.geo.rnode[gi];
        }
        const double lq = (q.lam == q.lam) ? q.lam : 0.0;
        lam = (lam < lq) ? lq : lam;
    }
    __syncthreads();
    auto node = [&](int s) {
        NodeQ<DIM> q;
        q.rho = sQ(el, 0, s);
#pragma unroll
        for (int d = 0; d < DIM; d++) q.v[d] = sQ(el, 1 + d, s);
        q.beta = sQ(el, NV - 1, s);
        return q;
    };
    auto face_node = [&](int s) {
        NodeQ<DIM> q = node(s);
        q.lam = sQ(el, NV, s);
        q.ibeta = rcp_nr(q.beta);
        return q;
    };
    const double nr = GEN ? 0.0 : lane_pick3(A.geo.nrm[0], A.geo.nrm[1], A.geo.nrm[2], r);
    double nvec[DIM];
#pragma unroll
    for (int d = 0; d < DIM; d++) nvec[d] = (d == r) ? nr : 0.0;

    // ---- surface point ----
    double acc[NV];
#pragma unroll
    for (int v = 0; v < NV; v++) acc[v] = 0.0;
    if (end) {
        if constexpr (AXI) axis_state(A.y, A.geo, K, NK, gt, xn, pn);
        const double iw0 = 1.0 / A.tab.w[0];
        double F[NV];
        if ((OPEN || GEN) && bt != BC_PERIODIC) {
            // boundary point, as in line_body
            double bs[5], nn[DIM], lbd;
            if constexpr (GEN) {
                const int at = code >> 4;
#pragma unroll
                for (int v = 0; v < 5; v++) bs[v] = A.geo.bcs[at * 5 + v];
                if (A.geo.bfn && A.geo.bfn[at * 16] != 0.0) {
                    const double *fn = A.geo.bfn + at * 16;
                    const double *xp = A.geo.fxy + (ef * NFP + l) * 2;
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
                for (int d = 0; d < DIM; d++) nn[d] = nv[d];
                lbd = boundary_flux_vn<DIM>(bt, nn, pn, bs, P, quirk3d, F);
            } else {
#pragma unroll
                for (int v = 0; v < 5; v++) bs[v] = A.geo.bcs[(2 * r + side) * 5 + v];
#pragma unroll
                for (int d = 0; d < DIM; d++) nn[d] = side ? nvec[d] : -nvec[d];
                lbd = boundary_flux<DIM>(bt, r, side ? nr : -nr, nr, pn, bs, P, quirk3d, F);
            }
            lam = (lam < lbd) ? lbd : lam;
            if constexpr (AXI) {
                const double rf = S.R[el][lo];
#pragma unroll
                for (int v = 0; v < NV; v++) F[v] *= rf;
            }
            if (VISC && A.parabolic && (bt == BC_OUTFLOW || bt == BC_NOSLIP)) {
                double fn[NV], n2q = nn[0] * nn[0];
#pragma unroll
                for (int d = 1; d < DIM; d++) n2q = n2q + nn[d] * nn[d];
#pragma unroll
                for (int v = 1; v < NV; v++) fn[v] = GEN ? (double)ftn[v - 1] : (double)ftn[v - 1] * (side ? nr : -nr);
                if (bt == BC_NOSLIP) {
                    double en = bs[0] * fn[1];
#pragma unroll
                    for (int d = 1; d < DIM; d++) en = en + bs[d] * fn[1 + d];
                    fn[NV - 1] = en + bs[3] * sqrt(n2q);
                }
#pragma unroll
                for (int v = 1; v < NV; v++) F[v] -= fn[v];
            }
#pragma unroll
            for (int v = 0; v < NV; v++) acc[v] = iw0 * F[v];
        } else {
            NodeQ<DIM> qo = face_node(lo), qn = node_quants<DIM>(pn, P);
            qn.ibeta = rcp_nr(qn.beta);
            if (VISC && A.parabolic && A.quirks) {
                alias_quants<DIM>(qo, P);
                alias_quants<DIM>(qn, P);
            }
            const bool own = GEN ? (code & 1) != 0 : side != 0;
            NodeQ<DIM> q1, q2;
            q1.rho = own ? qo.rho : qn.rho; q2.rho = own ? qn.rho : qo.rho;
            q1.beta = own ? qo.beta : qn.beta; q2.beta = own ? qn.beta : qo.beta;
            q1.ibeta = own ? qo.ibeta : qn.ibeta; q2.ibeta = own ? qn.ibeta : qo.ibeta;
            q1.lam = own ? qo.lam : qn.lam; q2.lam = own ? qn.lam : qo.lam;
#pragma unroll
            for (int d = 0; d < DIM; d++) { q1.v[d] = own ? qo.v[d] : qn.v[d]; q2.v[d] = own ? qn.v[d] : qo.v[d]; }
            if constexpr (GEN) {
                ec_flux<DIM, true, DIM == 3>(nv, normal_length<DIM>(nv, A.geo.nsc, A.geo.insc), q1, q2, P, quirk3d, F);
            } else {
                if (A.ec) ec_flux<DIM, false>(nvec, nr, q1, q2, P, false, F);
                else ec_flux<DIM, true, DIM == 3>(nvec, nr, q1, q2, P, quirk3d, F);
            }
            if constexpr (AXI) {
                const double rl = S.R[el][lo], rg = A.geo.rnode[gn];
                const double rf = own ? rl : rg;
#pragma unroll
                for (int v = 0; v < NV; v++) F[v] *= rf;
            }
            if (VISC && A.parabolic) {
                const double hn = GEN ? 0.5 : 0.5 * nr;
#pragma unroll
                for (int v = 1; v < NV; v++) F[v] -= (double)ftn[v - 1] * hn;
            }
            const double sg = own ? iw0 : -iw0;
#pragma unroll
            for (int v = 0; v < NV; v++) acc[v] = sg * F[v];
        }
    }

    // ---- modal indicator and blending coefficient (line_body's, one mode per thread) ----
    double alpha_e = 0.0;
    if constexpr (BLEND) {
#pragma unroll
        for (int rr = 0; rr < DIM; rr++) {
            if (lact && r == rr) {
                double s = 0.0;
#pragma unroll
                for (int q = 0; q < NP; q++) {
                    const double x = S.X[rr & 1][el][ls[q]];
                    s = (q == 0) ? S.V1[m * NP] * x : fma(S.V1[m * NP + q], x, s);
                }
                S.X[1 - (rr & 1)][el][lo] = s;
            }
            __syncthreads();
        }
        if (lact && r == DIM - 1 && m == 0) {
            const double(*X)[KP] = S.X[DIM & 1];
            double e0 = 0.0;
#pragma unroll
            for (int a = 0; a < NP - 2; a++) { const double x = X[el][ls[a]]; e0 = fma(x, x, e0); }
            const double x1 = X[el][ls[NP - 2]], x2 = X[el][ls[NP - 1]];
            const double mid = x1 * x1, top = x2 * x2;
            const bool in1 = (DIM == 1 || la <= NP - 2) && lb <= NP - 2;
            const bool in2 = NP > 2 && (DIM == 1 || la <= NP - 3) && (DIM < 3 || lb <= NP - 3);
            S.E[el][0][l] = in1 ? top : e0 + mid + top;
            S.E[el][1][l] = in2 ? mid : (in1 ? e0 + mid : 0.0);
            S.E[el][2][l] = in2 ? e0 : 0.0;
        }
        __syncthreads();
        if constexpr (DIM == 3) {
            if (lact && rem < 3 * NP) {
                const int c = rem / NP, row = rem - c * NP;
                double s = 0.0;
#pragma unroll
                for (int q = 0; q < NP; q++) s += S.E[el][c][row * NP + q];
                S.X[1 - (DIM & 1)][el][rem] = s;
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
                    for (int q = 0; q < NP; q++) m3[c] += S.X[1 - (DIM & 1)][el][c * NP + q];
                } else {
#pragma unroll
                    for (int q = 0; q < NFP; q++) m3[c] += S.E[el][c][q];
                }
            }
            const double m1 = m3[2] + m3[1];
            double eta = m3[0] / (m1 + m3[0]);
            const double eta2 = m3[1] / m1;
            eta = (eta < eta2) ? eta2 : eta;
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

    // ---- volume pairs of the node, partners in ascending order ----
    if (lact) {
        const double om = BLEND ? 1.0 - alpha_e : 1.0;
        constexpr int MO = DIM == 3 ? 3 : 2;
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
        const NodeQ<DIM> qa = node(lo);
        const double xa = S.Xn[m];
        const double ra = AXI ? S.R[el][lo] : 1.0;
        auto pairs = [&](auto range) {
            constexpr int RANGE = decltype(range)::value;
#pragma unroll
            for (int j = 1; j < NP; j++) {
                const int b = j - 1 + (j > m ? 1 : 0);   // the j-th of the others
                if constexpr (QNS3) {
                    if (r == 2 && b < m) {
                        // zeta partners b < m, as in line_body: the eta flux of
                        // node b with node (i, NP-1, b) of its eta line
                        if (lb < NP - 1) {
                            const NodeQ<DIM> qz = node(slot_of(b)), qe = node(lines_slot<DIM, NP>(la, NP - 1, b));
                            double n1[DIM], g[NV];
                            if constexpr (GEN) {
                                double m1[MO][DIM];
                                line_metric<DIM>(S.Cn[el], 1, S.Xn[la], S.Xn[b], m1);
                                const double xb = S.Xn[lb], xe = S.Xn[NP - 1];
#pragma unroll
                                for (int d = 0; d < DIM; d++)
                                    n1[d] = om * (m1[0][d] + 0.5 * (xb + xe) * m1[1][d] + 0.5 * (xb * xb + xe * xe) * m1[MO - 1][d]);
                            } else {
#pragma unroll
                                for (int d = 0; d < DIM; d++) n1[d] = d == 1 ? om * A.geo.nrm[1] : 0.0;
                            }
                            ec_flux<DIM, false>(n1, 0.0, qz, qe, P, false, g);
                            const double d2 = S.D2[m * NP + b];
#pragma unroll
                            for (int v = 0; v < NV; v++) acc[v] = fma(d2, g[v], acc[v]);
                        }
                        continue;
                    }
                }
                const NodeQ<DIM> qb = node(slot_of(b));
                double F[NV], n[DIM];
                if constexpr (GEN) {
                    // (the lower node first, as line_body writes the sums)
                    const double xb = S.Xn[b], p = b < m ? xb : xa, q = b < m ? xa : xb;
                    const double x1 = 0.5 * (p + q), x2 = 0.5 * (p * p + q * q);
#pragma unroll
                    for (int d = 0; d < DIM; d++) {
                        n[d] = fma(mc[1][d], x1, mc[0][d]);
                        if constexpr (DIM == 3) n[d] = fma(mc[2][d], x2, n[d]);
                        if constexpr (AXI) n[d] *= 0.5 * (ra + S.R[el][slot_of(b)]);
                    }
                } else {
#pragma unroll
                    for (int d = 0; d < DIM; d++) n[d] = nvec[d];
                }
                if constexpr (RANGE == LM_PAIR) ec_flux<DIM, false>(n, 0.0, qa, qb, P, false, F);
                else ec_flux_r<DIM, false, RANGE>(n, 0.0, qa, qb, P, false, F);
                const double d2 = S.D2[m * NP + b];
#pragma unroll
                for (int v = 0; v < NV; v++) acc[v] = fma(d2, F[v], acc[v]);
            }
        };
        if constexpr (QNS3) {
            pairs(std::integral_constant<int, LM_PAIR>{});
        } else {
            double rlo = sQ(el, 0, ls[0]), rhi = rlo, blo = sQ(el, NV - 1, ls[0]), bhi = blo;
#pragma unroll
            for (int q = 1; q < NP; q++) {
                const double a = sQ(el, 0, ls[q]), b = sQ(el, NV - 1, ls[q]);
                rlo = fmin(rlo, a); rhi = fmax(rhi, a);
                blo = fmin(blo, b); bhi = fmax(bhi, b);
            }
            const double dr = rhi - rlo, rs = rhi + rlo, db = bhi - blo, bs = bhi + blo;
            if (DIM == 3 && ((dr < 0.01 * rs) & (db < 0.01 * bs))) pairs(std::integral_constant<int, LM_SHORT>{});
            else if (__any(lm_outside(rlo, rhi) | lm_outside(blo, bhi))) pairs(std::integral_constant<int, LM_ANY>{});
            else pairs(std::integral_constant<int, LM_MID>{});
        }

        if constexpr (BLEND) {
            if (alpha_e > 0.0) {
                // subcell interfaces below and above the node
#pragma unroll
                for (int up = 0; up < 2; up++) {
                    const int i = up ? m : m - 1;   // interface between nodes i and i + 1
                    if (i < 0 || i >= NP - 1) continue;
                    const NodeQ<DIM> q1 = face_node(slot_of(i)), q2 = face_node(slot_of(i + 1));
                    double ns[DIM], nd;
                    if constexpr (GEN) {
                        const double *sv = A.geo.subn + ((((size_t)e * DIM + r) * NFP + l) * (NP - 1) + i) * DIM;
#pragma unroll
                        for (int d = 0; d < DIM; d++) ns[d] = sv[d];
                        nd = normal_length<DIM>(ns, A.geo.nsc, A.geo.insc);
                        if constexpr (AXI) {
                            const double rh = 0.5 * (S.R[el][slot_of(i)] + S.R[el][slot_of(i + 1)]);
                            nd *= rh;
#pragma unroll
                            for (int d = 0; d < DIM; d++) ns[d] *= rh;
                        }
                    } else {
                        nd = A.tab.subn[0][0];
#pragma unroll
                        for (int q = 0; q < NP - 1; q++) {
                            const double x = lane_pick3(A.tab.subn[0][q], A.tab.subn[1][q], A.tab.subn[2][q], r);
                            nd = q == i ? x : nd;
                        }
#pragma unroll
                        for (int d = 0; d < DIM; d++) ns[d] = d == r ? nd : 0.0;
                    }
                    double G[NV];
                    ec_flux<DIM, true>(ns, nd, q1, q2, P, quirk3d, G);
                    const double f = alpha_e * rcp_nr(S.W[m]);
#pragma unroll
                    for (int v = 0; v < NV; v++) acc[v] = fma(up ? f : -f, G[v], acc[v]);
                }
            }
        }
    }

    // ---- assembly's inputs, then the sums over the directions, in direction order ----
    const double dt = step_dt(A);
    const bool in = t < nact;
    double u0v[NV], vs[NV - 1], jn = 1.0;
    if (GEN && in) jn = A.geo.jac[gi];
#pragma unroll
    for (int v = 0; v < NV; v++) {
        u0v[v] = (A.mode == 2 && in) ? A.u0[v * NK + gi] : 0.0;
        if constexpr (AXI) ys[v] = (A.mode != 0 && in) ? A.y[v * NK + gi] : 0.0;   // r U
        if (v > 0) vs[v - 1] = (VISC && A.parabolic && in) ? (double)static_cast<const VT *>(A.visc)[(v - 1) * NK + gi] : 0.0;
    }
    __syncthreads();   // the partial sums take the rows' place
#pragma unroll
    for (int rr = 0; rr < DIM; rr++) {
        if (lact && r == rr)
#pragma unroll
            for (int v = 0; v < NV; v++) sQ(el, v, lo) = (rr == 0) ? acc[v] : sQ(el, v, lo) + acc[v];
        __syncthreads();
    }
    if (in) {
        const double iJ = GEN ? rcp_nr(jn) : A.geo.invJ;
#pragma unroll
        for (int v = 0; v < NV; v++) {
            double tot = -sQ(e2, v, sn);
            if (v > 0) tot += vs[v - 1];
            tot *= iJ;
            if constexpr (AXI) {
                if (v == 2) {
                    // pressure source and ZeroAxisRadialMom, as in line_body
                    tot += S.Pr[e2][sn];
                    const int ax = A.geo.axm[gi];
                    if (ax >= 0 && (ax & 1)) tot = 0.0;
                }
            }
            double o = tot;
            if (A.mode != 0) {
                o = fma(dt, tot, ys[v]);
                if (A.mode == 2) o = fma(A.c1, o, A.c0 * u0v[v]);
            }
            A.out[v * NK + gi] = o;
        }
    }
    block_lam_max<BLOCK>(lam, lam_old, A.lam, S.Red, slot);
}

template <int DIM, int NP, bool BLEND, bool QNS3, typename VT, bool OPEN, bool GEN, bool AXI = false>
__global__ void __launch_bounds__((PtCfg<DIM, NP>::BLOCK)) k_rhs_p(const KArgs A)
{
    __shared__ PointSmem<DIM, NP, BLEND, 0, GEN, AXI> S;
    point_body<DIM, NP, BLEND, QNS3, VT, 0, OPEN, GEN, AXI>(A, xcd_remap(blockIdx.x, gridDim.x), blockIdx.x, S);
}

} // namespace prandtl
