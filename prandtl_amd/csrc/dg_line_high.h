// k_rhs_lh: the flux-differencing RHS of Cartesian boxes at high order (3-D,
// N = 5..7), one thread per tensor line (gfx950).
//
// The operator and the decomposition are k_rhs_ln's (dg_line.h): a node phase
// into LDS, a line phase with the line's sums in registers, the DIM partial
// sums of a node added in LDS.  What differs follows from the line's length:
//
//  - LDS holds five rows per element (rho, v, beta): what a pair reads, and as
//    many as the partial sums need, which take the rows' place afterwards.
//    Everything else of a node is formed from them where it is used (face
//    points, subcell interfaces); the stage update reads the state again,
//    from the cache.  3-D N = 7: 20 KB per element instead of 75, so the
//    registers and not the LDS set the occupancy.
//  - The pairs of a line are straight-line code without branches.  A line's
//    smallest and largest rho and beta bound the ratio of every pair, so the
//    range of the log means (log_means) is chosen once per line, with one
//    unrolled pair loop per range.  The choice depends on the line's own
//    values alone, so results do not depend on the lanes that share a wave.
//  - Sums are kept in units of 1/J: a node's total is
//    (visc - acc) / J, acc = (1 - alpha) vol - alpha fv - surface / w0.
//  - The indicator's transforms run on the line threads: NP values in
//    registers, NP^2 multiply-adds with table entries from scalar registers.
//
// What bounds it (3-D N = 7, 32^3 elements, Navier-Stokes, blended): 3,025
// vector instructions per wave, 0.53 ms of issue, and about 3 GB of HBM
// traffic, 0.55 ms at the copy rate; at three waves per SIMD (168 registers,
// 80 of them the line's sums) neither is hidden completely.  Against the
// tile kernel, which put every pair's flux through LDS in 12 chunks, summed
// by a quarter of the threads: 3.0 -> 0.93 ms per launch; the right-hand
// side 3.54 -> 1.60 ms.  Whole right-hand sides of smaller boxes: Euler 16^3
// N = 7 279 -> 95 us, 9x8x7 N = 6 39.8 -> 18.2, 10x9x8 N = 5 25.0 -> 18.2.
// Two waves per SIMD (256 registers) measured 1.16 times slower.
#pragma once
#include "dg_line.h"

namespace prandtl {

// The orders this kernel is built for: every 3-D order above k_rhs_ln's.
constexpr bool high_built(int DIM, int NP) { return DIM == 3 && NP >= 6; }

template <int DIM, int NP, int FB = 0> struct HCfg {
    static constexpr int NV = DIM + 2;
    static constexpr int K = npow(NP, DIM);
    static constexpr int NFP = npow(NP, DIM - 1);
    static constexpr int TE = DIM * NFP;
    static constexpr int EPB = FB ? FB / TE : line_epb(TE);
    static constexpr int BLOCK = FB ? FB : r64(EPB * TE);
    static constexpr int NPASS = (EPB * K + BLOCK - 1) / BLOCK;
    static_assert(EPB >= 1, "a workgroup holds an element's lines");
#ifndef PRANDTL_HIGH_WAVES
#define PRANDTL_HIGH_WAVES 3
#endif
    static constexpr int WAVES = PRANDTL_HIGH_WAVES;
};

// LDS slot of node (i, j, k).  NP = 8: row (j + k) mod 8, column (i + j + 2k)
// mod 8 of plane k.  32 lanes of a wave hold one direction's lines whose
// other two indices run over all 8 and over 4 consecutive values; in each of
// the planes i = m, j = m, k = m the slots of such lines are distinct mod 32,
// so every line-phase access and every node-order access covers the 32
// eight-byte banks once.  Rows are K doubles, a multiple of 64, so two rows'
// values load with one instruction.  Other orders: one double of padding per
// x-row (their lines do not align with half-waves).
template <int NP> __device__ __forceinline__ int high_slot(int i, int j, int k)
{
    if constexpr (NP == 8) return 64 * k + 8 * ((j + k) & 7) + ((i + j + 2 * k) & 7);
    else {
        const int n = (k * NP + j) * NP + i;
        return n + n / NP;
    }
}

// What a two-point flux with dissipation needs of a node beyond (rho, v,
// beta): 1/beta and lambda.  Both neighbours of a face point form them here
// from the same three, so that the point's flux is the same on both sides.
template <int DIM> __device__ __forceinline__ void face_quants(NodeQ<DIM> &q, const Phys &P)
{
    double vsq = 0.0;
#pragma unroll
    for (int d = 0; d < DIM; d++) vsq = (d == 0) ? q.v[d] * q.v[d] : fma(q.v[d], q.v[d], vsq);
    q.ibeta = rcp_nr(q.beta);
    q.lam = sqrt(vsq) + sqrt(0.5 * P.gamma * q.ibeta);
}

template <int DIM, int NP, bool BLEND, bool QNS3, typename VT, int FB, bool OPEN>
__global__ void __launch_bounds__((HCfg<DIM, NP, FB>::BLOCK))
__attribute__((amdgpu_waves_per_eu((HCfg<DIM, NP, FB>::WAVES)))) k_rhs_lh(const KArgs A)
{
    using C = HCfg<DIM, NP, FB>;
    constexpr int NV = C::NV, K = C::K, NFP = C::NFP, TE = C::TE, EPB = C::EPB, BLOCK = C::BLOCK, NPASS = C::NPASS;
    constexpr int KP = NP == 8 ? K : K + K / NP;
    static_assert(DIM == 3, "high-order line kernel: 3-D boxes");
    __shared__ double sQ[EPB][NV][KP];                      // rho, v, beta; then the partial sums
    __shared__ double sX[BLEND ? EPB : 1][BLEND ? KP : 1];   // indicator: rho p and its transforms
    __shared__ double sE[BLEND ? EPB : 1][3][BLEND ? NFP : 1];
    __shared__ double sAl[EPB];
    __shared__ double sRed[(BLOCK + 63) / 64];

    if (A.skip && *A.skip) return;   // uniform: before any barrier
    const int t = threadIdx.x;
    const int ebase = xcd_remap(blockIdx.x, gridDim.x) * EPB;
    const int NE = A.geo.NE;
    const size_t NK = (size_t)NE * K;
    const Phys &P = A.phys;
    const bool quirk3d = A.quirks != 0;
    const double dt = step_dt(A);
    const double lam_old = (t == 0) ? A.lam[blockIdx.x] : 0.0;

    // this thread's line: element el, direction r, line l with the other two
    // indices la, lb.  NP = 8: a wave is one direction, so r is scalar
    const int el = EPB == 1 ? 0 : t / TE;
    const int rem = t - el * TE;
    int r = rem / NFP;
    if constexpr (NP == 8 && EPB == 1) r = __builtin_amdgcn_readfirstlane(r);
    const int l = rem - r * NFP;
    const int la = l % NP, lb = l / NP;
    const int e = ebase + el;
    const bool lact = (el < EPB) && (rem < TE) && (e < NE);
    const int base = r == 0 ? l * NP : (r == 1 ? lb * NP * NP + la : l);
    const int stride = r == 0 ? 1 : (r == 1 ? NP : NP * NP);
    int ls[NP];
#pragma unroll
    for (int m = 0; m < NP; m++) ls[m] = high_slot<NP>(r == 0 ? m : la, r == 1 ? m : (r == 0 ? la : lb), r == 2 ? m : lb);
    const double nr = lane_pick3(A.geo.nrm[0], A.geo.nrm[1], A.geo.nrm[2], r);
    const double nvec[3] = {r == 0 ? nr : 0.0, r == 1 ? nr : 0.0, r == 2 ? nr : 0.0};

    // ---- start loads: the nodes first, then the traces at the line's ends
    // (see k_rhs_ln: every load on every path, lanes without one read index 0)
    const int nact = (NE - ebase) < EPB ? (NE - ebase) * K : EPB * K;
    double ysp[NPASS][NV];
#pragma unroll
    for (int p = 0; p < NPASS; p++) {
        const int i = t + p * BLOCK;
        const size_t gi = (i < nact) ? (size_t)ebase * K + i : 0;
#pragma unroll
        for (int v = 0; v < NV; v++) {
            const double y = A.y[v * NK + gi];
            ysp[p][v] = (i < nact) ? y : 1.0;
        }
    }
    double pt[2][NV];       // neighbour states; on a boundary side this element's own face node
    int bt[2] = {BC_PERIODIC, BC_PERIODIC};
    VT fto[2][NV - 1], ftn[2][NV - 1];
#pragma unroll
    for (int side = 0; side < 2; side++) {
        int en = lact ? neighbor_lane(A.geo, e, r, side) : 0;
        int nn = base + (side ? 0 : (NP - 1) * stride);
        if (OPEN && lact) {
            bt[side] = boundary_of(A.geo, e, r, side);
            if (bt[side] != BC_PERIODIC) { en = e; nn = base + (side ? (NP - 1) * stride : 0); }
        }
        const size_t g = lact ? (size_t)en * K + nn : 0;
#pragma unroll
        for (int v = 0; v < NV; v++) {
            const double y = A.y[v * NK + g];
            pt[side][v] = lact ? y : 1.0;
        }
        const bool vact = A.parabolic && lact;
        const VT *fv = A.parabolic ? static_cast<const VT *>(A.fvf) : reinterpret_cast<const VT *>(A.y);
        const size_t oo = vact ? (((size_t)e * 2 * DIM + 2 * r + side) * (NV - 1)) * NFP + l : 0;
        const size_t on = vact ? (((size_t)en * 2 * DIM + 2 * r + 1 - side) * (NV - 1)) * NFP + l : 0;
#pragma unroll
        for (int v = 0; v < NV - 1; v++) {
            const VT a = fv[oo + v * NFP], b = fv[on + v * NFP];
            fto[side][v] = vact ? a : VT(0);
            ftn[side][v] = vact ? b : VT(0);
        }
    }

    // ---- node phase ----
    double lam = 0.0;
#pragma unroll
    for (int p = 0; p < NPASS; p++) {
        const int i = t + p * BLOCK;
        if (i >= nact) continue;
        const int e2 = EPB == 1 ? 0 : i / K, n = i - e2 * K;
        const int s = high_slot<NP>(n % NP, (n / NP) % NP, n / (NP * NP));
        const NodeQ<DIM> q = node_quants<DIM>(ysp[p], P);
        sQ[e2][0][s] = q.rho;
#pragma unroll
        for (int d = 0; d < DIM; d++) sQ[e2][1 + d][s] = q.v[d];
        sQ[e2][NV - 1][s] = q.beta;
        if constexpr (BLEND) {
            double vsq = 0.0;
#pragma unroll
            for (int d = 0; d < DIM; d++) vsq = (d == 0) ? q.v[d] * q.v[d] : vsq + q.v[d] * q.v[d];
            sX[e2][s] = q.rho * (P.gm1 * (ysp[p][NV - 1] - 0.5 * q.rho * vsq));   // rho p
        }
        const double lq = (q.lam == q.lam) ? q.lam : 0.0;
        lam = (lam < lq) ? lq : lam;
    }
    __syncthreads();
    auto node = [&](int m) {
        NodeQ<DIM> q;
        q.rho = sQ[el][0][ls[m]];
#pragma unroll
        for (int d = 0; d < DIM; d++) q.v[d] = sQ[el][1 + d][ls[m]];
        q.beta = sQ[el][NV - 1][ls[m]];
        return q;
    };

    // ---- surface points of the line's ends, flux toward +e_r (elem1 = low
    // side): the first terms of the end nodes' sums
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
            double fvn[NV];
            fvn[0] = 0.0;
#pragma unroll
            for (int v = 1; v < NV; v++) fvn[v] = (((double)fto[side][v - 1] + (double)ftn[side][v - 1]) * 0.5) * nr;
            double F[NV];
            if (OPEN && bt[side] != BC_PERIODIC) {
                // boundary point: F_b for the outward normal (k_rhs has the
                // citations); turned back to +e_r for the sum below
                const double ns = side ? nr : -nr;
                double bs[5];
#pragma unroll
                for (int v = 0; v < 5; v++) bs[v] = A.geo.bcs[(2 * r + side) * 5 + v];
                const double lb = boundary_flux<DIM>(bt[side], r, ns, nr, pn, bs, P, quirk3d, F);
                lam = (lam < lb) ? lb : lam;
                double d[NV];
#pragma unroll
                for (int v = 0; v < NV; v++) d[v] = F[v];
                if (A.parabolic && (bt[side] == BC_OUTFLOW || bt[side] == BC_NOSLIP)) {
                    double fn[NV];
#pragma unroll
                    for (int v = 1; v < NV; v++) fn[v] = (double)fto[side][v - 1] * ns;
                    if (bt[side] == BC_NOSLIP) {
                        double en = bs[0] * fn[1];
#pragma unroll
                        for (int dd = 1; dd < DIM; dd++) en = en + bs[dd] * fn[1 + dd];
                        fn[NV - 1] = en + bs[3] * sqrt(ns * ns);
                    }
#pragma unroll
                    for (int v = 1; v < NV; v++) d[v] -= fn[v];
                }
#pragma unroll
                for (int v = 0; v < NV; v++) acc[side ? NP - 1 : 0][v] = iw0 * d[v];
                continue;
            }
            NodeQ<DIM> qo = node(side ? NP - 1 : 0), qn;
            qn = node_quants<DIM>(pn, P);
            if (A.parabolic && A.quirks) {
                // ComputeViscousFlux left velocities in the momentum slots of
                // both states (DGSEMIntegrator.cpp:471-481)
                auto alias = [&](NodeQ<DIM> &q) {
                    const double ri = rcp_nr(q.rho);
                    const double ke = 0.5 * q.rho;
                    double p = 0.5 * q.rho * rcp_nr(q.beta), v0 = 0.0, v1 = 0.0;
#pragma unroll
                    for (int d = 0; d < DIM; d++) {
                        v0 += q.v[d] * q.v[d];
                        q.v[d] *= ri;
                        v1 += q.v[d] * q.v[d];
                    }
                    p += P.gm1 * ke * (v0 - v1);
                    q.beta = 0.5 * q.rho * rcp_nr(p);
                };
                alias(qo);
                alias(qn);
            }
            face_quants<DIM>(qo, P);
            face_quants<DIM>(qn, P);
            const NodeQ<DIM> &q1 = side ? qo : qn;
            const NodeQ<DIM> &q2 = side ? qn : qo;
            if (A.ec) ec_flux<DIM, false>(nvec, nr, q1, q2, P, false, F);
            else ec_flux<DIM, true>(nvec, nr, q1, q2, P, quirk3d, F);
            const double sg = side ? iw0 : -iw0;
#pragma unroll
            for (int v = 0; v < NV; v++) acc[side ? NP - 1 : 0][v] = sg * (A.parabolic ? F[v] - fvn[v] : F[v]);
        }
    }

    // ---- modal indicator and blending coefficient ----
    double alpha_e = 0.0;
    if constexpr (BLEND) {
        // modes = V^-1 (rho p), one direction at a time on that direction's
        // line threads (V^-1 = kron of 1-D inverses); after the last the
        // thread holds its line's modes and sums their squares: e2 over the
        // modes of degree <= N-2 in every direction, e1 over the others of
        // degree <= N-1, e0 over the rest.  The energies of
        // PerssonPeraireIndicator.cpp:38-52 are e2, e2 + e1 and e2 + e1 + e0,
        // and its 1 - m1/m = e0/m and 1 - m2/m1 = e1/m1, here without the
        // cancellation, which alpha's steep logistic magnifies
#pragma unroll
        for (int rr = 0; rr < DIM; rr++) {
            if (lact && r == rr) {
                double q[NP], md[NP];
#pragma unroll
                for (int m = 0; m < NP; m++) q[m] = sX[el][ls[m]];
#pragma unroll
                for (int a = 0; a < NP; a++) {
                    double s = 0.0;
#pragma unroll
                    for (int m = 0; m < NP; m++) s = (m == 0) ? A.tab.V1i[a * MAXNP] * q[0] : fma(A.tab.V1i[a * MAXNP + m], q[m], s);
                    md[a] = s;
                }
                if (rr < DIM - 1) {
#pragma unroll
                    for (int m = 0; m < NP; m++) sX[el][ls[m]] = md[m];
                } else {
                    double lo = 0.0;
#pragma unroll
                    for (int a = 0; a < NP - 2; a++) lo = fma(md[a], md[a], lo);
                    const double mid = md[NP - 2] * md[NP - 2], top = md[NP - 1] * md[NP - 1];
                    const bool in1 = la <= NP - 2 && lb <= NP - 2, in2 = la <= NP - 3 && lb <= NP - 3;
                    sE[el][0][l] = in1 ? top : lo + mid + top;
                    sE[el][1][l] = in2 ? mid : (in1 ? lo + mid : 0.0);
                    sE[el][2][l] = in2 ? lo : 0.0;
                }
            }
            __syncthreads();
        }
        // rows of NP partial sums, then the NP row sums
        if (lact && rem < 3 * NP) {
            const int c = rem / NP, row = rem - c * NP;
            double s = 0.0;
#pragma unroll
            for (int m = 0; m < NP; m++) s += sE[el][c][row * NP + m];
            sX[el][rem] = s;
        }
        __syncthreads();
        if (lact && rem == 0) {
            double m3[3];
#pragma unroll
            for (int c = 0; c < 3; c++) {
                m3[c] = 0.0;
#pragma unroll
                for (int m = 0; m < NP; m++) m3[c] += sX[el][c * NP + m];
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
            sAl[el] = al;
            A.alpha[e] = al;
            A.eta[e] = eta;
        }
        __syncthreads();
        if (lact) alpha_e = sAl[el];
    }

    // ---- volume pairs ----
    // (1 - alpha) goes into the metric vector, in which the fluxes are linear
    if (lact) {
        const double om = BLEND ? 1.0 - alpha_e : 1.0;
        const double nvs[3] = {om * nvec[0], om * nvec[1], om * nvec[2]};
        auto pairs = [&](auto range) {
            constexpr int RANGE = decltype(range)::value;
            const bool zq = QNS3 && r == 2;
#pragma unroll
            for (int a = 0; a < NP; a++) {
                const NodeQ<DIM> qa = node(a);
#pragma unroll
                for (int b = a + 1; b < NP; b++) {
                    // (read node b here: kept from pair to pair, a line's
                    // nodes would need 80 registers more)
                    asm volatile("" ::: "memory");
                    const NodeQ<DIM> qb = node(b);
                    double F[NV];
                    ec_flux<DIM, false, RANGE>(nvs, nr, qa, qb, P, false, F);
                    const double dab = A.tab.Dh2[a * MAXNP + b], dba = A.tab.Dh2[b * MAXNP + a];
#pragma unroll
                    for (int v = 0; v < NV; v++) {
                        acc[a][v] = fma(dab, F[v], acc[a][v]);
                        if (!zq) acc[b][v] = fma(dba, F[v], acc[b][v]);
                        // (not to be moved past the next pair's branches,
                        // which would keep every F)
                        if constexpr (RANGE == LM_ANY) asm volatile("" : "+v"(acc[a][v]), "+v"(acc[b][v]));
                    }
                }
                if (QNS3 && zq && a < NP - 1 && lb < NP - 1) {
                    // zeta partners a < b of node b: the eta flux of node a
                    // with node (i, NP-1, a) of its eta line; 0 on the eta
                    // line's last node (DGSEMIntegrator.cpp:702)
                    const int se = high_slot<NP>(la, NP - 1, a);
                    NodeQ<DIM> qe;
                    qe.rho = sQ[el][0][se];
#pragma unroll
                    for (int d = 0; d < DIM; d++) qe.v[d] = sQ[el][1 + d][se];
                    qe.beta = sQ[el][NV - 1][se];
                    const double n1[3] = {0.0, om * A.geo.nrm[1], 0.0};
                    double g[NV];
                    ec_flux<DIM, false>(n1, A.geo.nrm[1], qa, qe, P, false, g);
#pragma unroll
                    for (int b = a + 1; b < NP; b++)
#pragma unroll
                        for (int v = 0; v < NV; v++) {
                            acc[b][v] = fma(A.tab.Dh2[b * MAXNP + a], g[v], acc[b][v]);
                            asm volatile("" : "+v"(acc[b][v]));
                        }
                }
            }
        };
        if constexpr (QNS3) {
            // one loop: its second flux per node leaves no registers for three
            pairs(std::integral_constant<int, LM_ANY>{});
        } else {
            double rlo = sQ[el][0][ls[0]], rhi = rlo, blo = sQ[el][NV - 1][ls[0]], bhi = blo;
#pragma unroll
            for (int m = 1; m < NP; m++) {
                const double a = sQ[el][0][ls[m]], b = sQ[el][NV - 1][ls[m]];
                rlo = fmin(rlo, a); rhi = fmax(rhi, a);
                blo = fmin(blo, b); bhi = fmax(bhi, b);
            }
            // |y - x| / (y + x) of every pair is at most that of the extremes
            // (positive values; others fail every test and take LM_ANY)
            const double dr = rhi - rlo, rs = rhi + rlo, db = bhi - blo, bs = bhi + blo;
            if ((dr < 0.01 * rs) & (db < 0.01 * bs)) pairs(std::integral_constant<int, LM_SHORT>{});
            else if ((3.0 * dr < rs) & (3.0 * db < bs)) pairs(std::integral_constant<int, LM_MID>{});
            else pairs(std::integral_constant<int, LM_ANY>{});
        }

        if constexpr (BLEND) {
            if (alpha_e > 0.0) {
                // blended element: subcell FV fluxes G along the line, 0 at the
                // element boundary (DGSEMIntegrator.cpp:972-1196)
                NodeQ<DIM> qa = node(0);
                face_quants<DIM>(qa, P);
#pragma unroll
                for (int i = 0; i < NP - 1; i++) {
                    NodeQ<DIM> qb = node(i + 1);
                    face_quants<DIM>(qb, P);
                    const double si = lane_pick3(A.tab.subn[0][i], A.tab.subn[1][i], A.tab.subn[2][i], r);
                    const double ns[3] = {r == 0 ? si : 0.0, r == 1 ? si : 0.0, r == 2 ? si : 0.0};
                    double G[NV];
                    ec_flux<DIM, true>(ns, si, qa, qb, P, quirk3d, G);
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
    __syncthreads();   // the partial sums take the rows' place

    // ---- node sums over the directions, in direction order ----
#pragma unroll
    for (int rr = 0; rr < DIM; rr++) {
        if (lact && r == rr) {
#pragma unroll
            for (int a = 0; a < NP; a++)
#pragma unroll
                for (int v = 0; v < NV; v++) sQ[el][v][ls[a]] = (rr == 0) ? acc[a][v] : sQ[el][v][ls[a]] + acc[a][v];
        }
        __syncthreads();
    }

    // ---- viscous volume term, stage update, store ----
#pragma unroll
    for (int p = 0; p < NPASS; p++) {
        const int i = t + p * BLOCK;
        if (i >= nact) continue;
        const int e2 = EPB == 1 ? 0 : i / K, n = i - e2 * K;
        const int s = high_slot<NP>(n % NP, (n / NP) % NP, n / (NP * NP));
        const size_t gi = (size_t)ebase * K + i;
#pragma unroll
        for (int v = 0; v < NV; v++) {
            double tot = -sQ[e2][v][s];
            if (A.parabolic && v > 0) tot += (double)static_cast<const VT *>(A.visc)[(v - 1) * NK + gi];
            tot *= A.geo.invJ;
            double o = tot;
            if (A.mode != 0) {
                o = fma(dt, tot, A.y[v * NK + gi]);
                if (A.mode == 2) o = fma(A.c1, o, A.c0 * A.u0[v * NK + gi]);
            }
            A.out[v * NK + gi] = o;
        }
    }
    block_lam_max<BLOCK>(lam, lam_old, A.lam, sRed, blockIdx.x);
}

} // namespace prandtl
