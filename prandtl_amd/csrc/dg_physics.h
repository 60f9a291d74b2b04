// Point physics of the DGSEM hot path, device side (gfx950, FP64).
//
// Restates, in the reference's operation order, the two-point fluxes of
// ChandrashekarFlux.cpp:11-161, the log mean of BasicOperations.cpp:6-12, the
// entropy/primitive transforms of BasicOperations.cpp:31-186 and the viscous
// flux of NavierStokesFlux.cpp:12-90.  Normals are axis-aligned on the
// Cartesian meshes this library builds, so a normal is a direction r and a
// positive magnitude; the zero components of the reference's dot products
// are dropped (they add +0 exactly for finite data).
#pragma once
#include <hip/hip_runtime.h>

namespace prandtl {

struct Phys {
    double gamma, gm1, gm1i;
    double mu, lam_h;      // mu and mu*gamma*(1/Pr) (NavierStokesFlux.cpp:38)
    double alpha_max, alpha_min, thresh;
    int sutherland;        // mu(T) per point (NavierStokesFlux.hpp:32-36)
    double R_gas, PrInv;
};

// Viscosity coefficients of one viscous-flux evaluation, in arithmetic R:
// constant mu and lam = mu*gamma*(1/Pr), or Sutherland's law per point.
template <typename R> struct ViscCoef {
    R mu, lam_h;
    bool suth;
    R R_gas, gamma, PrInv;
};

// NavierStokesFlux::ComputeViscosity (NavierStokesFlux.hpp:32-36) with the
// constants of Physics.hpp:35-37; T0pTs = T0 + Ts as in the constructor.
template <typename R>
__device__ __forceinline__ R sutherland_mu(R rho, R p, R R_gas)
{
    const R mu0 = R(1.716e-5), T0 = R(273.15), Ts = R(110.4), T0pTs = R(273.15 + 110.4);
    const R T = p / (rho * R_gas);
    return mu0 * T0pTs / (T + Ts) * (T / T0) * sqrt(T / T0);
}

// Reciprocals: the hardware estimate (v_rcp_f64 / v_rcp_f32) refined by
// Newton-Raphson steps r <- r + r (1 - x r) (two for FP64, one for FP32),
// within an ulp or two of 1/x; the pointwise transforms multiply by them
// where the reference divides.
__device__ __forceinline__ double rcp_nr(double x)
{
    double r = __builtin_amdgcn_rcp(x);
    double e = fma(-x, r, 1.0);
    r = fma(r, e, r);
    e = fma(-x, r, 1.0);
    return fma(r, e, r);
}

__device__ __forceinline__ float rcp_nr(float x)
{
    const float r = __builtin_amdgcn_rcpf(x);
    return fmaf(r, fmaf(-x, r, 1.0f), r);
}

// Per-node quantities shared by every two-point flux touching the node.
template <int DIM> struct NodeQ {
    double rho, v[DIM], beta, ibeta, lam;
};

// rho, v = m/rho, p = (gamma-1)(E - rho|v|^2/2), beta = rho/(2p), 1/beta,
// lam = |v| + sqrt(gamma p/rho)  (ChandrashekarFlux.cpp:17-68).  Reciprocals
// of rho and p replace the reference's divisions.
template <int DIM>
__device__ __forceinline__ NodeQ<DIM> node_quants(const double *s, const Phys &P)
{
    NodeQ<DIM> q;
    q.rho = s[0];
    const double ri = rcp_nr(q.rho);
    double vsq = 0.0;
#pragma unroll
    for (int d = 0; d < DIM; d++) {
        q.v[d] = s[1 + d] * ri;
        vsq = (d == 0) ? q.v[d] * q.v[d] : vsq + q.v[d] * q.v[d];
    }
    const double p = P.gm1 * (s[DIM + 1] - 0.5 * q.rho * vsq);
    q.beta = 0.5 * q.rho * rcp_nr(p);
    q.ibeta = 2.0 * p * ri;
    q.lam = sqrt(vsq) + sqrt(P.gamma * p * ri);
    return q;
}

// The two logarithmic means of a two-point flux (ComputeLogMean,
// BasicOperations.cpp:6-12): rho_ln, 1/beta_ln, and rbs = 1/(beta1 + beta2),
// which the mean pressure needs as well.  With f = (y-x)/(y+x) and u = f^2,
// log(y/x) = 2 atanh(f) = 2 f T(u), so LM = (x+y)/(2 T(u)) and 1/LM =
// 2 T(u)/(x+y): the beta mean costs one reciprocal, shared with the pressure,
// and no logarithm.  Three ranges of u, chosen for both means together:
//   u < 1e-4 (y/x within 2%; the reference's own series range): T and the
//     series of 1/T to u^3 (the next terms are below 1e-17);
//   u < 1/9 (y/x up to 2): T by a degree-10 polynomial, the Chebyshev
//     interpolant of atanh(sqrt u)/sqrt u on [0, 1/9], relative error 2.4e-18;
//   else (shocks, values of two signs or not finite): (y-x)/log(y/x)
//     with log(y/x) = k log 2 + log(y/(2^k x)), k the difference of the binary
//     exponents, which brings the second logarithm into T's range: 45
//     instructions against 130 of the library's logarithm and quotient.
// Largest error against an extended-precision log mean: 2.7e-16, 3.8e-16 and
// 4.3e-16 in the three ranges; the quotient (y-x)/log(y/x) of the reference
// loses up to 5.3e-15 below a ratio of 2, where y/x is rounded.
// Next to a mean by the quotient or by one rational of s and d (four
// divisions or two reciprocals and a logarithm per pair) the fluxes of all
// kernels became faster by: 2-D N = 4 with blending, 64^2 boxes, 38.2 ->
// 28.2 us per RK3 step and 2-D N = 3, 384^2, 172 -> 147 us per right-hand
// side (shear layers, whose logarithms go); 3-D N = 3 Navier-Stokes,
// 45 x 43 x 41, 495 -> 462 us.
__device__ __forceinline__ double atanh_ratio(double u)
{
    double p = 0.08522081781390699;
    p = fma(p, u, 0.0416225325593041);
    p = fma(p, u, 0.06055084364034609);
    p = fma(p, u, 0.06650187016337313);
    p = fma(p, u, 0.07693307021152004);
    p = fma(p, u, 0.09090870416252403);
    p = fma(p, u, 0.11111112040373837);
    p = fma(p, u, 0.14285714272727057);
    p = fma(p, u, 0.20000000000092874);
    p = fma(p, u, 0.33333333333333076);
    return fma(p, u, 1.0);
}

// T or log(y/x) of one mean in the third range's form: T(u), as the second range
// has it, for values of one sign within a ratio of 2, |y - x| < min(|x|, |y|)
// (exact where it decides; negative values, of a state that has lost its
// physics, have a mean while both are negative); otherwise log(y/x), NaN for
// values of different sign, as the logarithm of their quotient is.  log 2 in two
// parts: the double with its last 21 bits cut off, so that k times it is exact,
// and the double nearest the rest.
__device__ __forceinline__ bool log_parts(double x, double y, double &TL)
{
    const double d = fabs(y - x);
    const bool in = (d < fabs(x)) & (d < fabs(y));
    const int k = in ? 0 : __builtin_amdgcn_frexp_exp(y) - __builtin_amdgcn_frexp_exp(x);
    const double xk = ldexp(x, k);
    const double f = (y - xk) * rcp_nr(xk + y);
    const double T = atanh_ratio(f * f);
    const double kd = (double)k, f2 = f + f;
    const double lg = fma(kd, 0.6931471803691238, f2 + fma(f2, T - 1.0, kd * 1.9082149292705877e-10));
    TL = in ? T : (x < 0.0) != (y < 0.0) ? __builtin_nan("") : lg;
    return in;
}

// RANGE: LM_SHORT is the first range alone, for callers that have bounded the
// ratio of a whole line's values; LM_MID the second (and valid in the first);
// LM_ANY every value, by the second range's formulas where they hold.  Where
// both hold MID and ANY agree bitwise, so a wave may take ANY for all its
// lanes as soon as one of them needs it (ec_flux below) without a lane's
// result depending on the others.
enum { LM_SHORT = 0, LM_MID = 1, LM_ANY = 2, LM_PAIR = 3 };

template <int RANGE>
__device__ __forceinline__ void log_means(double ra, double rb, double ba, double bb, double &rho_ln,
                                          double &ibeta_ln, double &rbs)
{
    const double rs = ra + rb, bs = ba + bb;
    const double dr = rb - ra, db = bb - ba;
    rbs = rcp_nr(bs);
    if constexpr (RANGE == LM_ANY) {
        double TL;
        bool in = log_parts(ra, rb, TL);
        rho_ln = (in ? 0.5 * rs : dr) * rcp_nr(TL);
        in = log_parts(ba, bb, TL);
        ibeta_ln = (2.0 * rcp_nr(in ? bs : db)) * (in ? TL : 0.5 * TL);
    } else {
        const double fr = dr * rcp_nr(rs), fb = db * rbs;
        const double ur = fr * fr, ub = fb * fb;
        if constexpr (RANGE == LM_SHORT) {
            // T = 1 + u/3 + u^2/5 + u^3/7, 1/T = 1 - u/3 - 4u^2/45 - 44u^3/945
            const double tr = fma(ur, fma(ur, fma(ur, -22.0 / 945.0, -2.0 / 45.0), -1.0 / 6.0), 0.5);
            const double tb = fma(ub, fma(ub, fma(ub, 2.0 / 7.0, 2.0 / 5.0), 2.0 / 3.0), 2.0);
            rho_ln = rs * tr;
            ibeta_ln = rbs * tb;
        } else {
            rho_ln = (0.5 * rs) * rcp_nr(atanh_ratio(ur));
            ibeta_ln = (2.0 * rbs) * atanh_ratio(ub);
        }
    }
}

// Whether the second range's formulas do not hold for the pair, or its values
// are not positive.
__device__ __forceinline__ bool lm_outside(double x, double y) { return !((y < x + x) & (x < y + y)); }

// Chandrashekar two-point flux for the normal (or mean metric) vector n.
// DISS = false: ComputeVolumeFlux (ChandrashekarFlux.cpp:11-83).  DISS =
// true: ComputeFaceFlux (lines 85-161), the dissipation scaled by nd = |n|
// (line 88); quirk3d keeps the 3-D energy dissipation term of line 131 as
// written.  Written with few operations (the kernels are bound by FP64
// issue and latency):
//  - v_mean^2 - mean(v^2)/2 = v1 v2 / 2 per component;
//  - the energy flux rho_ln Vn (h + p_hat/rho_ln) is rho_ln Vn h + Vn p_hat;
//  - the momentum jump is rho_mean dv + drho v_mean, and the energy jump
//    reuses drho h, so the conserved states are not read.
// Symmetric in (a, b) for DISS = false, as the symmetric pairs need.
template <int DIM, bool DISS, int RANGE>
__device__ __forceinline__ void ec_flux_r(const double *n, double nd, const NodeQ<DIM> &a, const NodeQ<DIM> &b,
                                        const Phys &P, bool quirk3d, double *F)
{
    double rho_ln, ibeta_ln, rbs;
    log_means<RANGE>(a.rho, b.rho, a.beta, b.beta, rho_ln, ibeta_ln, rbs);
    double vs[DIM];
    double h2 = 0.0, w = 0.0;
#pragma unroll
    for (int d = 0; d < DIM; d++) {
        vs[d] = a.v[d] + b.v[d];
        h2 = (d == 0) ? a.v[d] * b.v[d] : fma(a.v[d], b.v[d], h2);
        w = (d == 0) ? vs[d] * n[d] : fma(vs[d], n[d], w);
    }
    const double rm = 0.5 * (a.rho + b.rho);
    const double p_hat = rm * rbs;
    const double h = 0.5 * fma(P.gm1i, ibeta_ln, h2);
    const double Vn = 0.5 * w;
    const double rV = rho_ln * Vn;
    const double rVh = 0.5 * rV;
    F[0] = rV;
#pragma unroll
    for (int d = 0; d < DIM; d++) F[1 + d] = fma(p_hat, n[d], rVh * vs[d]);
    F[DIM + 1] = fma(Vn, p_hat, rV * h);
    if (DISS) {
        const double drho = b.rho - a.rho;
        const double lam = (a.lam < b.lam) ? b.lam : a.lam;
        const double hl = 0.5 * lam * nd;
        const double hdr = 0.5 * drho;
        double e = P.gm1i * (b.ibeta - a.ibeta);   // sum of dv (v1 + v2) and the internal energy's jump
        double q3 = 0.0;
        F[0] = fma(-hl, drho, F[0]);
#pragma unroll
        for (int d = 0; d < DIM; d++) {
            const double dv = b.v[d] - a.v[d];
            F[1 + d] = fma(-hl, fma(rm, dv, hdr * vs[d]), F[1 + d]);
            if (DIM == 3 && d == 2 && quirk3d) q3 = fma(rm, dv, 0.5 * vs[d]);
            else e = fma(dv, vs[d], e);
        }
        F[DIM + 1] = fma(-hl, fma(drho, h, fma(0.5 * rm, e, q3)), F[DIM + 1]);
    }
}

// ec_flux_r with the range of the wave's active lanes: MID unless a lane is
// outside it.  TRY_SHORT: lanes in the first range take it (worth the second
// path where most waves hold such lanes only: the face points of 3-D flows).
template <int DIM, bool DISS, bool TRY_SHORT = false>
__device__ __forceinline__ void ec_flux(const double *n, double nd, const NodeQ<DIM> &a, const NodeQ<DIM> &b,
                                        const Phys &P, bool quirk3d, double *F)
{
    if (TRY_SHORT && ((fabs(b.rho - a.rho) < 0.01 * (a.rho + b.rho)) & (fabs(b.beta - a.beta) < 0.01 * (a.beta + b.beta))))
        ec_flux_r<DIM, DISS, LM_SHORT>(n, nd, a, b, P, quirk3d, F);
    else if (__any(lm_outside(a.rho, b.rho) | lm_outside(a.beta, b.beta)))
        ec_flux_r<DIM, DISS, LM_ANY>(n, nd, a, b, P, quirk3d, F);
    else ec_flux_r<DIM, DISS, LM_MID>(n, nd, a, b, P, quirk3d, F);
}

// MFEM Vector::Norml2 of a 2-vector (scaled, overflow-safe), the face
// normal's magnitude in ChandrashekarFlux::ComputeFaceFlux (line 88).
__device__ __forceinline__ double norml2_2(const double *n)
{
    double scale = 0.0, sum = 0.0;
#pragma unroll
    for (int i = 0; i < 2; i++) {
        if (n[i] != 0.0) {
            const double a = fabs(n[i]);
            if (scale <= a) {
                const double q = scale / a;
                sum = 1.0 + sum * (q * q);
                scale = a;
            } else {
                const double q = a / scale;
                sum += q * q;
            }
        }
    }
    return scale * sqrt(sum);
}

// MFEM Vector::Norml2 of a 3-vector (the same scaled sum).
__device__ __forceinline__ double norml2_3(const double *n)
{
    double scale = 0.0, sum = 0.0;
#pragma unroll
    for (int i = 0; i < 3; i++) {
        if (n[i] != 0.0) {
            const double a = fabs(n[i]);
            if (scale <= a) {
                const double q = scale / a;
                sum = 1.0 + sum * (q * q);
                scale = a;
            } else {
                const double q = a / scale;
                sum += q * q;
            }
        }
    }
    return scale * sqrt(sum);
}

// |n| of a mesh's face or subcell normal: the squares of the components times sc,
// a power of two that brings the mesh's largest normal near 1 (isc = 1/sc), so
// that they neither under- nor overflow (normals of 3-D meshes are squares of
// lengths).  The scaling is exact: the result is that of the plain sum where
// that is in range.
template <int DIM>
__device__ __forceinline__ double normal_length(const double *n, double sc, double isc)
{
    double s = 0.0;
#pragma unroll
    for (int d = 0; d < DIM; d++) {
        const double x = n[d] * sc;
        s = (d == 0) ? x * x : fma(x, x, s);
    }
    return sqrt(s) * isc;
}

// Boundary types (PRANDTL_BC_*)
enum { BC_PERIODIC = 0, BC_SLIP = 1, BC_INFLOW = 2, BC_OUTFLOW = 3, BC_SYMMETRY = 4, BC_SPECIFIED = 5,
       BC_NOSLIP = 6 };

// SlipWallBdrFaceIntegrator::ComputeBdrFaceInviscidFlux
// (SlipWallBdrFaceIntegrator.cpp:15-60) for the outward normal ns e_r.  The
// unit normal is ns * (1/|ns|) (Normalize, BasicOperations.hpp:39-42);
// RotateState (BasicOperations.cpp:238-259) of an axis-aligned normal
// reduces to the component permutations below: its tangents Normal(n) and
// n x Normal(n) have unit entries, whose products are exact.  p* is the
// wall pressure of the shock (u_n > 0) or rarefaction (u_n <= 0, base
// clipped at 1e-4) branch; F = (0, p* ns e_r, 0).  Returns the face-frame
// |v| + a.
template <int DIM>
__device__ __forceinline__ double slip_wall_flux(int r, double ns, const double *s, const Phys &P,
                                                 double *F)
{
    const double u = ns * (1.0 / fabs(ns));
    double m[DIM];
    // 1-D: state2(1) * nor(0) (SlipWallBdrFaceIntegrator.cpp:22-30)
    if constexpr (DIM == 1) m[0] = s[1] * ns;
    if constexpr (DIM == 2) {
        const double s1 = s[1], s2 = s[2];
        m[0] = (r == 0 ? s1 : s2) * u;
        m[1] = r == 0 ? s2 * u : -(s1 * u);
    }
    if constexpr (DIM == 3) {
        // selects, not branches: r differs between the lanes of a wave, and
        // the compiler (ROCm 7.2), sinking the -s[1] that the branches for
        // r = 1 and r = 2 share, left m[1] unset in the lanes with r = 2.
        // Between values already loaded: a choice of elements of s would put
        // the caller's state into scratch memory
        const double s1 = s[1], s2 = s[2], s3 = s[3];
        m[0] = (r == 0 ? s1 : r == 1 ? s2 : s3) * u;
        m[1] = r == 0 ? s2 : -s1;
        m[2] = r == 2 ? -(s2 * u) : s3 * u;
    }
    // Conserv2Prim (BasicOperations.cpp:172-186): velocities by division,
    // the pressure's by the reciprocal (ComputePressure, lines 31-37)
    const double rho = s[0];
    const double ri = 1.0 / rho;
    double vel[DIM], vv = 0.0, VV = 0.0;
#pragma unroll
    for (int d = 0; d < DIM; d++) {
        vel[d] = m[d] / rho;
        const double V = m[d] * ri;
        VV = (d == 0) ? V * V : VV + V * V;
        vv = (d == 0) ? vel[d] * vel[d] : vv + vel[d] * vel[d];
    }
    const double p = P.gm1 * (s[DIM + 1] - 0.5 * rho * VV);
    const double an = sqrt(P.gamma * p / rho);
    const double un = vel[0];
    const double gp1 = 1.0 + P.gamma, gp1i = 1.0 / gp1;
    double p_star;
    if (un > 0.0)
        p_star = p + 0.25 * un * gp1 * rho * (un + sqrt(un * un + 8.0 * gp1i / rho * p * (P.gm1 * gp1i + 1.0)));
    else {
        double base = 1.0 + 0.5 * P.gm1 * un / an;
        base = (base < 0.0001) ? 0.0001 : base;
        p_star = p * pow(base, 2.0 * P.gamma * P.gm1i);
    }
#pragma unroll
    for (int v = 0; v < DIM + 2; v++) F[v] = 0.0;
#pragma unroll
    for (int d = 0; d < DIM; d++)
        if (d == r) F[1 + d] = p_star * ns;
    return sqrt(vv) + an;
}

// slip_wall_flux for a general 2-D outward normal n: Normalize, then
// RotateState with Normal(n) = (-n1, n0) (BasicOperations.cpp:211-259).
__device__ __forceinline__ double slip_wall_flux_v2(const double *n, const double *s, const Phys &P, double *F)
{
    const double inv = 1.0 / norml2_2(n);
    const double u0 = n[0] * inv, u1 = n[1] * inv;
    const double m[2] = {s[1] * u0 + s[2] * u1, s[1] * -u1 + s[2] * u0};
    const double rho = s[0];
    const double ri = 1.0 / rho;
    double vel[2], vv = 0.0, VV = 0.0;
#pragma unroll
    for (int d = 0; d < 2; d++) {
        vel[d] = m[d] / rho;
        const double V = m[d] * ri;
        VV = (d == 0) ? V * V : VV + V * V;
        vv = (d == 0) ? vel[d] * vel[d] : vv + vel[d] * vel[d];
    }
    const double p = P.gm1 * (s[3] - 0.5 * rho * VV);
    const double an = sqrt(P.gamma * p / rho);
    const double un = vel[0];
    const double gp1 = 1.0 + P.gamma, gp1i = 1.0 / gp1;
    double p_star;
    if (un > 0.0)
        p_star = p + 0.25 * un * gp1 * rho * (un + sqrt(un * un + 8.0 * gp1i / rho * p * (P.gm1 * gp1i + 1.0)));
    else {
        double base = 1.0 + 0.5 * P.gm1 * un / an;
        base = (base < 0.0001) ? 0.0001 : base;
        p_star = p * pow(base, 2.0 * P.gamma * P.gm1i);
    }
    F[0] = 0.0;
    F[1] = p_star * n[0];
    F[2] = p_star * n[1];
    F[3] = 0.0;
    return sqrt(vv) + an;
}

// boundary_flux for a general 2-D outward normal n (general quadrilateral
// meshes); symmetry mirrors m - 2 (m.u) u with the unit normal u.
__device__ __forceinline__ double boundary_flux_v2(int type, const double *n, const double *s, const double *outer,
                                                   const Phys &P, double *F)
{
    if (type == BC_SLIP || type == BC_NOSLIP) return slip_wall_flux_v2(n, s, P, F);
    const double nd = norml2_2(n);
    double g[4];
#pragma unroll
    for (int v = 0; v < 4; v++) g[v] = (type == BC_INFLOW || type == BC_SPECIFIED) ? outer[v] : s[v];
    if (type == BC_SYMMETRY) {
        const double inv = 1.0 / nd;
        const double u0 = n[0] * inv, u1 = n[1] * inv;
        const double mn = s[1] * u0 + s[2] * u1;
        g[1] = s[1] + -2.0 * mn * u0;
        g[2] = s[2] + -2.0 * mn * u1;
    }
    const NodeQ<2> q1 = node_quants<2>(s, P);
    const NodeQ<2> q2 = node_quants<2>(g, P);
    ec_flux<2, true>(n, nd, q1, q2, P, false, F);
    return (q1.lam < q2.lam) ? q2.lam : q1.lam;
}

// slip_wall_flux for a general 3-D outward normal n.  RotateState with the
// unit normal u and its two tangents (BasicOperations.cpp:211-259) gives the
// normal momentum m.u; the tangential ones enter only |v|, which the
// rotation keeps, so |m| is used directly.
__device__ __forceinline__ double slip_wall_flux_v3(const double *n, const double *s, const Phys &P, double *F)
{
    const double inv = 1.0 / norml2_3(n);
    const double u0 = n[0] * inv, u1 = n[1] * inv, u2 = n[2] * inv;
    const double mn = s[1] * u0 + s[2] * u1 + s[3] * u2;
    const double rho = s[0];
    const double ri = 1.0 / rho;
    const double mm = s[1] * s[1] + s[2] * s[2] + s[3] * s[3];
    const double vv = mm / (rho * rho);
    const double VV = mm * (ri * ri);
    const double p = P.gm1 * (s[4] - 0.5 * rho * VV);
    const double an = sqrt(P.gamma * p / rho);
    const double un = mn / rho;
    const double gp1 = 1.0 + P.gamma, gp1i = 1.0 / gp1;
    double p_star;
    if (un > 0.0)
        p_star = p + 0.25 * un * gp1 * rho * (un + sqrt(un * un + 8.0 * gp1i / rho * p * (P.gm1 * gp1i + 1.0)));
    else {
        double base = 1.0 + 0.5 * P.gm1 * un / an;
        base = (base < 0.0001) ? 0.0001 : base;
        p_star = p * pow(base, 2.0 * P.gamma * P.gm1i);
    }
    F[0] = 0.0;
    F[1] = p_star * n[0];
    F[2] = p_star * n[1];
    F[3] = p_star * n[2];
    F[4] = 0.0;
    return sqrt(vv) + an;
}

// boundary_flux for a general 3-D outward normal n (hexahedral meshes).
__device__ __forceinline__ double boundary_flux_v3(int type, const double *n, const double *s, const double *outer,
                                                   const Phys &P, bool quirk3d, double *F)
{
    if (type == BC_SLIP || type == BC_NOSLIP) return slip_wall_flux_v3(n, s, P, F);
    const double nd = norml2_3(n);
    double g[5];
#pragma unroll
    for (int v = 0; v < 5; v++) g[v] = (type == BC_INFLOW || type == BC_SPECIFIED) ? outer[v] : s[v];
    if (type == BC_SYMMETRY) {
        const double inv = 1.0 / nd;
        const double u[3] = {n[0] * inv, n[1] * inv, n[2] * inv};
        const double mn = s[1] * u[0] + s[2] * u[1] + s[3] * u[2];
#pragma unroll
        for (int d = 0; d < 3; d++) g[1 + d] = s[1 + d] + -2.0 * mn * u[d];
    }
    const NodeQ<3> q1 = node_quants<3>(s, P);
    const NodeQ<3> q2 = node_quants<3>(g, P);
    ec_flux<3, true>(n, nd, q1, q2, P, quirk3d, F);
    return (q1.lam < q2.lam) ? q2.lam : q1.lam;
}

template <int DIM>
__device__ __forceinline__ double boundary_flux_vn(int type, const double *n, const double *s, const double *outer,
                                                   const Phys &P, bool quirk3d, double *F)
{
    if constexpr (DIM == 2) return boundary_flux_v2(type, n, s, outer, P, F);
    else return boundary_flux_v3(type, n, s, outer, P, quirk3d, F);
}

// ComputeBdrFaceInviscidFlux of a boundary point (BdrFaceIntegrator.cpp:
// 252-258): the outer state of ComputeOuterInviscidState and the face flux
// with state1 = interior s, normal ns e_r (ns signed outward, nd = |ns|).
// Symmetry (SymmetryBdrFaceIntegrator.cpp) mirrors the normal momentum with
// the unit normal u: m_r - 2 (m_r u) u.  Slip walls replace the flux.
// Returns the point's wave speed.
template <int DIM>
__device__ __forceinline__ double boundary_flux(int type, int r, double ns, double nd, const double *s,
                                                const double *outer, const Phys &P, bool quirk3d,
                                                double *F)
{
    // no-slip walls inherit the slip wall's inviscid flux
    if (type == BC_SLIP || type == BC_NOSLIP) return slip_wall_flux<DIM>(r, ns, s, P, F);
    double g[DIM + 2];
#pragma unroll
    for (int v = 0; v < DIM + 2; v++) g[v] = (type == BC_INFLOW || type == BC_SPECIFIED) ? outer[v] : s[v];
    if (type == BC_SYMMETRY) {
        const double u = ns * (1.0 / nd);
#pragma unroll
        for (int d = 0; d < DIM; d++)
            if (d == r) {
                const double mn = s[1 + d] * u;
                g[1 + d] = s[1 + d] + -2.0 * mn * u;
            }
    }
    const NodeQ<DIM> q1 = node_quants<DIM>(s, P);
    const NodeQ<DIM> q2 = node_quants<DIM>(g, P);
    double n[DIM];
#pragma unroll
    for (int d = 0; d < DIM; d++) n[d] = (d == r) ? ns : 0.0;
    ec_flux<DIM, true>(n, nd, q1, q2, P, quirk3d, F);
    return (q1.lam < q2.lam) ? q2.lam : q1.lam;
}

// Conserv2Entropy, BasicOperations.cpp:81-104 (beta = rho/p); FIRST = false:
// all but w[0], which alone needs logarithms
template <int DIM, bool FIRST = true>
__device__ __forceinline__ void cons2entropy(const double *s, const Phys &P, double *w)
{
    const double r = rcp_nr(s[0]);
    double vel[DIM], vv = 0.0;
#pragma unroll
    for (int d = 0; d < DIM; d++) {
        vel[d] = s[1 + d] * r;
        vv = (d == 0) ? vel[d] * vel[d] : vv + vel[d] * vel[d];
    }
    const double v_sq = 0.5 * vv;
    const double p = P.gm1 * (s[DIM + 1] - s[0] * v_sq);
    const double beta = s[0] * rcp_nr(p);
    // log(p rho^-gamma) as log p - gamma log rho: two logs instead of a log
    // and a pow (rounding-level difference)
    if constexpr (FIRST) {
        const double sent = log(p) - P.gamma * log(s[0]);
        w[0] = (P.gamma - sent) * P.gm1i - beta * v_sq;
    }
#pragma unroll
    for (int d = 0; d < DIM; d++) w[1 + d] = beta * vel[d];
    w[DIM + 1] = -beta;
}

// ComputeBdrFaceLiftingFlux of a boundary point for the interior entropy
// variables w.  No-slip wall (NoSlipAdiabWallBdrFaceIntegrator.cpp): the
// wall's (w0, beta V, -beta) minus w, beta = -w_last, V = outer[0..DIM-1].
// Base (BdrFaceIntegrator.cpp:276-282): Entropy2Conserv (BasicOperations.cpp:
// 106-122) of w, the outer state (the state itself for outflow, outer for
// inflow / specified state), Conserv2Entropy, minus w, halved.  quirks:
// Entropy2Conserv's in-place `vel /= beta` leaves velocities in w's momentum
// slots, and those are what is subtracted.
template <int DIM>
__device__ __forceinline__ void lift_flux(int type, const double *w, const double *outer, const Phys &P,
                                          bool quirks, double *f)
{
    constexpr int NV = DIM + 2;
    if (type == BC_NOSLIP) {
        const double v = -w[NV - 1];
        f[0] = w[0] - w[0];
#pragma unroll
        for (int d = 0; d < DIM; d++) f[1 + d] = outer[d] * v - w[1 + d];
        f[NV - 1] = -v - w[NV - 1];
        return;
    }
    double wi[NV], cs[NV], g[NV];
#pragma unroll
    for (int k = 0; k < NV; k++) wi[k] = w[k];
    const double beta = -wi[NV - 1];
    const double ib = 1.0 / beta;
    double vv = 0.0;
#pragma unroll
    for (int d = 0; d < DIM; d++) {
        wi[1 + d] = wi[1 + d] * ib;
        vv = (d == 0) ? wi[1] * wi[1] : vv + wi[1 + d] * wi[1 + d];
    }
    const double sent = P.gamma - (wi[0] + 0.5 * beta * vv) * P.gm1;
    cs[0] = pow(exp(-sent) / beta, P.gm1i);
#pragma unroll
    for (int d = 0; d < DIM; d++) cs[1 + d] = cs[0] * wi[1 + d];
    cs[NV - 1] = cs[0] * (1.0 / beta * P.gm1i + 0.5 * vv);
    double gs[NV];
#pragma unroll
    for (int k = 0; k < NV; k++) gs[k] = (type == BC_OUTFLOW) ? cs[k] : outer[k];
    cons2entropy<DIM>(gs, P, g);
#pragma unroll
    for (int k = 0; k < NV; k++) f[k] = (g[k] - (quirks ? wi[k] : w[k])) * 0.5;
}

// EntropyGrad2PrimGrad, BasicOperations.cpp:126-170, one direction in place,
// in arithmetic R (double, or float in the mixed form).  quirks: the density
// term multiplies velocities (the aliased row, lines 137-138 and 164)
// instead of momenta.
template <int DIM, typename R>
__device__ __forceinline__ void entgrad2primgrad(const R *s, R gm1, R gm1i, bool quirks, R *g)
{
    const R half = 0.5;
    const R r = rcp_nr(s[0]);
    R vel[DIM], vv = 0;
#pragma unroll
    for (int d = 0; d < DIM; d++) {
        vel[d] = s[1 + d] * r;
        vv = (d == 0) ? vel[d] * vel[d] : vv + vel[d] * vel[d];
    }
    const R v_sq = half * vv;
    const R p = gm1 * (s[DIM + 1] - s[0] * v_sq);
    const R KE = v_sq * s[0];
    const R pr = p * r, rp = s[0] * rcp_nr(p);   // p/rho, rho/p
    const R g0 = g[0], gL = g[DIM + 1];
    R mdot = 0;
#pragma unroll
    for (int d = 0; d < DIM; d++) {
        g[1 + d] = pr * (g[1 + d] + vel[d] * gL);
        const R md = quirks ? vel[d] : s[1 + d];
        mdot = (d == 0) ? md * g[1 + d] : mdot + md * g[1 + d];
    }
    g[0] = s[0] * g0 - gL * (KE - p * gm1i) + rp * mdot;
    g[DIM + 1] = pr * (g[0] + p * gL);
}

// EntropyGrad2PrimGrad in corrected mode, as far as viscous_flux with the same
// state needs it: grad v = T (grad(beta v) - v grad beta) and, in the place of
// the pressure's, rho grad T = rho T^2 grad(-beta) with a density gradient of
// zero: the density gradient, which the first entropy variable's is for,
// drops out of the heat flux.
template <int DIM, typename R>
__device__ __forceinline__ void entgrad2velgrad(const R *s, R gm1, R *g)
{
    const R half = 0.5;
    const R r = rcp_nr(s[0]);
    R vel[DIM], vv = 0;
#pragma unroll
    for (int d = 0; d < DIM; d++) {
        vel[d] = s[1 + d] * r;
        vv = (d == 0) ? vel[d] * vel[d] : vv + vel[d] * vel[d];
    }
    const R p = gm1 * (s[DIM + 1] - s[0] * (half * vv));
    const R T = p * r, gL = g[DIM + 1];
#pragma unroll
    for (int d = 0; d < DIM; d++) g[1 + d] = T * (g[1 + d] + vel[d] * gL);
    g[0] = 0;
    g[DIM + 1] = p * T * gL;
}

// NavierStokesFlux::ComputeViscousFlux (NavierStokesFlux.cpp:12-90), mu_bulk =
// 2/3, in arithmetic R; constant mu or Sutherland's law (ViscCoef).  dq[c][v] = d(prim_v)/dx_c; out
// fl[v][c], v = 1..nv-1 (the mass row is zero and not stored: fl[v-1][c]).
template <int DIM, typename R>
__device__ __forceinline__ void viscous_flux(const R *s, const R (*dq)[DIM + 2], R gm1, R gm1i,
                                             const ViscCoef<R> &vc, R (*fl)[DIM])
{
    constexpr int NV = DIM + 2;
    const R mu_bulk = R(2) / R(3), two = 2, half = 0.5;
    const R rho = s[0];
    const R rr = rcp_nr(rho);
    R vel[DIM];
#pragma unroll
    for (int d = 0; d < DIM; d++) vel[d] = s[1 + d] * rr;
    R vv = 0;
#pragma unroll
    for (int d = 0; d < DIM; d++) vv = (d == 0) ? vel[d] * vel[d] : vv + vel[d] * vel[d];
    const R p = gm1 * (s[NV - 1] - half * rho * vv);
    R mu = vc.mu, lam_h = vc.lam_h;
    if (vc.suth) {
        // SUTHERLAND build: mu from Conserv2Prim's rho and p, lambda = mu*gamma*(1/Pr)
        mu = sutherland_mu<R>(rho, p, vc.R_gas);
        lam_h = mu * vc.gamma * vc.PrInv;
    }
    R div = dq[0][1];
#pragma unroll
    for (int d = 1; d < DIM; d++) div += dq[d][1 + d];
    const R gr = gm1i * rr, pr = p * rr;
#pragma unroll
    for (int c = 0; c < DIM; c++) {
        const R cvdT = gr * (dq[c][NV - 1] - pr * dq[c][0]);
#pragma unroll
        for (int a = 0; a < DIM; a++) {
            R t;
            if (a == c) t = mu * (two * dq[a][1 + a] - mu_bulk * div);
            else t = mu * (dq[c][1 + a] + dq[a][1 + c]);
            fl[a][c] = t;
        }
        R e = vel[0] * fl[0][c];
#pragma unroll
        for (int a = 1; a < DIM; a++) e = e + vel[a] * fl[a][c];
        fl[NV - 2][c] = e + lam_h * cvdT;
    }
}

} // namespace prandtl
