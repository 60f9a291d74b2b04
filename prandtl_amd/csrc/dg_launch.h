// Host-side launch templates of the viscous and RHS kernels and the context they read.
// Each (dimension, order) pair is instantiated in its own translation unit
// (inst_*.hip, listed by PRANDTL_ORDERS) so the library builds in parallel.
#pragma once
#include <string>
#include <vector>
#include "dg_device.h"
#include "dg_points.h"
#include "dg_visc_lines.h"

using namespace prandtl;

struct prandtl_ctx {
    int dim, order, Np, K, NE, nv, Nfp;
    prandtl_mesh_desc mesh;
    prandtl_params prm;
    Tables tab;
    EvenOdd eD;
    Geo geo;
    Phys phys;
    double *d_visc = nullptr, *d_fvf = nullptr, *d_alpha = nullptr, *d_eta = nullptr;
    double *d_ya = nullptr, *d_yb = nullptr;
    double *d_lam = nullptr;       // per-block running maxima (NE slots)
    double *d_lam_out = nullptr;
    int *d_flag = nullptr;
    std::string err;
    // kernel timing (prandtl_profile_begin/end): events bracketing every launch
    bool prof = false;
    std::vector<hipEvent_t> ev_pool;
    std::vector<int> ev_kind;   // 0: RHS kernel, 1: viscous kernel
    size_t ev_used = 0;
    // SSP-RK3 step captured as a hipGraph (dt read from d_dt), replayed per step
    bool use_graph = true;
    double *d_dt = nullptr;
    double *d_bcs = nullptr;       // [3][2][5] outer boundary states (open boxes only)
    void *d_geo = nullptr;         // general quadrilateral geometry tables
    bool gen = false;              // quadrilateral or hexahedral mesh (general-geometry kernels)
    bool axi = false;              // axisymmetric (state r U)
    double *d_axU = nullptr;       // [nv][NE][K] the state recovered from r U (checks, output)
    double hmin = 0.0;             // smallest element size (the dt policy's h_min)
    hipGraph_t graph = nullptr;
    hipGraphExec_t graph_exec = nullptr;
    const double *graph_u = nullptr;
    hipStream_t graph_stream = nullptr;
    const double *dtp = nullptr;  // set while launching stages for a graph
    // time (TimeDependentOperator::t): host mirror, device copy, the device
    // time a stage reads (the loop's while prandtl_run launches) and the
    // stage's offset factor (0, 1, 1/2 of dt in an RK3 step)
    double t = 0.0;
    double *d_time = nullptr;
    uint64_t geom_fp = 0;   // geometry fingerprint kept in checkpoints
    const double *tp = nullptr;
    double stage_tc = 0.0;
    double *d_bfn = nullptr;       // split outer states per attribute (quadrilateral meshes)
    int nattr = 0;
    double graph_dt = 0.0;        // value last copied to d_dt
    bool graph_dt_set = false;
    int rhs_algo = 0;             // PRANDTL_ALGO_TILE or _LINE (line_ok)
    int rhs_shape = 0;            // RHS launch shape (only shapes rhs_shape_ok accepts are set)
    int visc_shape = 0;           // k_visc / k_visc_l launch shape (visc_shape_ok)
    // device time loop (prandtl_run)
    LoopState *d_loop = nullptr;
    LoopState *h_loop = nullptr;            // pinned, two snapshots
    hipEvent_t loop_ev[2] = {nullptr, nullptr};
    const int *skip = nullptr;    // set while launching the loop's stages
};

namespace prandtl {

// message of the last failed create (no context to hold it)
inline std::string g_create_err;

inline int fail(prandtl_ctx *c, int code, const std::string &msg)
{
    if (c) c->err = msg;
    else g_create_err = msg;
    return code;
}

inline int hip_check(prandtl_ctx *c, hipError_t e, const char *what)
{
    if (e == hipSuccess) return PRANDTL_OK;
    return fail(c, PRANDTL_ERR_HIP, std::string(what) + ": " + hipGetErrorString(e));
}

// Event pair around one launch when profiling is on (start before, stop after).
struct ProfScope {
    prandtl_ctx *c;
    hipStream_t s;
    size_t i;
    ProfScope(prandtl_ctx *cc, hipStream_t ss, int kind) : c(cc), s(ss), i(0)
    {
        if (!c->prof) return;
        i = c->ev_used;
        while (c->ev_pool.size() < i + 2) {
            hipEvent_t e;
            if (hipEventCreate(&e) != hipSuccess) { c->prof = false; return; }
            c->ev_pool.push_back(e);
        }
        c->ev_kind.resize((i + 2) / 2);
        c->ev_kind[i / 2] = kind;
        c->ev_used = i + 2;
        (void)hipEventRecord(c->ev_pool[i], s);
    }
    ~ProfScope()
    {
        if (c->prof && c->ev_used >= i + 2) (void)hipEventRecord(c->ev_pool[i + 1], s);
    }
};

// k_visc in one launch shape (boxes in faithful mode, FP64).
template <int DIM, int NP, int FB> void launch_visc_fb(prandtl_ctx *c, const VArgs &a, hipStream_t s)
{
    using Cf = VCfg<DIM, NP, FB>;
    const int nb = (c->NE + Cf::EPB - 1) / Cf::EPB;
    hipLaunchKernelGGL((k_visc<DIM, NP, false, FB>), dim3(nb), dim3(Cf::BLOCK), 0, s, a);
}

// k_visc_l in one launch shape.
template <int DIM, int NP, int FB, bool OPEN> void launch_visc_l(prandtl_ctx *c, const VArgs &a, hipStream_t s)
{
    using Cf = VlCfg<DIM, NP, FB>;
    const int nb = (c->NE + Cf::EPB - 1) / Cf::EPB;
    if (c->prm.precision == PRANDTL_MIXED)
        hipLaunchKernelGGL((k_visc_l<DIM, NP, true, FB, OPEN>), dim3(nb), dim3(Cf::BLOCK), 0, s, a);
    else hipLaunchKernelGGL((k_visc_l<DIM, NP, false, FB, OPEN>), dim3(nb), dim3(Cf::BLOCK), 0, s, a);
}

// A smaller workgroup for meshes too small for the natural one: with fewer
// natural workgroups than CUs (256), one or two elements per workgroup spread
// over more of them.  Euler right-hand sides, natural against this: 3-D N = 3
// 512 elements 9.3 -> 8.0 us (2,197 elements 15.7 against 14.0, 4,096 18.6
// against 18.7), N = 4 252 elements 10.8 -> 8.9, N = 2 125 elements 10.7 -> 8.5.
// At N = 2, whose natural workgroup holds 7 elements, a single wave of 2 is
// better up to 13,824 elements: 4,096 RHS 11.5 -> 9.8, k_visc_l 9.5 -> 8.3; right-
// hand sides at 13,800 Euler 21.4 -> 21.1, blended 32.4 -> 31.3, mixed 36.0 -> 35.5,
// hexahedra 29.5 and 29.6; at 17,550 25.4 against 25.8, 45.8 against 46.7.
// Not the faithful NS-3D form at N = 4, whose small workgroup fills 75 of 128
// threads: 720 elements 27.7 -> 25.6, walls 32.8 -> 30.1, hexahedra 35.2 -> 33.6.
inline bool qns3(const prandtl_ctx *c) { return c->dim == 3 && c->prm.parabolic && c->prm.quirks; }
constexpr int lines_small_fb(int DIM, int NP) { return DIM != 3 || NP > 6 ? 0 : NP <= 4 ? 64 : 128; }
template <int DIM, int NP> bool lines_small(const prandtl_ctx *c)
{
    if (NP == 5 && qns3(c)) return false;
    if (DIM == 3 && NP == 3) return c->NE <= 13824;
    return lines_small_fb(DIM, NP) > 0 && c->NE < 256 * LnCfg<DIM, NP>::EPB;
}

// Orders the general-geometry kernels are built for: 2-D N = 1..5, 3-D N = 2..4.
constexpr bool gen_built(int DIM, int NP) { return DIM == 2 ? NP <= 6 : DIM == 3 && NP <= 5; }

// The mixed form under PRANDTL_ALGO_LINE at N = 3 (periodic 3-D boxes) has no
// choice of viscous launch shape.
inline bool visc_shape_fixed(const prandtl_ctx *c)
{
    return c->rhs_algo == PRANDTL_ALGO_LINE && c->prm.precision == PRANDTL_MIXED && c->dim == 3 && c->Np == 4 &&
           !c->gen && !c->axi && c->geo.bcmask == 0;
}

template <int DIM, int NP> int launch_visc_nd(prandtl_ctx *c, const double *y, double *grad, hipStream_t s)
{
    VArgs a;
    a.tab = c->tab; a.eD = c->eD; a.iw0 = 1.0 / c->tab.w[0]; a.geo = c->geo; a.phys = c->phys;
    a.quirks = c->prm.quirks;
    a.y = y; a.visc = c->d_visc; a.fvf = c->d_fvf; a.grad = grad;
    a.skip = c->skip;
    ProfScope ps(c, s, 1);
    if constexpr (gen_built(DIM, NP)) {
        if (c->gen) {
            // quadrilateral or hexahedral mesh, natural shape
            using Cf = VCfg<DIM, NP, 0>;
            const dim3 nb((c->NE + Cf::EPB - 1) / Cf::EPB), bl(Cf::BLOCK);
            const bool mixed = c->prm.precision == PRANDTL_MIXED, red = !c->prm.quirks && !grad;
            if (mixed && red) hipLaunchKernelGGL((k_visc<DIM, NP, true, 0, false, true, true>), nb, bl, 0, s, a);
            else if (mixed) hipLaunchKernelGGL((k_visc<DIM, NP, true, 0, false, true>), nb, bl, 0, s, a);
            else if (red) hipLaunchKernelGGL((k_visc<DIM, NP, false, 0, false, true, true>), nb, bl, 0, s, a);
            else hipLaunchKernelGGL((k_visc<DIM, NP, false, 0, false, true>), nb, bl, 0, s, a);
            return hip_check(c, hipGetLastError(), "k_visc launch");
        }
    }
    if (!c->prm.quirks && !grad) {
        constexpr int SM = lines_small_fb(DIM, NP);
        const bool small = lines_small<DIM, NP>(c);
        if (c->geo.bcmask) {
            if (small) launch_visc_l<DIM, NP, SM, true>(c, a, s);
            else launch_visc_l<DIM, NP, 0, true>(c, a, s);
        } else {
            switch (c->visc_shape) {
            case 1:
                if constexpr (visc_shape_ok(DIM, NP, 1)) launch_visc_l<DIM, NP, 64, false>(c, a, s);
                break;
            case 2:
                if constexpr (visc_shape_ok(DIM, NP, 2)) launch_visc_l<DIM, NP, 128, false>(c, a, s);
                break;
            case 3:
                if constexpr (visc_shape_ok(DIM, NP, 3)) launch_visc_l<DIM, NP, 256, false>(c, a, s);
                break;
            default:
                if (small) launch_visc_l<DIM, NP, SM, false>(c, a, s);
                else launch_visc_l<DIM, NP, 0, false>(c, a, s);
                break;
            }
        }
        return hip_check(c, hipGetLastError(), "k_visc_l launch");
    }
    if (c->geo.bcmask || grad) {
        // boundary sides, or the gradient output: natural shape
        using Cf = VCfg<DIM, NP, 0>;
        const dim3 nb((c->NE + Cf::EPB - 1) / Cf::EPB), bl(Cf::BLOCK);
        const bool mixed = c->prm.precision == PRANDTL_MIXED;
        if (c->geo.bcmask && mixed) hipLaunchKernelGGL((k_visc<DIM, NP, true, 0, true>), nb, bl, 0, s, a);
        else if (c->geo.bcmask) hipLaunchKernelGGL((k_visc<DIM, NP, false, 0, true>), nb, bl, 0, s, a);
        else if (mixed) hipLaunchKernelGGL((k_visc<DIM, NP, true, 0>), nb, bl, 0, s, a);
        else hipLaunchKernelGGL((k_visc<DIM, NP, false, 0>), nb, bl, 0, s, a);
        return hip_check(c, hipGetLastError(), "k_visc launch");
    }
    switch (c->visc_shape) {
    case 1:
        if constexpr (visc_shape_ok(DIM, NP, 1)) launch_visc_fb<DIM, NP, 64>(c, a, s);
        break;
    case 2:
        if constexpr (visc_shape_ok(DIM, NP, 2)) launch_visc_fb<DIM, NP, 128>(c, a, s);
        break;
    case 3:
        if constexpr (visc_shape_ok(DIM, NP, 3)) launch_visc_fb<DIM, NP, 256>(c, a, s);
        break;
    default:
        launch_visc_fb<DIM, NP, 0>(c, a, s);
        break;
    }
    return hip_check(c, hipGetLastError(), "k_visc launch");
}

// 1-D operators are Euler operators (prandtl_create refuses parabolic ones):
// no viscous kernel is built for them.
template <int DIM, int NP> int launch_visc(prandtl_ctx *c, const double *y, double *grad, hipStream_t s)
{
    if constexpr (DIM == 1) return fail(c, PRANDTL_ERR_UNSUPPORTED, "no viscous kernel in 1-D");
    else return launch_visc_nd<DIM, NP>(c, y, grad, s);
}

// The orders whose periodic 3-D boxes have a choice of algorithm (N = 2..4).
constexpr bool line_built(int DIM, int NP) { return DIM == 3 && NP >= 3 && NP <= 5; }
inline bool line_ok(const prandtl_ctx *c)
{
    return line_built(c->dim, c->Np) && !c->gen && !c->axi && c->geo.bcmask == 0;
}

// The default there.  Both values run the same kernels; TILE admits the forced
// launch shapes.
inline bool line_default(const prandtl_ctx *c)
{
    return line_ok(c) && (c->Np <= 4 || c->prm.blending);
}

// The form of the right-hand side a context's equations take: calls f with
// (QNS3, element type of the viscous terms, AXI) as constants: the faithful NS-3D
// form, the mixed form, an axisymmetric mesh, or plain FP64.
template <int DIM, bool GEN, typename Fn> void rhs_form(const prandtl_ctx *c, Fn f)
{
    using std::false_type;
    using std::true_type;
    if constexpr (DIM == 2 && GEN)
        if (c->axi) return f(false_type{}, 0.0, true_type{});
    if constexpr (DIM == 3)
        if (qns3(c)) return f(true_type{}, 0.0, false_type{});
    if constexpr (DIM > 1)
        if (c->prm.parabolic && c->prm.precision == PRANDTL_MIXED) return f(false_type{}, 0.0f, false_type{});
    f(false_type{}, 0.0, false_type{});
}

template <int DIM, int NP, bool BLEND, int FB, bool OPEN, bool GEN>
int launch_lines(prandtl_ctx *c, const KArgs &a, hipStream_t s)
{
    using Lc = LnCfg<DIM, NP, FB>;
    rhs_form<DIM, GEN>(c, [&](auto q, auto vt, auto axi) {
        hipLaunchKernelGGL((k_rhs_l<DIM, NP, BLEND, decltype(q)::value, decltype(vt), FB, OPEN, GEN, decltype(axi)::value>),
                           dim3((c->NE + Lc::EPB - 1) / Lc::EPB), dim3(Lc::BLOCK), 0, s, a);
    });
    return hip_check(c, hipGetLastError(), "k_rhs_l launch");
}

template <int DIM, int NP, bool BLEND, bool OPEN, bool GEN>
int launch_points(prandtl_ctx *c, const KArgs &a, hipStream_t s)
{
    using Pc = PtCfg<DIM, NP>;
    rhs_form<DIM, GEN>(c, [&](auto q, auto vt, auto axi) {
        hipLaunchKernelGGL((k_rhs_p<DIM, NP, BLEND, decltype(q)::value, decltype(vt), OPEN, GEN, decltype(axi)::value>),
                           dim3((c->NE + Pc::EPB - 1) / Pc::EPB), dim3(Pc::BLOCK), 0, s, a);
    });
    return hip_check(c, hipGetLastError(), "k_rhs_p launch");
}

// Whether a mesh takes k_rhs_p instead of k_rhs_l: by the waves its node
// threads fill (1024 are one per SIMD).  The longer a line's chain (pairs,
// mesh metrics, subcell fluxes), the later its line threads win.  us per
// right-hand side, line / node threads, below and above the limit:
//   2-D N = 2 3,906 quadrilaterals 11.3 / 9.6, 6,480 boxes 7.6 / 8.6; N = 3 3,906
//   blended 10.2 / 9.1, 4,692 8.2 / 9.2; N = 4 1,640 8.6 / 8.1, 2,162 8.7 / 9.6,
//   blended 1,640 13.5 / 9.1, 2,756 13.7 / 11.1, 4,692 14.5 / 15.9; N = 5 2,162
//   quadrilaterals 15.1 / 12.6, 2,756 15.4 / 15.7;
//   3-D N = 2 blended 336 11.1 / 10.3, 1,716 11.6 / 13.2 (without blending no gain);
//   N = 3 120 hexahedra 10.4 / 8.2, 720 10.0 / 10.5; N = 4 210 10.6 / 8.6, 336
//   hexahedra 12.8 / 16.1; N = 5 210 14.0 / 11.2, 336 14.4 / 18.1.
// Where the line's chain is longer still, later:
//   axisymmetric (a line thread recovers up to five nodes' states): N = 1 14,520
//   quadrilaterals 13.7 / 10.7, N = 2 10,100 16.6 / 14.9, 14,520 17.1 / 17.3, N = 3
//   6,480 16.9 / 15.4, 10,100 17.9 / 18.1, N = 4 4,160 18.9 / 18.0, 6,480 21.0 /
//   22.5, N = 5 3,192 20.7 / 19.3, 4,160 21.4 / 22.6;
//   2-D walls: N = 4 3,192 12.7 / 12.2, 4,160 12.8 / 14.1, N = 5 2,352 14.6 / 13.0,
//   3,192 14.8 / 15.6;
//   faithful NS-3D: N = 3 walls 504 23.2 / 21.1, 720 23.2 / 22.6, 990 23.3 / 24.0, N =
//   4 336 25.2 / 21.6, 504 25.6 / 22.1, 720 27.7 / 27.8, walls 504 30.5 / 25.1, 720 32.8
//   / 31.6, but hexahedra 336 31.1 / 33.0.
template <int DIM, int NP, bool BLEND, bool OPEN, bool GEN> int points_waves(const prandtl_ctx *c)
{
    if constexpr (DIM == 2) {
        if (GEN && c->axi) return NP == 2 ? 1920 : NP <= 4 ? 3584 : 4608;
        if (OPEN && !BLEND && NP >= 5) return 3328;
        return NP == 2 ? 768 : NP == 3 ? 1792 : NP == 4 ? 2048 : NP == 5 && !BLEND && !GEN ? 1792 : 3072;
    }
    if constexpr (!BLEND) {
        if (qns3(c) && NP == 4 && (OPEN || GEN)) return 2304;
        if (qns3(c) && NP == 5 && !GEN) return 3328;
    }
    return NP == 3 ? (BLEND ? 512 : 0) : NP == 4 ? 1024 : NP == 5 ? 1536 : 2560;
}

template <int DIM, int NP, bool BLEND, bool OPEN, bool GEN> bool points_ok(const prandtl_ctx *c)
{
    using Pc = PtCfg<DIM, NP>;
    return (long long)(c->NE + Pc::EPB - 1) / Pc::EPB * (Pc::BLOCK / 64) <= points_waves<DIM, NP, BLEND, OPEN, GEN>(c);
}

template <int DIM, int NP, bool BLEND, bool OPEN, bool GEN>
int launch_lines_sized(prandtl_ctx *c, const KArgs &a, hipStream_t s)
{
    if constexpr (points_built(DIM, NP)) {
        if (points_ok<DIM, NP, BLEND, OPEN, GEN>(c)) return launch_points<DIM, NP, BLEND, OPEN, GEN>(c, a, s);
    }
    constexpr int SM = lines_small_fb(DIM, NP);
    if constexpr (SM > 0) {
        if (lines_small<DIM, NP>(c)) return launch_lines<DIM, NP, BLEND, SM, OPEN, GEN>(c, a, s);
    }
    return launch_lines<DIM, NP, BLEND, 0, OPEN, GEN>(c, a, s);
}

template <int DIM, int NP, bool BLEND>
int launch_rhs_t(prandtl_ctx *c, const KArgs &a, hipStream_t s)
{
    ProfScope ps(c, s, 0);
    if constexpr (DIM == 1) {
        if (c->geo.bcmask) return launch_points<DIM, NP, BLEND, true, false>(c, a, s);
        return launch_points<DIM, NP, BLEND, false, false>(c, a, s);
    } else {
        if constexpr (gen_built(DIM, NP)) {
            if (c->gen) return launch_lines_sized<DIM, NP, BLEND, false, true>(c, a, s);
        }
        if (c->geo.bcmask) return launch_lines_sized<DIM, NP, BLEND, true, false>(c, a, s);
        // forced shapes: line threads (64 is the natural size in 2-D)
        if constexpr (rhs_shape_ok(DIM, NP, BLEND, 1))
            if (c->rhs_shape == 1) return launch_lines<DIM, NP, BLEND, DIM == 2 ? 0 : 64, false, false>(c, a, s);
        if constexpr (rhs_shape_ok(DIM, NP, BLEND, 2))
            if (c->rhs_shape == 2) return launch_lines<DIM, NP, BLEND, 128, false, false>(c, a, s);
        if constexpr (rhs_shape_ok(DIM, NP, BLEND, 3))
            if (c->rhs_shape == 3) return launch_lines<DIM, NP, BLEND, 256, false, false>(c, a, s);
        return launch_lines_sized<DIM, NP, BLEND, false, false>(c, a, s);
    }
}

inline KArgs make_kargs(const prandtl_ctx *c, const double *y, const double *u0, double *out, int mode,
                 double dt, double c0, double c1, const double *dtp)
{
    KArgs a;
    a.tab = c->tab; a.geo = c->geo; a.phys = c->phys;
    a.blend = c->prm.blending; a.parabolic = c->prm.parabolic;
    a.ec = c->prm.ec_surface; a.quirks = c->prm.quirks;
    a.mode = mode; a.dt = dt; a.c0 = c0; a.c1 = c1;
    a.dtp = dtp;
    a.tp = c->tp ? c->tp : c->d_time;
    a.tc = c->stage_tc;
    a.y = y; a.u0 = u0; a.out = out;
    a.visc = c->d_visc; a.fvf = c->d_fvf; a.alpha = c->d_alpha; a.eta = c->d_eta;
    a.lam = c->d_lam;
    a.skip = c->skip;
    return a;
}

template <int DIM, int NP>
int launch_rhs(prandtl_ctx *c, const double *y, const double *u0, double *out, int mode, double dt,
               double c0, double c1, hipStream_t s)
{
    const KArgs a = make_kargs(c, y, u0, out, mode, dt, c0, c1, c->dtp);
    if (c->prm.blending) return launch_rhs_t<DIM, NP, true>(c, a, s);
    return launch_rhs_t<DIM, NP, false>(c, a, s);
}

template <int DIM, int NP>
int stage_t(prandtl_ctx *c, const double *y, const double *u0, double *out, int mode, double dt,
            double c0, double c1, hipStream_t s)
{
    if (c->prm.parabolic) {
        int rc = launch_visc<DIM, NP>(c, y, nullptr, s);
        if (rc) return rc;
    }
    return launch_rhs<DIM, NP>(c, y, u0, out, mode, dt, c0, c1, s);
}


// Every (dimension, order) the library is built for: X(DIM, NP).
#define PRANDTL_ORDERS(X) \
    X(1, 2) X(1, 3) X(1, 4) X(1, 5) X(1, 6) X(1, 7) X(1, 8) \
    X(2, 2) X(2, 3) X(2, 4) X(2, 5) X(2, 6) \
    X(3, 3) X(3, 4) X(3, 5) X(3, 6) X(3, 7) X(3, 8)

// The per-order entry points the host unit calls (explicitly instantiated
// in inst_*.hip; "extern" there is empty).
#define PRANDTL_INSTANTIATE(EXT, D, N) \
    EXT template int stage_t<D, N>(prandtl_ctx *, const double *, const double *, double *, int, double, double, \
                                   double, hipStream_t); \
    EXT template int launch_visc<D, N>(prandtl_ctx *, const double *, double *, hipStream_t); \
    EXT template int launch_rhs<D, N>(prandtl_ctx *, const double *, const double *, double *, int, double, double, \
                                      double, hipStream_t);

} // namespace prandtl
