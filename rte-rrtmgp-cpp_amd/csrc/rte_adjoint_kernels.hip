// Adjoint (reverse-mode) kernels of the RTE solvers.  No counterpart in the reference, whose LW
// path has only the surface-temperature Jacobian (src/Rte_lw.cpp:140, do_jacobians).
//
// Longwave.  The forward solver (lw_solver_noscat, F90:58-376) runs, per column, g-point and
// angle, with layers j = 0..n-1 counted from the top and levels j = 0..n:
//     down  I^d_0 = inc / fac,   I^d_{j+1} = T_j I^d_j + Sd_j
//     sfc   I^u_n = (1 - e) I^d_n + e B_s
//     up    I^u_j = T_j I^u_{j+1} + Su_j
// with T = e^{-t}, t = D tau, f = (1 - T)/t - T, Sd = (1 - T) Bd + 2 f (Bl - Bd), Su likewise
// with Bu; broadband fluxes are sums of fac I over g-points and angles.  For cotangents a^u, a^d
// of the broadband fluxes at every level, the adjoint intensities obey
//     lu_0 = fac a^u_0,          lu_{j+1} = fac a^u_{j+1} + T_j lu_j        (top-down)
//     ld_n = fac a^d_n + (1 - e) lu_n,   ld_j = fac a^d_j + T_j ld_{j+1}   (bottom-up)
// and layer j receives dL/dT_j = lu_j I^u_{j+1} + ld_{j+1} I^d_j, dL/dSu_j = lu_j,
// dL/dSd_j = ld_{j+1}.  lu needs only T, so it runs top-down next to the forward down sweep;
// a bottom-up sweep then carries I^u and ld together and replays each K-layer segment's I^d and
// lu from checkpoints (the two-sided scheme of the forward SW solver).  Per (column, g-point)
// the inputs are read twice; no per-layer state is stored.
//
// Shortwave.  With layers j counted from the top, the direct beam dir_{j+1} = dir_j Tn_j and the layer
// sources SU_j = Rdir_j dir_j, SD_j = Tdir_j dir_j, the diffuse fluxes solve
//     dn_{j+1} = T_j dn_j + R_j up_{j+1} + SD_j,      dn_0 = inc_dif
//     up_j     = T_j up_{j+1} + R_j dn_j + SU_j,      up_n = A_s dn_n + alb_dir dir_n.
// For cotangents c^u, c^d of up and dn, the multipliers lam_{j+1}, mu_j of these equations solve
//     mu_{j+1} = T_j mu_j + R_j lam_{j+1} + c^u_{j+1},   mu_0 = c^u_0
//     lam_j    = T_j lam_{j+1} + R_j mu_j + c^d_j,       lam_n = A_s mu_n + c^d_n:
// the same two-stream problem with mu in the place of dn, lam of up and the cotangents as sources.
// So one pair of adding recursions (R_up above, albedo A below) serves both, with two sources each:
// top-down dn = D + R_up up and mu = E + R_up lam, bottom-up up = A dn + S and lam = A mu + F.  A
// top-down sweep stores R_up, D, E and dir at every level; a bottom-up sweep carries A, S, F and the
// beam's adjoint, forms dn, up, mu and lam at each level from both sides, and with them the layer's
// cotangents (gR = lam_{j+1} up_{j+1} + mu_j dn_j, gT = lam_{j+1} dn_j + mu_j up_{j+1}, gSU = mu_j,
// gSD = lam_{j+1}), which it carries through the layer formulas in reverse mode.  Everything is FP64
// but the inputs, the stored level states and the outputs.
#include <algorithm>

#include "common.h"
#include "solver_groups.h"
#include "solver_math.h"

namespace rrtmgp_hip
{
constexpr int ADJ_COLS = 64;
constexpr int ADJ_GPTS = 16;
template<typename Real> struct AdjSeg;
template<> struct AdjSeg<float> { static constexpr int K = 4; };
template<> struct AdjSeg<double> { static constexpr int K = 4; };

template<typename Real>
__device__ __forceinline__ const Real& ld32(const Real* base, uint32_t i)
{
    return *reinterpret_cast<const Real*>(reinterpret_cast<const char*>(base) + i * uint32_t(sizeof(Real)));
}

template<typename Real>
__device__ __forceinline__ Real& st32(Real* base, uint32_t i)
{
    return *reinterpret_cast<Real*>(reinterpret_cast<char*>(base) + i * uint32_t(sizeof(Real)));
}

// T, f and df/dt of the linear-in-tau source (lw_source_noscat, F90:616-653).  Below the switch
// point both f and f' come from the series f = t/2 - t^2/3 + t^3/8 - t^4/30 + t^5/144 - t^6/840
// + t^7/5760; above it from the closed forms, f' = (t T - 1 + T)/t^2 + T.  The switch (1/4 in
// FP32, 1/100 in FP64) keeps both the series truncation and the cancellation of the closed
// form below the precision's rounding.
template<typename Real>
__device__ __forceinline__ void lw_layer_d(Real t, Real& T, Real& f, Real& df)
{
    constexpr Real sw = sizeof(Real) == 4 ? Real(0.25) : Real(0.01);
    T = exp(-t);
    Real q = Real(1. / 840.) - t * Real(1. / 5760.);
    q = Real(1. / 144.) - t * q;
    q = Real(1. / 30.) - t * q;
    q = Real(1. / 8.) - t * q;
    q = Real(1. / 3.) - t * q;
    q = Real(.5) - t * q;
    Real dq = Real(6. / 840.) - t * Real(7. / 5760.);
    dq = Real(5. / 144.) - t * dq;
    dq = Real(4. / 30.) - t * dq;
    dq = Real(3. / 8.) - t * dq;
    dq = Real(2. / 3.) - t * dq;
    dq = Real(.5) - t * dq;
    if (t < sw)
    {
        f = t * q;
        df = dq;
    }
    else
    {
        const Real r = Real(1) / t;
        f = (Real(1) - T) * r - T;
        df = (t * T - Real(1) + T) * r * r + T;
    }
}

// One (column, g-point) per thread, 64 columns x 16 g-points per work-group.
template<typename Real, int NMU>
__global__ __launch_bounds__(ADJ_COLS * ADJ_GPTS)
void lw_adjoint_kernel(int64_t ncol, int64_t nlay, int64_t ngpt, int top_at_1, int nmus,
                       const Real* __restrict__ secants, const Real* __restrict__ weights,
                       const Real* __restrict__ tau, const Real* __restrict__ lay_src,
                       const Real* __restrict__ lev_inc, const Real* __restrict__ lev_dec,
                       const Real* __restrict__ emis, const Real* __restrict__ sfc_src,
                       const Real* __restrict__ inc_flux, const Real* __restrict__ a_up,
                       const Real* __restrict__ a_dn, Real* __restrict__ ckpt,
                       Real* __restrict__ d_tau, Real* __restrict__ d_lay, Real* __restrict__ d_lev_inc,
                       Real* __restrict__ d_lev_dec, Real* __restrict__ d_sfc_src, Real* __restrict__ d_emis)
{
    constexpr int K = AdjSeg<Real>::K;
    const int lane = threadIdx.x;
    const int w = __builtin_amdgcn_readfirstlane(int(threadIdx.y));
    const int64_t icol = int64_t(blockIdx.x) * ADJ_COLS + lane;
    const int64_t igpt = int64_t(blockIdx.y) * ADJ_GPTS + w;
    if (icol >= ncol || igpt >= ngpt) return;     // no barriers in this kernel
    const int64_t n = nlay;
    const int64_t nseg = (n + K - 1) / K;
    const int64_t c2 = icol + ncol * igpt;
    const int64_t lslab = ncol * nlay * igpt;
    const Real* tau_g = tau + lslab;
    const Real* lay_g = lay_src + lslab;
    const Real* bd_g = (top_at_1 ? lev_inc : lev_dec) + lslab;     // source at the layer's lower level
    const Real* bu_g = (top_at_1 ? lev_dec : lev_inc) + lslab;     // source at the layer's upper level
    Real* dtau_g = d_tau + lslab;
    Real* dlay_g = d_lay + lslab;
    Real* dbd_g = (top_at_1 ? d_lev_inc : d_lev_dec) + lslab;
    Real* dbu_g = (top_at_1 ? d_lev_dec : d_lev_inc) + lslab;
    const uint32_t ucol = uint32_t(icol), uncol = uint32_t(ncol);
    auto lay_of = [&](int64_t j) -> uint32_t { return uint32_t(top_at_1 ? j : n - 1 - j); };   // layer j from the top
    auto lev_of = [&](int64_t j) -> uint32_t { return uint32_t(top_at_1 ? j : n - j); };       // level j from the top
    // Checkpoint q of segment s: q < NMU: I^d, NMU <= q: lu, at the segment's top level.
    auto ck = [&](int64_t s, int q) -> Real& { return ckpt[((s * 2 * NMU + q) * ngpt + igpt) * ncol + icol]; };
    const Real pi = Real(3.14159265358979323846);

    Real D[NMU], fac[NMU], Id[NMU], Lu[NMU];
    const Real inc = inc_flux ? inc_flux[c2] : Real(0);
#pragma unroll
    for (int mu = 0; mu < NMU; ++mu)
    {
        const bool on = mu < nmus;
        D[mu] = on ? secants[c2 + ncol * ngpt * mu] : Real(0);
        fac[mu] = on ? Real(2) * pi * weights[mu] : Real(0);
        Id[mu] = on ? inc / fac[mu] : Real(0);
        Lu[mu] = fac[mu] * ld32(a_up, ucol + uncol * lev_of(0));
    }

    // Pass 1, top-down: forward I^d and the adjoint lu.
    for (int64_t s = 0; s < nseg; ++s)
    {
        const int64_t j0 = s * K;
        const int nk = int(std::min<int64_t>(K, n - j0));
#pragma unroll
        for (int mu = 0; mu < NMU; ++mu) { ck(s, mu) = Id[mu]; ck(s, NMU + mu) = Lu[mu]; }
        Real tv[K], lv[K], bv[K], au[K];
#pragma unroll
        for (int kk = 0; kk < K; ++kk)
            if (kk < nk)
            {
                const uint32_t l = ucol + uncol * lay_of(j0 + kk);
                tv[kk] = ld32(tau_g, l); lv[kk] = ld32(lay_g, l); bv[kk] = ld32(bd_g, l);
                au[kk] = ld32(a_up, ucol + uncol * lev_of(j0 + kk + 1));
            }
#pragma unroll
        for (int kk = 0; kk < K; ++kk)
            if (kk < nk)
#pragma unroll
                for (int mu = 0; mu < NMU; ++mu)
                {
                    Real T, f, df;
                    lw_layer_d(tv[kk] * D[mu], T, f, df);
                    Id[mu] = T * Id[mu] + ((Real(1) - T) * bv[kk] + Real(2) * f * (lv[kk] - bv[kk]));
                    Lu[mu] = fac[mu] * au[kk] + T * Lu[mu];
                }
    }

    // Surface.
    const Real e = emis[c2], bs = sfc_src[c2];
    const Real ad_s = ld32(a_dn, ucol + uncol * lev_of(n));
    Real Iu[NMU], Ld[NMU];
    Real g_e = Real(0), g_bs = Real(0);
#pragma unroll
    for (int mu = 0; mu < NMU; ++mu)
    {
        Iu[mu] = (Real(1) - e) * Id[mu] + e * bs;
        g_e += Lu[mu] * (bs - Id[mu]);
        g_bs += e * Lu[mu];
        Ld[mu] = fac[mu] * ad_s + (Real(1) - e) * Lu[mu];
    }
    d_emis[c2] = g_e;
    d_sfc_src[c2] = g_bs;

    // Pass 2, bottom-up: forward I^u and the adjoint ld, replaying I^d and lu per segment.
    for (int64_t s = nseg - 1; s >= 0; --s)
    {
        const int64_t j0 = s * K;
        const int nk = int(std::min<int64_t>(K, n - j0));
        Real tv[K], lv[K], bdv[K], buv[K], au[K], adv[K];
#pragma unroll
        for (int kk = 0; kk < K; ++kk)
            if (kk < nk)
            {
                const uint32_t l = ucol + uncol * lay_of(j0 + kk);
                tv[kk] = ld32(tau_g, l); lv[kk] = ld32(lay_g, l);
                bdv[kk] = ld32(bd_g, l); buv[kk] = ld32(bu_g, l);
                au[kk] = ld32(a_up, ucol + uncol * lev_of(j0 + kk + 1));
                adv[kk] = ld32(a_dn, ucol + uncol * lev_of(j0 + kk));
            }
        Real sId[K][NMU], sLu[K][NMU], sT[K][NMU], sF[K][NMU], sDF[K][NMU];
        {
            Real id[NMU], lu[NMU];
#pragma unroll
            for (int mu = 0; mu < NMU; ++mu) { id[mu] = ck(s, mu); lu[mu] = ck(s, NMU + mu); }
#pragma unroll
            for (int kk = 0; kk < K; ++kk)
                if (kk < nk)
#pragma unroll
                    for (int mu = 0; mu < NMU; ++mu)
                    {
                        Real T, f, df;
                        lw_layer_d(tv[kk] * D[mu], T, f, df);
                        sId[kk][mu] = id[mu]; sLu[kk][mu] = lu[mu];
                        sT[kk][mu] = T; sF[kk][mu] = f; sDF[kk][mu] = df;
                        id[mu] = T * id[mu] + ((Real(1) - T) * bdv[kk] + Real(2) * f * (lv[kk] - bdv[kk]));
                        lu[mu] = fac[mu] * au[kk] + T * lu[mu];
                    }
        }
#pragma unroll
        for (int kk = K - 1; kk >= 0; --kk)
            if (kk < nk)
            {
                Real g_tau = Real(0), g_bl = Real(0), g_bd = Real(0), g_bu = Real(0);
#pragma unroll
                for (int mu = 0; mu < NMU; ++mu)
                {
                    const Real T = sT[kk][mu], f = sF[kk][mu];
                    const Real gSu = sLu[kk][mu], gSd = Ld[mu];
                    const Real gT = sLu[kk][mu] * Iu[mu] + Ld[mu] * sId[kk][mu]
                                  - bdv[kk] * gSd - buv[kk] * gSu;
                    const Real gf = Real(2) * ((lv[kk] - bdv[kk]) * gSd + (lv[kk] - buv[kk]) * gSu);
                    g_tau += D[mu] * (-T * gT + sDF[kk][mu] * gf);
                    g_bd += gSd * ((Real(1) - T) - Real(2) * f);
                    g_bu += gSu * ((Real(1) - T) - Real(2) * f);
                    g_bl += Real(2) * f * (gSd + gSu);
                    Iu[mu] = T * Iu[mu] + ((Real(1) - T) * buv[kk] + Real(2) * f * (lv[kk] - buv[kk]));
                    Ld[mu] = fac[mu] * adv[kk] + T * Ld[mu];
                }
                const uint32_t l = ucol + uncol * lay_of(j0 + kk);
                st32(dtau_g, l) = g_tau;
                st32(dlay_g, l) = g_bl;
                st32(dbd_g, l) = g_bd;
                st32(dbu_g, l) = g_bu;
            }
    }
}

template<typename Real>
int lw_adjoint(int64_t ncol, int64_t nlay, int64_t ngpt, int top_at_1, int64_t nmus, const Real* secants,
               const Real* weights, const Real* tau, const Real* lay, const Real* linc, const Real* ldec,
               const Real* emis, const Real* sfc_src, const Real* inc_flux, const Real* a_up, const Real* a_dn,
               Real* d_tau, Real* d_lay, Real* d_linc, Real* d_ldec, Real* d_sfc_src, Real* d_emis, void* stream)
{
    if (ncol <= 0 || nlay <= 0 || ngpt <= 0) return arg_error("lw_adjoint: empty extents");
    if (nmus < 1 || nmus > 4) return arg_error("lw_adjoint: n_gauss_angles must be 1..4");
    if (!secants || !weights || !tau || !lay || !linc || !ldec || !emis || !sfc_src || !a_up || !a_dn ||
        !d_tau || !d_lay || !d_linc || !d_ldec || !d_sfc_src || !d_emis)
        return arg_error("lw_adjoint: NULL array");
    if (ncol * (nlay + 1) * int64_t(sizeof(Real)) >= (int64_t(1) << 32))
        return arg_error("lw_adjoint: ncol * (nlay + 1) values of one g-point must stay below 4 GiB");
    hipStream_t s = as_stream(stream);
    constexpr int K = AdjSeg<Real>::K;
    const int nmu_t = nmus == 1 ? 1 : 4;
    const int64_t nseg = (nlay + K - 1) / K;
    Real* ck = nullptr;
    RRTMGP_TRY(scratch_alloc(&ck, size_t(nseg * 2 * nmu_t * ngpt * ncol), s));
    const dim3 grid(grid1(ncol, ADJ_COLS), grid1(ngpt, ADJ_GPTS));
    const dim3 block(ADJ_COLS, ADJ_GPTS);
    int rc;
    {
        RRTMGP_TIMED("lw_adjoint_kernel", s);
        auto launch = [&](auto kernel) {
            hipLaunchKernelGGL(kernel, grid, block, 0, s, ncol, nlay, ngpt, top_at_1, int(nmus), secants, weights,
                               tau, lay, linc, ldec, emis, sfc_src, inc_flux, a_up, a_dn, ck, d_tau, d_lay, d_linc,
                               d_ldec, d_sfc_src, d_emis);
        };
        if (nmus == 1) launch(lw_adjoint_kernel<Real, 1>);
        else launch(lw_adjoint_kernel<Real, 4>);
        rc = check_hip(hipGetLastError(), "lw_adjoint_kernel");
    }
    scratch_free(ck, s);
    return rc;
}
// ---------------------------------------------------------------------------------------------
// The longwave adjoint on factored sources: each source is a Planck fraction (per g-point) times the band's
// Planck function at the layer or a level (lw_solver_kernel's FACT form), one Gaussian angle.  Read and
// written per g-point are tau, the fraction and their cotangents (24 values of traffic a layer became 8); the
// cotangents of the band Planck functions are summed over the work-group's g-points (one band's) in LDS every
// K layers, in a fixed order, into (ncol, nlay, groups).  Layers and recurrences as in lw_adjoint_kernel.
template<typename Real> struct AdjFactSeg;
template<> struct AdjFactSeg<float> { static constexpr int K = 4; };    // 48 KiB of LDS: two work-groups a CU
template<> struct AdjFactSeg<double> { static constexpr int K = 2; };

template<typename Real>
struct LwAdjFactArgs
{
    int64_t ncol, nlay, ngpt, emis_nbnd;
    int top_at_1;
    Real D, fac;                                       // secant; 2 pi times the weight
    const Real *tau, *pf, *blay, *blev, *emis, *sfc_src, *a_up, *a_dn;
    Real *ckpt, *d_tau, *d_pf, *d_blay, *d_blo, *d_bhi, *d_sfc_src, *d_emis;
};

template<typename Real>
__global__ __launch_bounds__(SB_COLS * SB_GPTS) __attribute__((amdgpu_waves_per_eu(sizeof(Real) == 4 ? 8 : 4)))
void lw_adjoint_factored_kernel(LwAdjFactArgs<Real> a, Groups grp)
{
    constexpr int K = AdjFactSeg<Real>::K;
    __shared__ Real red[3][K][SB_GPTS][SB_COLS];
    const int lane = threadIdx.x;
    const int w = __builtin_amdgcn_readfirstlane(int(threadIdx.y));
    const int gi = blockIdx.y, gcount = grp.count[gi];
    const int64_t ncol = a.ncol, n = a.nlay, col0 = int64_t(blockIdx.x) * SB_COLS, icol = col0 + lane;
    const int64_t igpt = grp.start[gi] + w;
    const bool active = icol < ncol && w < gcount;
    const int64_t nseg = (n + K - 1) / K;
    const int64_t c2 = icol + ncol * igpt, lslab = ncol * n * igpt;
    const Real* tau_g = a.tau + lslab;
    const Real* pf_g = a.pf + lslab;
    Real* dtau_g = a.d_tau + lslab;
    Real* dpf_g = a.d_pf + lslab;
    const Real* blay_g = a.blay + ncol * n * grp.band[gi];
    const Real* blev_g = a.blev + ncol * (n + 1) * grp.band[gi];
    Real* ck_g = a.ckpt + ncol * nseg * 2 * igpt;
    const uint32_t ucol = uint32_t(icol), uncol = uint32_t(ncol);
    auto lay_of = [&](int64_t j) -> uint32_t { return uint32_t(a.top_at_1 ? j : n - 1 - j); };   // layer j from the top
    auto lev_of = [&](int64_t j) -> uint32_t { return uint32_t(a.top_at_1 ? j : n - j); };       // level j from the top
    auto ck = [&](int64_t s, int q) -> Real& { return st32(ck_g, ucol + uncol * uint32_t(s * 2 + q)); };
    const Real D = a.D, fac = a.fac;

    Real Id = Real(0), Lu = Real(0);
    if (active)
    {
        // Down: forward I^d and the adjoint lu; checkpoints at the top of each segment.
        Lu = fac * ld32(a.a_up, ucol + uncol * lev_of(0));
        for (int64_t s = 0; s < nseg; ++s)
        {
            const int64_t j0 = s * K;
            const int nk = int(std::min<int64_t>(K, n - j0));
            ck(s, 0) = Id; ck(s, 1) = Lu;
            Real tv[K], pv[K], bl[K], bd[K], au[K];
#pragma unroll
            for (int kk = 0; kk < K; ++kk)
                if (kk < nk)
                {
                    const uint32_t l = ucol + uncol * lay_of(j0 + kk);
                    tv[kk] = ld32(tau_g, l); pv[kk] = ld32(pf_g, l); bl[kk] = ld32(blay_g, l);
                    bd[kk] = ld32(blev_g, ucol + uncol * lev_of(j0 + kk + 1));
                    au[kk] = ld32(a.a_up, ucol + uncol * lev_of(j0 + kk + 1));
                }
#pragma unroll
            for (int kk = 0; kk < K; ++kk)
                if (kk < nk)
                {
                    Real T, f, df;
                    lw_layer_d(tv[kk] * D, T, f, df);
                    Id = T * Id + pv[kk] * ((Real(1) - T) * bd[kk] + Real(2) * f * (bl[kk] - bd[kk]));
                    Lu = fac * au[kk] + T * Lu;
                }
        }
    }
    // Surface.
    Real Iu = Real(0), Ld = Real(0);
    if (active)
    {
        const Real e = a.emis[grp.band[gi] + a.emis_nbnd * icol], bs = a.sfc_src[c2];
        Iu = (Real(1) - e) * Id + e * bs;
        a.d_emis[c2] = Lu * (bs - Id);
        a.d_sfc_src[c2] = e * Lu;
        Ld = fac * ld32(a.a_dn, ucol + uncol * lev_of(n)) + (Real(1) - e) * Lu;
    }
    // Up: forward I^u and the adjoint ld, replaying I^d and lu per segment.
    for (int64_t s = nseg - 1; s >= 0; --s)
    {
        const int64_t j0 = s * K;
        const int nk = int(std::min<int64_t>(K, n - j0));
        Real gbl[K], gbd[K], gbu[K];
#pragma unroll
        for (int kk = 0; kk < K; ++kk) { gbl[kk] = Real(0); gbd[kk] = Real(0); gbu[kk] = Real(0); }
        if (active)
        {
            Real tv[K], pv[K], bl[K], bv[K + 1], au[K], adv[K], sId[K], sLu[K];
            bv[0] = ld32(blev_g, ucol + uncol * lev_of(j0));
#pragma unroll
            for (int kk = 0; kk < K; ++kk)
                if (kk < nk)
                {
                    const uint32_t l = ucol + uncol * lay_of(j0 + kk);
                    tv[kk] = ld32(tau_g, l); pv[kk] = ld32(pf_g, l); bl[kk] = ld32(blay_g, l);
                    bv[kk + 1] = ld32(blev_g, ucol + uncol * lev_of(j0 + kk + 1));
                    au[kk] = ld32(a.a_up, ucol + uncol * lev_of(j0 + kk + 1));
                    adv[kk] = ld32(a.a_dn, ucol + uncol * lev_of(j0 + kk));
                }
            {
                Real id = ck(s, 0), lu = ck(s, 1);
#pragma unroll
                for (int kk = 0; kk < K; ++kk)
                    if (kk < nk)
                    {
                        Real T, f, df;
                        lw_layer_d(tv[kk] * D, T, f, df);
                        sId[kk] = id; sLu[kk] = lu;
                        id = T * id + pv[kk] * ((Real(1) - T) * bv[kk + 1] + Real(2) * f * (bl[kk] - bv[kk + 1]));
                        lu = fac * au[kk] + T * lu;
                    }
            }
#pragma unroll
            for (int kk = K - 1; kk >= 0; --kk)
                if (kk < nk)
                {
                    Real T, f, df;
                    lw_layer_d(tv[kk] * D, T, f, df);
                    const Real p = pv[kk], Bl = bl[kk], Bu = bv[kk], Bd = bv[kk + 1];
                    const Real gSu = sLu[kk], gSd = Ld;
                    const Real gT = sLu[kk] * Iu + Ld * sId[kk] - p * (Bd * gSd + Bu * gSu);
                    const Real gf = Real(2) * p * ((Bl - Bd) * gSd + (Bl - Bu) * gSu);
                    const Real c = (Real(1) - T) - Real(2) * f, f2 = Real(2) * f;
                    // dL/dp and, times p, dL/dB.
                    const uint32_t l = ucol + uncol * lay_of(j0 + kk);
                    st32(dtau_g, l) = D * (-T * gT + df * gf);
                    st32(dpf_g, l) = gSd * (c * Bd + f2 * Bl) + gSu * (c * Bu + f2 * Bl);
                    gbl[kk] = p * f2 * (gSd + gSu);
                    gbd[kk] = p * c * gSd;
                    gbu[kk] = p * c * gSu;
                    Iu = T * Iu + p * ((Real(1) - T) * Bu + f2 * (Bl - Bu));
                    Ld = fac * adv[kk] + T * Ld;
                }
        }
#pragma unroll
        for (int kk = 0; kk < K; ++kk)
        {
            red[0][kk][w][lane] = gbl[kk]; red[1][kk][w][lane] = gbd[kk]; red[2][kk][w][lane] = gbu[kk];
        }
        __syncthreads();
        // Row r of the 3 K rows: component r / K at layer j0 + r % K.
        for (int r = w; r < 3 * K; r += SB_GPTS)
        {
            const int c = r / K, kk = r % K;
            if (kk >= nk || icol >= ncol) continue;
            Real v = red[c][kk][0][lane];
            for (int q = 1; q < gcount; ++q) v += red[c][kk][q][lane];
            // The lower source (c = 1) is at level L + 1 with the top at layer 1, else at level L.
            Real* out = c == 0 ? a.d_blay : ((c == 1) == (a.top_at_1 != 0) ? a.d_bhi : a.d_blo);
            out[icol + ncol * (int64_t(lay_of(j0 + kk)) + n * gi)] = v;
        }
        __syncthreads();
    }
}

template<typename Real>
int lw_adjoint_factored(int64_t ncol, int64_t nlay, int64_t ngpt, int top_at_1, double secant, double weight,
                        const Real* tau, const Real* pf, const Real* blay, const Real* blev, int64_t nbnd,
                        const int* band_lims, const Real* emis, int64_t emis_nbnd, const Real* sfc_src,
                        const Real* a_up, const Real* a_dn, Real* d_tau, Real* d_pf, Real* d_blay, Real* d_blo,
                        Real* d_bhi, Real* d_sfc_src, Real* d_emis, void* stream)
{
    if (ncol <= 0 || nlay <= 0 || ngpt <= 0 || nbnd <= 0) return arg_error("lw_adjoint_factored: empty extents");
    if (!tau || !pf || !blay || !blev || !band_lims || !emis || emis_nbnd < nbnd || !sfc_src || !a_up || !a_dn ||
        !d_tau || !d_pf || !d_blay || !d_blo || !d_bhi || !d_sfc_src || !d_emis)
        return arg_error("lw_adjoint_factored: NULL array");
    constexpr int K = AdjFactSeg<Real>::K;
    const int64_t nseg = (nlay + K - 1) / K;
    if (ncol * std::max<int64_t>(nlay + 1, 2 * nseg) * int64_t(sizeof(Real)) >= (int64_t(1) << 32))
        return arg_error("lw_adjoint_factored: ncol * (nlay + 1) values of one g-point must stay below 4 GiB");
    Groups grp;
    RRTMGP_TRY(make_groups(ngpt, nbnd, band_lims, grp));
    hipStream_t s = as_stream(stream);
    Real* ck = nullptr;
    RRTMGP_TRY(scratch_alloc(&ck, size_t(nseg * 2 * ngpt * ncol), s));
    const Real pi = Real(3.14159265358979323846);
    const LwAdjFactArgs<Real> args{ncol, nlay, ngpt, emis_nbnd, top_at_1, Real(secant), Real(2) * pi * Real(weight),
                                   tau, pf, blay, blev, emis, sfc_src, a_up, a_dn, ck, d_tau, d_pf, d_blay, d_blo,
                                   d_bhi, d_sfc_src, d_emis};
    int rc;
    {
        RRTMGP_TIMED("lw_adjoint_factored_kernel", s);
        hipLaunchKernelGGL(lw_adjoint_factored_kernel<Real>, dim3(grid1(ncol, SB_COLS), unsigned(grp.n)),
                           dim3(SB_COLS, SB_GPTS), 0, s, args, grp);
        rc = check_hip(hipGetLastError(), "lw_adjoint_factored_kernel");
    }
    scratch_free(ck, s);
    return rc;
}

// ---------------------------------------------------------------------------------------------
// Shortwave adjoint: one (column, g-point) per thread, 64 columns x 4 g-points per work-group.
constexpr int SWA_GPTS = 4;
constexpr int SWA_NS = 4;    // stored level states: R_up, D, E, dir

template<typename Real>
struct SwAdjArgs
{
    int64_t ncol, nlay, ngpt;
    int top_at_1;
    const Real *tau, *ssa, *gasy, *mu0, *alb_dir, *alb_dif, *inc_dir, *inc_dif, *a_up, *a_dn, *a_dir;
    Real *st, *d_tau, *d_ssa, *d_g, *d_alb_dir, *d_alb_dif;
};

// 1/x to within a rounding: the approximation and two Newton steps.
__device__ __forceinline__ double rcp_full(double x)
{
    const double r = rcp_f64(x);
    return fma(r, fma(-x, r, 1.), r);
}

// The two-stream layer (F90:1043-1104 with the clamp of rte_solver_kernels.cu:581-583) and what its
// reverse mode reads again.  The direct-beam terms are written with G = (e^{-k tau} - Tn) / (1 - k mu0),
// in which the reference's factor 1 / (1 - (k mu0)^2) cancels to 1 / (1 + k mu0) identically (see
// sw_layer_fp32): no term grows as k mu0 approaches 1.  With x = (1 - k mu0) tau / mu0 and
// chi = ((1 - e^{-x}) / x - 1) / x,
//     G = e^{-k tau} (tau / mu0) (1 + x chi),   dG/dk = tau e^{-k tau} (tau / mu0) chi,
//     dG/dtau = (e^{-k tau} - G) / mu0;
// chi comes from its series for |x| < 1/4 (truncation < 1e-16); elsewhere G and dG/dk are difference
// quotients, which lose less than 1 / x^2 there.
struct SwLayerAdj
{
    double R, T, Rd, Td, Tn;                                            // the layer's properties
    double w0, om, g, k, g1, g2, g3, g4, a1, a2, e1, c2, RT, r, P, Q, G, dGdk, rd, td, b;

    __device__ __forceinline__ void eval(double tau, double w0_, double g_, double mu0, double inv_mu0)
    {
        w0 = w0_; g = g_;
        om = 1. - w0;
        g1 = 2. - w0 * (1.25 + .75 * g);
        g2 = .75 * w0 * (1. - g);
        g3 = .5 - .75 * mu0 * g;
        g4 = 1. - g3;
        a1 = g1 * g4 + g2 * g3;
        a2 = g1 * g3 + g2 * g4;
        k = sqrt(fmax(2. * om * (g1 + g2), Limits<double>::k_min));     // gamma1 - gamma2 = 2 (1 - w0)
        e1 = exp(-tau * k);
        const double y = tau * inv_mu0;
        Tn = exp(-y);
        c2 = 1. - e1 * e1;
        const double km = k * mu0, ek = 1. - km, x = y * ek;
        if (fabs(x) < .25)
        {
            double c = 1. / 479001600.;                                 // 1/12!, alternating down to 1/2!
            c = 1. / 39916800. - x * c;
            c = 1. / 3628800. - x * c;
            c = 1. / 362880. - x * c;
            c = 1. / 40320. - x * c;
            c = 1. / 5040. - x * c;
            c = 1. / 720. - x * c;
            c = 1. / 120. - x * c;
            c = 1. / 24. - x * c;
            c = 1. / 6. - x * c;
            c = .5 - x * c;                                             // -chi
            const double ey = e1 * y;
            G = ey * (1. - x * c);
            dGdk = -tau * ey * c;
        }
        else
        {
            const double iek = rcp_full(ek);
            G = (e1 - Tn) * iek;
            dGdk = (mu0 * G - tau * e1) * iek;
        }
        const double d0 = k * (2. - c2) + g1 * c2, opk = 1. + km;
        const double q = rcp_full(d0 * opk);
        RT = q * opk;
        r = q * d0;                                                     // 1 / (1 + k mu0)
        R = RT * g2 * c2;
        T = 2. * RT * k * e1;
        P = (a2 + k * g3) * c2 + 2. * k * (g3 - a2 * mu0) * e1 * G;
        Q = (a1 - k * g4) * c2 * Tn - 2. * k * (g4 + a1 * mu0) * G;
        const double s = w0 * RT * r;
        rd = s * P;
        td = -s * Q;
        b = 1. - Tn;
        Rd = fmax(fmin(rd, b), Limits<double>::eps);
        Td = fmax(fmin(td, b - Rd), Limits<double>::eps);
    }

    // Cotangents of (tau, w0, g) for those of (R, T, Rd, Td, Tn).  max and min pass the cotangent of the
    // operand they picked.
    __device__ __forceinline__ void reverse(double tau, double mu0, double inv_mu0, double gR, double gT, double gRd,
                                            double gTd, double gTn, double& g_tau, double& g_w0, double& g_g) const
    {
        const double eps = Limits<double>::eps;
        const double m2 = fmin(td, b - Rd), m1 = fmin(rd, b);
        double g_td = 0.;
        if (m2 >= eps)
        {
            if (td <= b - Rd) g_td = gTd;
            else { gTn -= gTd; gRd -= gTd; }
        }
        double g_rd = 0.;
        if (m1 >= eps)
        {
            if (rd <= b) g_rd = gRd;
            else gTn -= gRd;
        }
        const double wr = w0 * r, s = wr * RT, km = k * mu0;
        const double g_s = g_rd * P - g_td * Q, gP = s * g_rd, gQ = -s * g_td;
        const double eG = 2. * e1 * G, g3a = g3 - a2 * mu0, g4a = g4 + a1 * mu0, c2T = c2 * Tn, G2 = 2. * G;
        double g_k = gP * (g3 * c2 + g3a * eG) - gQ * (g4 * c2T + g4a * G2);
        double g_c2 = gP * (a2 + k * g3) + gQ * (a1 - k * g4) * Tn;
        const double g_e1G = 2. * k * g3a * gP;
        const double g_G = g_e1G * e1 - 2. * k * g4a * gQ;
        double g_e1 = g_e1G * G;
        gTn += gQ * (a1 - k * g4) * c2;
        const double g_a1 = gQ * (c2T - km * G2), g_a2 = gP * (c2 - km * eG);
        double g_g3 = gP * k * (c2 + eG);
        const double g_g4 = -gQ * k * (c2T + G2);
        // s = w0 RT r, R = RT gamma2 c2, T = 2 RT k e1, RT = 1 / (k (2 - c2) + gamma1 c2).
        g_k -= g_s * s * mu0 * r;
        const double ke = 2. * k * e1;
        const double g_RT = g_s * wr + gR * g2 * c2 + gT * ke;
        const double g_d0 = -g_RT * RT * RT;
        g_c2 += gR * RT * g2 + g_d0 * (g1 - k);
        g_k += 2. * gT * RT * e1 + g_d0 * (2. - c2) + g_G * dGdk;
        g_e1 += 2. * (gT * RT * k - e1 * g_c2);
        double g_g1 = g_d0 * c2, g_g2 = gR * RT * c2;
        const double ge = g_e1 * e1;
        g_k -= ge * tau;
        g_tau = g_G * (e1 - G) * inv_mu0 - ge * k - gTn * Tn * inv_mu0;
        const double q = 2. * om * (g1 + g2);
        const double g_kk = q >= Limits<double>::k_min ? g_k * rcp_full(k) : 0.;        // k^2 = q = 2 om (gamma1 + gamma2)
        const double g_q = g_kk * om;
        g_w0 = g_s * RT * r - g_kk * (g1 + g2);
        g_g1 += g_a1 * g4 + g_a2 * g3 + g_q;
        g_g2 += g_a1 * g3 + g_a2 * g4 + g_q;
        g_g3 += g_a1 * g2 + g_a2 * g1 - (g_g4 + g_a1 * g1 + g_a2 * g2);
        g_w0 += .75 * (1. - g) * g_g2 - (1.25 + .75 * g) * g_g1;
        g_g = -.75 * (w0 * (g_g1 + g_g2) + mu0 * g_g3);
    }
};

// One thread's place: offsets of its (column, g-point) in the layer arrays, the cotangents and the
// level-state store (state q of level j at st[((4 j + q) ngpt + igpt) ncol + icol], j from the top).
template<typename Real>
struct SwAdjAt
{
    int64_t icol, c2, lay0, dlay, lev0, dlev, st0, dst, dq;
    bool in;
    __device__ explicit SwAdjAt(const SwAdjArgs<Real>& a)
    {
        icol = int64_t(blockIdx.x) * ADJ_COLS + threadIdx.x;
        const int64_t igpt = int64_t(blockIdx.y) * SWA_GPTS + threadIdx.y;
        in = icol < a.ncol && igpt < a.ngpt;
        c2 = icol + a.ncol * igpt;
        lay0 = icol + a.ncol * a.nlay * igpt + (a.top_at_1 ? 0 : a.ncol * (a.nlay - 1));   // top layer
        dlay = a.top_at_1 ? a.ncol : -a.ncol;
        lev0 = icol + (a.top_at_1 ? 0 : a.ncol * a.nlay);                                  // top level
        dlev = dlay;
        dq = a.ncol * a.ngpt;
        st0 = c2;
        dst = SWA_NS * dq;
    }
};

// Sweep down: the column above each level, for the fluxes (D) and for the multipliers (E).
template<typename Real>
__global__ __launch_bounds__(ADJ_COLS * SWA_GPTS)
void sw_adjoint_down_kernel(SwAdjArgs<Real> a)
{
    const SwAdjAt<Real> t(a);
    if (!t.in) return;
    const int64_t n = a.nlay;
    const double m0 = double(a.mu0[t.icol]), im0 = 1. / m0;
    double dir = double(a.inc_dir[t.c2]) * m0, D = a.inc_dif ? double(a.inc_dif[t.c2]) : 0., Ru = 0.;
    double E = double(a.a_up[t.lev0]);
    Real* st = a.st + t.st0;
    int64_t l = t.lay0, v = t.lev0;
    // The next layer's inputs are requested before this layer's chain starts.
    Real nt = a.tau[l], nw = a.ssa[l], ng = a.gasy[l], ncd = a.a_dn[v], ncu = a.a_up[v + t.dlev];
    for (int64_t j = 0; j < n; ++j)
    {
        const double tau = double(nt), w0 = double(nw), g = double(ng), cd = double(ncd), cu = double(ncu);
        l += t.dlay; v += t.dlev;
        if (j + 1 < n)
        {
            nt = a.tau[l]; nw = a.ssa[l]; ng = a.gasy[l]; ncd = a.a_dn[v]; ncu = a.a_up[v + t.dlev];
        }
        st[0] = Real(Ru); st[t.dq] = Real(D); st[2 * t.dq] = Real(E); st[3 * t.dq] = Real(dir);
        st += t.dst;
        SwLayerAdj L;
        L.eval(tau, w0, g, m0, im0);
        const double Te = L.T * rcp_full(1. - L.R * Ru);
        D = L.Td * dir + Te * (D + Ru * L.Rd * dir);
        E = cu + Te * (E + Ru * cd);
        Ru = L.R + L.T * Te * Ru;
        dir *= L.Tn;
    }
    st[0] = Real(Ru); st[t.dq] = Real(D); st[2 * t.dq] = Real(E); st[3 * t.dq] = Real(dir);
}

// Sweep up: the column below each level, the fluxes and multipliers of the level, the layer's gradients.
// With CHAIN the cotangents of tau, ssa and g are carried on to the gases' absorption and Rayleigh optical
// depths (d_tau and d_ssa receive those; the band cloud is held fixed): with the scattering optical depth
// ts = ssa tau, tau = abs + ray + cloud and g a cloud quantity over ts,
//     d_abs = d_tau - d_ssa ssa / tau,   d_ray = d_abs + d_ssa / tau - d_g g / ts.
// (The combine rule's cut-off is on the gases' optical depth, which the gas-optics adjoint knows: there
// d_ray = d_abs where that is up to 2 eps.)
// Bound by its FP64 arithmetic (153 VGPRs, 3 wavefronts per SIMD) next to 10 values of traffic a layer.
// The pair of sweeps takes 3.4 + 5.4 ms for the 14 bands of 16384 columns x 128 layers in FP32; the four
// it replaced (two forward and two reverse recursions through 12 stored states a level, the layer
// Jacobian on forward-mode dual numbers) took 22.9 ms.
template<typename Real, bool CHAIN>
__global__ __launch_bounds__(ADJ_COLS * SWA_GPTS)
void sw_adjoint_up_kernel(SwAdjArgs<Real> a)
{
    const SwAdjAt<Real> t(a);
    if (!t.in) return;
    const int64_t n = a.nlay;
    const double m0 = double(a.mu0[t.icol]), im0 = 1. / m0;
    const Real* st = a.st + t.st0 + n * t.dst;
    int64_t l = t.lay0 + (n - 1) * t.dlay, v = t.lev0 + n * t.dlev;
    double A, S, F, up, lam, ldir, cu;
    {
        const double ad = double(a.alb_dir[t.c2]);
        const double Ru = double(st[0]), D = double(st[t.dq]), E = double(st[2 * t.dq]), dir = double(st[3 * t.dq]);
        const double cd = double(a.a_dn[v]);
        cu = double(a.a_up[v]);
        A = double(a.alb_dif[t.c2]);
        S = dir * ad;
        F = cd;
        const double den = rcp_full(1. - Ru * A);
        const double dn = (D + Ru * S) * den, mu = (E + Ru * F) * den;
        up = A * dn + S;
        lam = A * mu + F;
        ldir = cd + double(a.a_dir[v]) + mu * ad;
        a.d_alb_dif[t.c2] = Real(mu * dn);
        a.d_alb_dir[t.c2] = Real(mu * dir);
    }
    st -= t.dst; v -= t.dlev;
    Real nt = a.tau[l], nw = a.ssa[l], ng = a.gasy[l], ncd = a.a_dn[v], ncu = a.a_up[v], ncr = a.a_dir[v];
    Real nR = st[0], nD = st[t.dq], nE = st[2 * t.dq], ndir = st[3 * t.dq];
    for (int64_t j = n - 1; j >= 0; --j)
    {
        const double tau = double(nt), w0 = double(nw), g = double(ng), cd = double(ncd), cr = double(ncr);
        const double cu0 = double(ncu), Ru = double(nR), D = double(nD), E = double(nE), dir = double(ndir);
        const int64_t lo = l;
        l -= t.dlay; v -= t.dlev; st -= t.dst;
        if (j > 0)
        {
            nt = a.tau[l]; nw = a.ssa[l]; ng = a.gasy[l]; ncd = a.a_dn[v]; ncu = a.a_up[v]; ncr = a.a_dir[v];
            nR = st[0]; nD = st[t.dq]; nE = st[2 * t.dq]; ndir = st[3 * t.dq];
        }
        SwLayerAdj L;
        L.eval(tau, w0, g, m0, im0);
        const double Te = L.T * rcp_full(1. - L.R * A);
        S = L.Rd * dir + Te * (S + A * L.Td * dir);
        F = cd + Te * (F + A * cu);
        A = L.R + L.T * Te * A;
        const double den = rcp_full(1. - Ru * A);
        const double dn = (D + Ru * S) * den, mu = (E + Ru * F) * den;
        double gt, gw, gg;
        L.reverse(tau, m0, im0, lam * up + mu * dn, lam * dn + mu * up, mu * dir, lam * dir, ldir * dir, gt, gw, gg);
        if constexpr (CHAIN)
        {
            const double op_eps = 3. * double(Limits<Real>::tiny), ts = w0 * tau;
            const double it = tau > op_eps ? rcp_full(tau) : 0.;
            const double da = gt - gw * w0 * it;
            const double dr = gw * it - (ts > op_eps ? gg * g * rcp_full(ts) : 0.);
            a.d_tau[lo] = Real(da); a.d_ssa[lo] = Real(da + dr);
        }
        else
        {
            a.d_tau[lo] = Real(gt); a.d_ssa[lo] = Real(gw); a.d_g[lo] = Real(gg);
        }
        ldir = cd + cr + mu * L.Rd + lam * L.Td + ldir * L.Tn;
        up = A * dn + S;
        lam = A * mu + F;
        cu = cu0;
    }
}

template<typename Real>
int sw_adjoint(int64_t ncol, int64_t nlay, int64_t ngpt, int top_at_1, const Real* tau, const Real* ssa,
               const Real* g, const Real* mu0, const Real* alb_dir, const Real* alb_dif, const Real* inc_dir,
               const Real* inc_dif, const Real* a_up, const Real* a_dn, const Real* a_dir, Real* d_tau,
               Real* d_ssa, Real* d_g, Real* d_alb_dir, Real* d_alb_dif, void* stream, bool chain = false)
{
    if (ncol <= 0 || nlay <= 0 || ngpt <= 0) return arg_error("sw_adjoint: empty extents");
    if (!tau || !ssa || !g || !mu0 || !alb_dir || !alb_dif || !inc_dir || !a_up || !a_dn || !a_dir || !d_tau ||
        !d_ssa || (!chain && !d_g) || !d_alb_dir || !d_alb_dif)
        return arg_error("sw_adjoint: NULL array");
    hipStream_t s = as_stream(stream);
    Real* st = nullptr;
    RRTMGP_TRY(scratch_alloc(&st, SWA_NS * size_t((nlay + 1) * ngpt * ncol), s));
    const SwAdjArgs<Real> args{ncol, nlay, ngpt, top_at_1, tau, ssa, g, mu0, alb_dir, alb_dif, inc_dir, inc_dif,
                               a_up, a_dn, a_dir, st, d_tau, d_ssa, d_g, d_alb_dir, d_alb_dif};
    const dim3 grid(grid1(ncol, ADJ_COLS), grid1(ngpt, SWA_GPTS));
    const dim3 block(ADJ_COLS, SWA_GPTS);
    int rc = RRTMGP_OK;
    {
        RRTMGP_TIMED("sw_adjoint_down_kernel", s);
        hipLaunchKernelGGL(sw_adjoint_down_kernel<Real>, grid, block, 0, s, args);
        rc = check_hip(hipGetLastError(), "sw_adjoint_down_kernel");
    }
    if (rc == RRTMGP_OK)
    {
        RRTMGP_TIMED("sw_adjoint_up_kernel", s);
        auto kernel = chain ? sw_adjoint_up_kernel<Real, true> : sw_adjoint_up_kernel<Real, false>;
        hipLaunchKernelGGL(kernel, grid, block, 0, s, args);
        rc = check_hip(hipGetLastError(), "sw_adjoint_up_kernel");
    }
    scratch_free(st, s);
    return rc;
}


// ---------------------------------------------------------------------------------------------
// Assembly of the gas-optics gradients.

// col_gas(gas) = vmr(gas) col_dry for gas >= 1 and col_gas(0) = col_dry, so
//   d vmr(gas) = d col_gas(gas) col_dry,   d col_dry = d col_gas(0) + sum_gas d col_gas(gas) vmr(gas).
// d_col (ncol, nlay, ngas+1) -> d_vmr (ncol, nlay, ngas) (overwritten), d_col_dry (ncol, nlay).
template<typename Real>
__global__ void col_chain_kernel(int64_t ncol, int64_t nlay, int ngas, const rrtmgp_gas_vmr gases,
                                 const Real* __restrict__ col_dry, const Real* __restrict__ d_col,
                                 Real* __restrict__ d_vmr, Real* __restrict__ d_col_dry)
{
    const int64_t i = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
    const int64_t ncl = ncol * nlay;
    if (i >= ncl) return;
    const Real cd = col_dry[i];
    for (int gas = 0; gas < ngas; ++gas)
        d_vmr[i + ncl * gas] = d_col[i + ncl * (gas + 1)] * cd;
    // The derivative at fixed mixing ratios, formed by the gas-optics adjoint (slot ngas + 1).
    d_col_dry[i] = d_col[i + ncl * (ngas + 1)];
}

// d_tlev (ncol, nlev): level i receives d_lo of layer i and d_hi of layer i-1.
template<typename Real>
__global__ void levels_kernel(int64_t ncol, int64_t nlay, const Real* __restrict__ lo, const Real* __restrict__ hi,
                              Real* __restrict__ d_tlev)
{
    const int64_t i = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
    if (i >= ncol * (nlay + 1)) return;
    const int64_t ilev = i / ncol;
    Real v = Real(0);
    if (ilev < nlay) v += lo[i];
    if (ilev > 0) v += hi[i - ncol];
    d_tlev[i] = v;
}

// out (nbnd, ncol) = sums over each band's g-points of in (ncol, ngpt); band_lims (2, nbnd) 1-based.
template<typename Real>
__global__ void gpt_to_band_kernel(int64_t ncol, int64_t nbnd, const int* __restrict__ band_lims,
                                   const Real* __restrict__ in, Real* __restrict__ out)
{
    const int64_t i = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
    if (i >= ncol * nbnd) return;
    const int64_t b = i % nbnd, icol = i / nbnd;
    Real s = Real(0);
    for (int g = band_lims[2 * b] - 1; g < band_lims[2 * b + 1]; ++g) s += in[icol + ncol * g];
    out[b + nbnd * icol] = s;
}
}  // namespace rrtmgp_hip

using namespace rrtmgp_hip;

#define RRTMGP_DEF_ADJOINT(S, T)                                                                   \
extern "C" int rrtmgp_hip_lw_solver_noscat_adjoint_##S(int64_t ncol, int64_t nlay, int64_t ngpt,   \
    int top_at_1, int64_t nmus, const T* secants, const T* weights, const T* tau,                   \
    const T* lay_source, const T* lev_source_inc, const T* lev_source_dec, const T* sfc_emis,       \
    const T* sfc_src, const T* inc_flux, const T* bb_up_cot, const T* bb_dn_cot, T* d_tau,          \
    T* d_lay_source, T* d_lev_source_inc, T* d_lev_source_dec, T* d_sfc_src, T* d_sfc_emis,         \
    void* stream)                                                                                   \
{                                                                                                   \
    return lw_adjoint<T>(ncol, nlay, ngpt, top_at_1, nmus, secants, weights, tau, lay_source,       \
                         lev_source_inc, lev_source_dec, sfc_emis, sfc_src, inc_flux, bb_up_cot,    \
                         bb_dn_cot, d_tau, d_lay_source, d_lev_source_inc, d_lev_source_dec,        \
                         d_sfc_src, d_sfc_emis, stream);                                            \
}                                                                                                   \
extern "C" int rrtmgp_hip_sw_solver_2stream_adjoint_##S(int64_t ncol, int64_t nlay, int64_t ngpt,  \
    int top_at_1, const T* tau, const T* ssa, const T* g, const T* mu0, const T* sfc_alb_dir,       \
    const T* sfc_alb_dif, const T* inc_flux_dir, const T* inc_flux_dif, const T* bb_up_cot,         \
    const T* bb_dn_cot, const T* bb_dir_cot, T* d_tau, T* d_ssa, T* d_g, T* d_sfc_alb_dir,           \
    T* d_sfc_alb_dif, void* stream)                                                                 \
{                                                                                                   \
    return sw_adjoint<T>(ncol, nlay, ngpt, top_at_1, tau, ssa, g, mu0, sfc_alb_dir, sfc_alb_dif,    \
                         inc_flux_dir, inc_flux_dif, bb_up_cot, bb_dn_cot, bb_dir_cot, d_tau, d_ssa,\
                         d_g, d_sfc_alb_dir, d_sfc_alb_dif, stream);                                \
}

RRTMGP_DEF_ADJOINT(f32, float)
RRTMGP_DEF_ADJOINT(f64, double)

#define RRTMGP_DEF_ADJOINT_BANDS(S, T)                                                             \
extern "C" int rrtmgp_hip_lw_adjoint_factored_##S(int64_t ncol, int64_t nlay, int64_t ngpt,        \
    int top_at_1, double secant, double weight, const T* tau, const T* planck_frac,                 \
    const T* band_lay_src, const T* band_lev_src, int64_t nbnd, const int* band_lims_gpt,           \
    const T* sfc_emis, int64_t emis_nbnd, const T* sfc_src, const T* bb_up_cot,                     \
    const T* bb_dn_cot, T* d_tau, T* d_planck_frac, T* d_lay_src, T* d_lev_src_lo, T* d_lev_src_hi, \
    T* d_sfc_src, T* d_sfc_emis, void* stream)                                                      \
{                                                                                                   \
    return lw_adjoint_factored<T>(ncol, nlay, ngpt, top_at_1, secant, weight, tau, planck_frac,     \
                                  band_lay_src, band_lev_src, nbnd, band_lims_gpt, sfc_emis,        \
                                  emis_nbnd, sfc_src, bb_up_cot, bb_dn_cot, d_tau, d_planck_frac,   \
                                  d_lay_src, d_lev_src_lo, d_lev_src_hi, d_sfc_src, d_sfc_emis,     \
                                  stream);                                                          \
}                                                                                                   \
extern "C" int rrtmgp_hip_sw_adjoint_gases_##S(int64_t ncol, int64_t nlay, int64_t ngpt,           \
    int top_at_1, const T* tau, const T* ssa, const T* g, const T* mu0, const T* sfc_alb_dir,       \
    const T* sfc_alb_dif, const T* inc_flux_dir, const T* inc_flux_dif, const T* bb_up_cot,         \
    const T* bb_dn_cot, const T* bb_dir_cot, T* d_tau_abs, T* d_tau_ray, T* d_sfc_alb_dir,           \
    T* d_sfc_alb_dif, void* stream)                                                                 \
{                                                                                                   \
    return sw_adjoint<T>(ncol, nlay, ngpt, top_at_1, tau, ssa, g, mu0, sfc_alb_dir, sfc_alb_dif,    \
                         inc_flux_dir, inc_flux_dif, bb_up_cot, bb_dn_cot, bb_dir_cot, d_tau_abs,   \
                         d_tau_ray, nullptr, d_sfc_alb_dir, d_sfc_alb_dif, stream, true);           \
}

RRTMGP_DEF_ADJOINT_BANDS(f32, float)
RRTMGP_DEF_ADJOINT_BANDS(f64, double)

#define RRTMGP_DEF_ADJ_HELPERS(S, T)                                                               \
extern "C" int rrtmgp_hip_adjoint_col_chain_##S(int64_t ncol, int64_t nlay,                        \
    const rrtmgp_gas_vmr* gases, const T* col_dry, const T* d_col_gas, T* d_vmr, T* d_col_dry,       \
    void* stream)                                                                                   \
{                                                                                                   \
    if (!gases || gases->ngas < 1 || gases->ngas > RRTMGP_MAX_GAS || !col_dry || !d_col_gas ||     \
        !d_vmr || !d_col_dry || ncol <= 0 || nlay <= 0)                                             \
        return arg_error("adjoint_col_chain: bad arguments");                                      \
    const int64_t n = ncol * nlay;                                                                  \
    RRTMGP_TIMED("col_chain_kernel", as_stream(stream));                                            \
    hipLaunchKernelGGL(col_chain_kernel<T>, dim3(grid1(n, 256)), dim3(256), 0, as_stream(stream),  \
                       ncol, nlay, int(gases->ngas), *gases, col_dry, d_col_gas, d_vmr, d_col_dry); \
    RRTMGP_LAUNCHED("col_chain_kernel");                                                           \
    return RRTMGP_OK;                                                                               \
}                                                                                                   \
extern "C" int rrtmgp_hip_adjoint_levels_##S(int64_t ncol, int64_t nlay, const T* d_lo,            \
    const T* d_hi, T* d_tlev, void* stream)                                                         \
{                                                                                                   \
    if (!d_lo || !d_hi || !d_tlev || ncol <= 0 || nlay <= 0) return arg_error("adjoint_levels: bad arguments"); \
    const int64_t n = ncol * (nlay + 1);                                                            \
    RRTMGP_TIMED("levels_kernel", as_stream(stream));                                               \
    hipLaunchKernelGGL(levels_kernel<T>, dim3(grid1(n, 256)), dim3(256), 0, as_stream(stream),     \
                       ncol, nlay, d_lo, d_hi, d_tlev);                                             \
    RRTMGP_LAUNCHED("levels_kernel");                                                              \
    return RRTMGP_OK;                                                                               \
}                                                                                                   \
extern "C" int rrtmgp_hip_gpt_to_band_##S(int64_t ncol, int64_t nbnd, const int* band_lims_gpt,    \
    const T* in, T* out, void* stream)                                                              \
{                                                                                                   \
    if (!band_lims_gpt || !in || !out || ncol <= 0 || nbnd <= 0) return arg_error("gpt_to_band: bad arguments"); \
    const int64_t n = ncol * nbnd;                                                                  \
    RRTMGP_TIMED("gpt_to_band_kernel", as_stream(stream));                                          \
    hipLaunchKernelGGL(gpt_to_band_kernel<T>, dim3(grid1(n, 256)), dim3(256), 0, as_stream(stream),\
                       ncol, nbnd, band_lims_gpt, in, out);                                         \
    RRTMGP_LAUNCHED("gpt_to_band_kernel");                                                         \
    return RRTMGP_OK;                                                                               \
}

RRTMGP_DEF_ADJ_HELPERS(f32, float)
RRTMGP_DEF_ADJ_HELPERS(f64, double)
