// Reverse-mode drivers of the column-radiation path (no reference counterpart; the forward
// sequence they differentiate is src_test/Radiation_solver.cu:489-580 LW and :763-893 SW).
#include "Radiation_adjoint.h"

#include <algorithm>
#include <stdexcept>
#include <vector>

#include "Optical_props.h"
#include "hip_dispatch.h"

using rrtmgp_cpp::hip_check;
using rrtmgp_cpp::stream;

namespace
{
// An output array: allocated (and zeroed) when empty, else checked for shape.
template<int N>
void ensure(Array_gpu<Float,N>& a, const std::array<int,N>& dims)
{
    if (a.size() == 0) { a = Array_gpu<Float,N>(dims); a.fill(Float(0)); return; }
    for (int i = 0; i < N; ++i)
        if (a.get_dims()[i] != dims[i]) throw std::invalid_argument("adjoint output has the wrong shape");
}

template<int N>
void zero(Array_gpu<Float,N>& a)
{
    if (a.size()) hip_check(rrtmgp_hip_memset(a.ptr(), 0, size_t(a.size()) * sizeof(Float), stream()));
}

// (nbnd, ncol) band values -> (ncol, ngpt) g-point values.
Array_gpu<Float,2> expand(const Gas_optics_rrtmgp_gpu& kd, const Array_gpu<Float,2>& bnd, int ncol)
{
    Array_gpu<Float,2> out({ncol, kd.get_ngpt()});
    hip_check(K<Float>::expand_and_transpose(ncol, kd.get_nband(), kd.get_ngpt(),
                                             kd.get_band_lims_gpoint_gpu().ptr(), bnd.ptr(), out.ptr(), stream()));
    return out;
}

// Bands processed together: consecutive bands whose per-g-point scratch (`arrays` values per column, layer
// and g-point) stays below `bytes`, at least one.  One launch per kernel then covers them: at a few thousand
// columns and fewer a single band's work-groups leave most of the GPU idle (250 x 60 columns and layers: 4 tiles
// x 16 g-points), at 16384 x 128 in FP32 two shortwave and four longwave bands share the staging of the
// gas-optics inputs.  A batch has at most 256 groups of 16 g-points of a band, which is what the longwave solver
// adjoint takes.  Cotangents are written over the optical properties they belong to, so that both drivers
// together take 2.6 GB of scratch there (one band at a time with 12 stored shortwave states took 3.1 GB).
constexpr double GiB = 1024. * 1024. * 1024.;

struct Batch
{
    int b0, nb, g0, ng;              // bands, first g-point (0-based), g-points
    int groups;                      // groups of up to 16 g-points of a band
    std::vector<int> lims;           // (2, nb) band limits, 1-based within the batch
};

std::vector<Batch> make_batches(const Gas_optics_rrtmgp_gpu& kd, int64_t ncl, double arrays, double bytes)
{
    const double most = bytes / (arrays * double(sizeof(Float)) * double(ncl));
    const Array<int,2>& bl = kd.get_band_lims_gpoint();
    std::vector<Batch> out;
    for (int b = 0; b < kd.get_nband(); ++b)
    {
        const int s = bl({1, b + 1}), e = bl({2, b + 1}), groups = (e - s + 16) / 16;
        if (out.empty() || double(out.back().ng + e - s + 1) > most || out.back().groups + groups > 256)
            out.push_back({b, 0, s - 1, 0, 0, {}});
        Batch& t = out.back();
        t.groups += groups;
        t.lims.push_back(s - t.g0);
        t.lims.push_back(e - t.g0);
        ++t.nb;
        t.ng += e - s + 1;
    }
    return out;
}

// A block of the library's caching allocator on the driver's stream.
struct Scratch
{
    Float* ptr = nullptr;
    explicit Scratch(int64_t n)
    {
        void* p = nullptr;
        hip_check(rrtmgp_hip_cache_malloc(&p, size_t(n) * sizeof(Float), stream()));
        ptr = static_cast<Float*>(p);
    }
    ~Scratch() { (void)rrtmgp_hip_cache_free(ptr, stream()); }
    Scratch(const Scratch&) = delete;
    Scratch& operator=(const Scratch&) = delete;
};

template<typename F>
int most_of(const std::vector<Batch>& v, F f)
{
    int m = 0;
    for (const Batch& t : v) m = std::max(m, f(t));
    return m;
}

// The adjoint differentiates the plain table gas optics.  With an MLP surrogate set, the forward
// solve_gpu runs the network instead, so a gradient from here would belong to another function.
void refuse_surrogate(const Gas_optics_rrtmgp_gpu& kdist)
{
    if (kdist.has_surrogate())
        throw std::invalid_argument("adjoint: the k-distribution has an MLP gas-optics surrogate set, whose "
                                    "forward the adjoint does not differentiate; clear it (set_surrogate(NULL)) "
                                    "before computing gradients");
}

// play(1, 1) and play(1, nlay), which decide the orientation, in one wait for the device.
std::pair<Float, Float> column_ends(const Array_gpu<Float,2>& p_lay)
{
    const Float* none = nullptr;
    const int64_t size = 0;
    const Float lo = Float(0.), hi = Float(0.);
    int64_t bad = 0;
    Float ends[2] = {Float(0.), Float(0.)};
    hip_check(K<Float>::check_ranges(1, &none, &size, &lo, &hi, &bad, p_lay.ptr(), p_lay.dim(1), p_lay.dim(2), ends,
                                     stream()));
    return {ends[0], ends[1]};
}

bool cloudy(const Cloud_optics_gpu* c, const Array_gpu<Float,2>& lwp)
{
    return c != nullptr && lwp.size() > 0;
}
}  // namespace


void lw_adjoint_gpu(Gas_optics_rrtmgp_gpu& kdist, Cloud_optics_gpu* cloud_optics, const Gas_concs_gpu& gas_concs,
                    const Array_gpu<Float,2>& p_lay, const Array_gpu<Float,2>& p_lev,
                    const Array_gpu<Float,2>& t_lay, const Array_gpu<Float,2>& t_lev,
                    const Array_gpu<Float,1>& t_sfc, const Array_gpu<Float,2>& emis_sfc,
                    const Array_gpu<Float,2>& lwp, const Array_gpu<Float,2>& iwp,
                    const Array_gpu<Float,2>& rel, const Array_gpu<Float,2>& rei,
                    const Array_gpu<Float,2>& g_flux_up, const Array_gpu<Float,2>& g_flux_dn,
                    Lw_adjoint_out& out)
{
    if (!kdist.source_is_internal()) throw std::invalid_argument("lw_adjoint_gpu needs a longwave k-distribution");
    refuse_surrogate(kdist);
    const int ncol = p_lay.dim(1), nlay = p_lay.dim(2), nlev = nlay + 1;
    const int ngpt = kdist.get_ngpt(), nbnd = kdist.get_nband(), ngas = kdist.get_ngas();
    const int64_t ncl = int64_t(ncol) * nlay;
    const rrtmgp_kdist_dev& kd = kdist.device_tables();
    rrtmgp_gas_vmr vmr;
    kdist.vmr_descriptor(gas_concs, ncol, nlay, vmr);
    const auto [p_first, p_last] = column_ends(p_lay);
    const Bool top_at_1 = p_first < p_last;
    const int sfc_lay = p_first > p_last ? 1 : nlay;

    ensure<2>(out.d_t_lay, {ncol, nlay}); ensure<2>(out.d_t_lev, {ncol, nlev}); ensure<1>(out.d_t_sfc, {ncol});
    ensure<2>(out.d_lnp_lay, {ncol, nlay}); ensure<2>(out.d_p_lev, {ncol, nlev});
    ensure<3>(out.d_vmr, {ncol, nlay, ngas}); ensure<2>(out.d_emis_sfc, {nbnd, ncol});

    Array_gpu<Float,2> col_dry({ncol, nlay});
    const Array_gpu<Float,2>& h2o = gas_concs.get_vmr("h2o");
    Gas_optics_rrtmgp_gpu::get_col_dry(col_dry, h2o, p_lev);
    std::unique_ptr<Optical_props_1scl_gpu> cl;
    if (cloudy(cloud_optics, lwp))
    {
        cl = std::make_unique<Optical_props_1scl_gpu>(ncol, nlay, *cloud_optics);
        cloud_optics->cloud_optics(lwp, iwp, rel, rei, *cl);
    }

    Array_gpu<Float,3> d_col({ncol, nlay, ngas + 2});
    Array_gpu<Float,2> d_lo({ncol, nlay}), d_hi({ncol, nlay}), d_col_dry({ncol, nlay}), d_emis_gpt({ncol, ngpt});
    zero(d_col); zero(d_lo); zero(d_hi); zero(out.d_t_lay); zero(out.d_t_sfc); zero(out.d_lnp_lay); zero(out.d_p_lev);

    // Factored sources, as the forward driver: per g-point only tau and the Planck fractions, with their cotangents
    // in the same place, and the solver's checkpoints (two values in four layers).
    const std::vector<Batch> batches = make_batches(kdist, ncl, 2.5, 1.25 * GiB);
    const int mg = most_of(batches, [](const Batch& t) { return t.ng; });
    const int mb = most_of(batches, [](const Batch& t) { return t.nb; });
    const int mq = most_of(batches, [](const Batch& t) { return t.groups; });
    // One block for all, so that the shortwave driver finds it large enough for its level states.
    const int64_t sizes[] = {ncl * mg, ncl * mg, ncl * mb, int64_t(ncol) * nlev * mb, ncl * mq, ncl * mq, ncl * mq,
                             int64_t(ncol) * mg, int64_t(ncol) * mg, int64_t(ncol) * mg};
    int64_t total = 0;
    for (const int64_t n : sizes) total += (n + 63) / 64 * 64;
    Scratch block(total);
    Float* part[10];
    Float* next = block.ptr;
    for (int i = 0; i < 10; ++i) { part[i] = next; next += (sizes[i] + 63) / 64 * 64; }
    const auto [tau, pf, blay, blev, dblay, dblo, dbhi, sfc, sfcj, dsfc] = part;
    const Float* ctau = cl ? cl->get_tau().ptr() : nullptr;
    for (const Batch& t : batches)
    {
        hip_check(K<Float>::gas_optics_lw_bands_factored(
                &kd, t.b0, t.nb, ncol, nlay, p_lay.ptr(), t_lay.ptr(), t_lev.ptr(), t_sfc.ptr(), col_dry.ptr(), &vmr,
                sfc_lay, ctau, tau, pf, blay, blev, sfc, sfcj, stream()));
        // One Gaussian angle, as the forward driver (src_test/Radiation_solver.cpp:533): D = 1.66, w = 0.5.
        hip_check(K<Float>::lw_adjoint_factored(
                ncol, nlay, t.ng, top_at_1, 1.66, 0.5, tau, pf, blay, blev, t.nb, t.lims.data(),
                emis_sfc.ptr() + t.b0, nbnd, sfc, g_flux_up.ptr(), g_flux_dn.ptr(), tau, pf, dblay, dblo, dbhi, dsfc,
                d_emis_gpt.ptr() + int64_t(ncol) * t.g0, stream()));
        hip_check(K<Float>::gas_optics_lw_adjoint_bands(
                &kd, t.b0, t.nb, ncol, nlay, p_lay.ptr(), t_lay.ptr(), t_lev.ptr(), t_sfc.ptr(), col_dry.ptr(), &vmr,
                sfc_lay, tau, pf, dblay, dblo, dbhi, dsfc, d_col.ptr(), out.d_t_lay.ptr(), out.d_lnp_lay.ptr(),
                d_lo.ptr(), d_hi.ptr(), out.d_t_sfc.ptr(), stream()));
    }
    hip_check(K<Float>::adjoint_levels(ncol, nlay, d_lo.ptr(), d_hi.ptr(), out.d_t_lev.ptr(), stream()));
    hip_check(K<Float>::adjoint_col_chain(ncol, nlay, &vmr, col_dry.ptr(), d_col.ptr(), out.d_vmr.ptr(),
                                          d_col_dry.ptr(), stream()));
    hip_check(K<Float>::get_col_dry_adjoint(ncol, nlay, h2o.ptr(), h2o.dim(1), h2o.dim(2), p_lev.ptr(),
                                            d_col_dry.ptr(), out.d_vmr.ptr() + ncl * (kd.idx_h2o - 1),
                                            out.d_p_lev.ptr(), stream()));
    hip_check(K<Float>::gpt_to_band(ncol, nbnd, kd.band_lims_gpt, d_emis_gpt.ptr(), out.d_emis_sfc.ptr(), stream()));
}


void sw_adjoint_gpu(Gas_optics_rrtmgp_gpu& kdist, Cloud_optics_gpu* cloud_optics, bool delta_cloud,
                    const Gas_concs_gpu& gas_concs,
                    const Array_gpu<Float,2>& p_lay, const Array_gpu<Float,2>& p_lev,
                    const Array_gpu<Float,2>& t_lay,
                    const Array_gpu<Float,2>& sfc_alb_dir, const Array_gpu<Float,2>& sfc_alb_dif,
                    const Array_gpu<Float,1>& tsi_scaling, const Array_gpu<Float,1>& mu0,
                    const Array_gpu<Float,2>& lwp, const Array_gpu<Float,2>& iwp,
                    const Array_gpu<Float,2>& rel, const Array_gpu<Float,2>& rei,
                    const Array_gpu<Float,2>& g_flux_up, const Array_gpu<Float,2>& g_flux_dn,
                    const Array_gpu<Float,2>& g_flux_dir, Sw_adjoint_out& out)
{
    if (!kdist.source_is_external()) throw std::invalid_argument("sw_adjoint_gpu needs a shortwave k-distribution");
    refuse_surrogate(kdist);
    const int ncol = p_lay.dim(1), nlay = p_lay.dim(2), nlev = nlay + 1;
    const int ngpt = kdist.get_ngpt(), nbnd = kdist.get_nband(), ngas = kdist.get_ngas();
    const int64_t ncl = int64_t(ncol) * nlay;
    const rrtmgp_kdist_dev& kd = kdist.device_tables();
    rrtmgp_gas_vmr vmr;
    kdist.vmr_descriptor(gas_concs, ncol, nlay, vmr);
    const auto [p_first, p_last] = column_ends(p_lay);
    const Bool top_at_1 = p_first < p_last;

    ensure<2>(out.d_t_lay, {ncol, nlay}); ensure<2>(out.d_lnp_lay, {ncol, nlay}); ensure<2>(out.d_p_lev, {ncol, nlev});
    ensure<3>(out.d_vmr, {ncol, nlay, ngas});
    ensure<2>(out.d_sfc_alb_dir, {nbnd, ncol}); ensure<2>(out.d_sfc_alb_dif, {nbnd, ncol});

    Array_gpu<Float,2> col_dry({ncol, nlay});
    const Array_gpu<Float,2>& h2o = gas_concs.get_vmr("h2o");
    Gas_optics_rrtmgp_gpu::get_col_dry(col_dry, h2o, p_lev);
    std::unique_ptr<Optical_props_2str_gpu> cl;
    if (cloudy(cloud_optics, lwp))
    {
        cl = std::make_unique<Optical_props_2str_gpu>(ncol, nlay, *cloud_optics);
        if (delta_cloud) cloud_optics->cloud_optics_delta_scaled(lwp, iwp, rel, rei, *cl);
        else cloud_optics->cloud_optics(lwp, iwp, rel, rei, *cl);
    }
    // Incoming direct flux per g-point: solar source times the TSI scaling
    // (src_test/Radiation_solver.cpp:739-743).
    Array_gpu<Float,2> toa({ncol, ngpt});
    hip_check(K<Float>::spread_col(ncol, ngpt, kdist.solar_source_device().ptr(), toa.ptr(), stream()));
    hip_check(K<Float>::scale_by_col(ncol, ngpt, toa.ptr(), tsi_scaling.ptr(), stream()));
    Array_gpu<Float,2> ad_gpt = expand(kdist, sfc_alb_dir, ncol), af_gpt = expand(kdist, sfc_alb_dif, ncol);

    Array_gpu<Float,3> d_col({ncol, nlay, ngas + 2});
    Array_gpu<Float,2> d_col_dry({ncol, nlay}), d_ad({ncol, ngpt}), d_af({ncol, ngpt});
    zero(d_col); zero(out.d_t_lay); zero(out.d_lnp_lay); zero(out.d_p_lev);

    // Three arrays, two of which receive the cotangents, and the solver's four level states.
    const std::vector<Batch> batches = make_batches(kdist, ncl, 7., 1.75 * GiB);
    const int mg = most_of(batches, [](const Batch& t) { return t.ng; });
    Array_gpu<Float,3> tau({ncol, nlay, mg}), ssa({ncol, nlay, mg}), g({ncol, nlay, mg});
    const Float* ct = cl ? cl->get_tau().ptr() : nullptr;
    const Float* cs = cl ? cl->get_ssa().ptr() : nullptr;
    const Float* cg = cl ? cl->get_g().ptr() : nullptr;
    for (const Batch& t : batches)
    {
        const int64_t o = int64_t(ncol) * t.g0;
        hip_check(K<Float>::gas_optics_sw_bands(&kd, t.b0, t.nb, ncol, nlay, p_lay.ptr(), t_lay.ptr(), col_dry.ptr(),
                                                &vmr, ct, cs, cg, tau.ptr(), ssa.ptr(), g.ptr(), stream()));
        hip_check(K<Float>::sw_adjoint_gases(
                ncol, nlay, t.ng, top_at_1, tau.ptr(), ssa.ptr(), g.ptr(), mu0.ptr(), ad_gpt.ptr() + o,
                af_gpt.ptr() + o, toa.ptr() + o, nullptr, g_flux_up.ptr(), g_flux_dn.ptr(), g_flux_dir.ptr(),
                tau.ptr(), ssa.ptr(), d_ad.ptr() + o, d_af.ptr() + o, stream()));
        hip_check(K<Float>::gas_optics_sw_adjoint_bands(&kd, t.b0, t.nb, ncol, nlay, p_lay.ptr(), t_lay.ptr(),
                                                        col_dry.ptr(), &vmr, tau.ptr(), ssa.ptr(), d_col.ptr(),
                                                        out.d_t_lay.ptr(), out.d_lnp_lay.ptr(), stream()));
    }
    hip_check(K<Float>::adjoint_col_chain(ncol, nlay, &vmr, col_dry.ptr(), d_col.ptr(), out.d_vmr.ptr(),
                                          d_col_dry.ptr(), stream()));
    hip_check(K<Float>::get_col_dry_adjoint(ncol, nlay, h2o.ptr(), h2o.dim(1), h2o.dim(2), p_lev.ptr(),
                                            d_col_dry.ptr(), out.d_vmr.ptr() + ncl * (kd.idx_h2o - 1),
                                            out.d_p_lev.ptr(), stream()));
    hip_check(K<Float>::gpt_to_band(ncol, nbnd, kd.band_lims_gpt, d_ad.ptr(), out.d_sfc_alb_dir.ptr(), stream()));
    hip_check(K<Float>::gpt_to_band(ncol, nbnd, kd.band_lims_gpt, d_af.ptr(), out.d_sfc_alb_dif.ptr(), stream()));
}
