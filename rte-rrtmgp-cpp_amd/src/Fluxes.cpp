// Flux reductions (reference src_cuda/Fluxes.cu:31-136 / src/Fluxes.cpp:87-197).
#include "Fluxes.h"

#include "Optical_props.h"
#include "hip_dispatch.h"

using rrtmgp_cpp::hip_check;
using rrtmgp_cpp::stream;

Fluxes_broadband_gpu::Fluxes_broadband_gpu(const int ncol, const int nlev) :
    flux_up({ncol, nlev}), flux_dn({ncol, nlev}), flux_dn_dir({ncol, nlev}), flux_net({ncol, nlev})
{}

namespace
{
// Bands that follow each other from g-point 1 to ngpt.
bool consecutive(const Array<int,2>& lims, const int nbnd, const int ngpt)
{
    int next = 1;
    for (int b = 1; b <= nbnd; ++b)
    {
        if (lims({1, b}) != next || lims({2, b}) < next) return false;
        next = lims({2, b}) + 1;
    }
    return next == ngpt + 1;
}
}

// One pass over the fluxes, except for bands with gaps, overlaps or another order, which are summed band by
// band after a broadband pass.
void reduce_fluxes(const int ncol, const int nlev, const int ngpt, const Float* up, const Float* dn,
                   const Float* dir, const Optical_props_gpu* bands, const Flux_outputs& o)
{
    const int nbnd = bands ? bands->get_nband() : 0;
    const bool fused = !bands || consecutive(bands->get_band_lims_gpoint(), nbnd, ngpt);
    const int* bl = bands ? bands->get_band_lims_gpoint_gpu().ptr() : nullptr;
    hip_check(K<Float>::reduce_fluxes(ncol, nlev, ngpt, nbnd, fused ? bl : nullptr, up, dn, dir, o.up, o.dn, o.net,
                                      o.dir, o.bnd_up, o.bnd_dn, o.bnd_net, o.bnd_dir, stream()));
    if (fused) return;
    Array_gpu<Float,3> tmp_up, tmp_dn;
    Float* bu = o.bnd_up;
    Float* bd = o.bnd_dn;
    if (!bu) { tmp_up.set_dims({ncol, nlev, nbnd}); bu = tmp_up.ptr(); }
    if (!bd) { tmp_dn.set_dims({ncol, nlev, nbnd}); bd = tmp_dn.ptr(); }
    hip_check(K<Float>::sum_byband(ncol, nlev, ngpt, nbnd, bl, up, bu, stream()));
    hip_check(K<Float>::sum_byband(ncol, nlev, ngpt, nbnd, bl, dn, bd, stream()));
    if (o.bnd_net) hip_check(K<Float>::net_broadband(ncol, int64_t(nlev) * nbnd, bd, bu, o.bnd_net, stream()));
    if (dir && o.bnd_dir) hip_check(K<Float>::sum_byband(ncol, nlev, ngpt, nbnd, bl, dir, o.bnd_dir, stream()));
}

void Fluxes_broadband_gpu::reduce(const Array_gpu<Float,3>& up, const Array_gpu<Float,3>& dn,
                                  const std::unique_ptr<Optical_props_arry_gpu>&, const Bool)
{
    Flux_outputs o;
    o.up = flux_up.ptr(); o.dn = flux_dn.ptr(); o.net = flux_net.ptr();
    reduce_fluxes(up.dim(1), up.dim(2), up.dim(3), up.ptr(), dn.ptr(), nullptr, nullptr, o);
}

void Fluxes_broadband_gpu::reduce(const Array_gpu<Float,3>& up, const Array_gpu<Float,3>& dn,
                                  const Array_gpu<Float,3>& dir,
                                  const std::unique_ptr<Optical_props_arry_gpu>&, const Bool)
{
    Flux_outputs o;
    o.up = flux_up.ptr(); o.dn = flux_dn.ptr(); o.net = flux_net.ptr(); o.dir = flux_dn_dir.ptr();
    reduce_fluxes(up.dim(1), up.dim(2), up.dim(3), up.ptr(), dn.ptr(), dir.ptr(), nullptr, o);
}

Fluxes_byband_gpu::Fluxes_byband_gpu(const int ncol, const int nlev, const int nbnd) :
    Fluxes_broadband_gpu(ncol, nlev), bnd_flux_up({ncol, nlev, nbnd}), bnd_flux_dn({ncol, nlev, nbnd}),
    bnd_flux_dn_dir({ncol, nlev, nbnd}), bnd_flux_net({ncol, nlev, nbnd})
{}

void Fluxes_byband_gpu::reduce(const Array_gpu<Float,3>& up, const Array_gpu<Float,3>& dn,
                               const std::unique_ptr<Optical_props_arry_gpu>& p, const Bool)
{
    Flux_outputs o;
    o.up = get_flux_up().ptr(); o.dn = get_flux_dn().ptr(); o.net = get_flux_net().ptr();
    o.bnd_up = bnd_flux_up.ptr(); o.bnd_dn = bnd_flux_dn.ptr(); o.bnd_net = bnd_flux_net.ptr();
    reduce_fluxes(up.dim(1), up.dim(2), up.dim(3), up.ptr(), dn.ptr(), nullptr, p.get(), o);
}

void Fluxes_byband_gpu::reduce(const Array_gpu<Float,3>& up, const Array_gpu<Float,3>& dn,
                               const Array_gpu<Float,3>& dir,
                               const std::unique_ptr<Optical_props_arry_gpu>& p, const Bool)
{
    Flux_outputs o;
    o.up = get_flux_up().ptr(); o.dn = get_flux_dn().ptr(); o.net = get_flux_net().ptr();
    o.dir = get_flux_dn_dir().ptr();
    o.bnd_up = bnd_flux_up.ptr(); o.bnd_dn = bnd_flux_dn.ptr(); o.bnd_net = bnd_flux_net.ptr();
    o.bnd_dir = bnd_flux_dn_dir.ptr();
    reduce_fluxes(up.dim(1), up.dim(2), up.dim(3), up.ptr(), dn.ptr(), dir.ptr(), p.get(), o);
}

void compute_heating_rate(const Array_gpu<Float,2>& up, const Array_gpu<Float,2>& dn,
                          const Array_gpu<Float,2>& p_lev, Array_gpu<Float,2>& hr)
{
    hip_check(K<Float>::heating_rate(up.dim(1), up.dim(2) - 1, up.ptr(), dn.ptr(), p_lev.ptr(), hr.ptr(), stream()));
}
