// G-point groups of the solver kernels: a work-group is 64 columns (the lanes of each wavefront) x up to
// 16 consecutive g-points of one band, one wavefront each.
#pragma once

#include <algorithm>

#include "common.h"

namespace rrtmgp_hip
{
constexpr int SB_COLS = 64;     // columns per work-group: the lanes of each wavefront
constexpr int SB_GPTS = 16;     // g-points per work-group: one wavefront each, within one band
constexpr int MAX_GROUPS = 256;

struct Groups
{
    int n;
    int start[MAX_GROUPS];
    int count[MAX_GROUPS];
    int band[MAX_GROUPS];
};

// Groups of at most gpts g-points from band limits (2, nbnd), 1-based inclusive; without band limits the
// g-points are cut into consecutive chunks (enough for broadband sums).
inline int make_groups(int64_t ngpt, int64_t nbnd, const int* band_lims, Groups& g, int gpts = SB_GPTS)
{
    g.n = 0;
    auto add = [&](int s, int e, int b) {
        for (int x = s; x < e; x += gpts)
        {
            if (g.n == MAX_GROUPS) return false;
            g.start[g.n] = x;
            g.count[g.n] = std::min(gpts, e - x);
            g.band[g.n] = b;
            ++g.n;
        }
        return true;
    };
    if (band_lims)
    {
        int expect = 1;
        for (int64_t b = 0; b < nbnd; ++b)
        {
            const int s = band_lims[2 * b], e = band_lims[2 * b + 1];
            if (s != expect || e < s || e > ngpt) return arg_error("solver: band limits do not tile the g-points");
            if (!add(s - 1, e, int(b))) return arg_error("solver: too many g-point groups");
            expect = e + 1;
        }
        if (expect != ngpt + 1) return arg_error("solver: band limits do not cover all g-points");
    }
    else if (!add(0, int(ngpt), 0))
        return arg_error("solver: too many g-point groups");
    return RRTMGP_OK;
}

// Groups for a launch over `tiles` column tiles, and the g-points (wavefronts) per work-group they were cut
// for.  A layer step of 16 wavefronts takes a compute unit four times as long as one of 4, one per SIMD: the
// solvers are bound by the issue rate there.  So where the work-groups of 16 would leave compute units idle,
// the bands are cut into halves or quarters as long as the chip holds the work-groups at once.  64 columns x
// 60 layers FP32: SW 125 us in groups of 16, 66 us in groups of 4; LW 80 and 37 us; 250 x 60 FP64: 269 and 110, 165
// and 64 us.  The small work-groups leave g-point fluxes, which are then added in the order of groups of 16.
inline int make_groups_for(int64_t tiles, int64_t ngpt, int64_t nbnd, const int* band_lims, Groups& g, int& gpts)
{
    gpts = SB_GPTS;
    RRTMGP_TRY(make_groups(ngpt, nbnd, band_lims, g, gpts));
    const int64_t cus = device_cu_count();
    while (gpts > 4 && tiles * g.n * 2 <= cus && g.n * 2 <= MAX_GROUPS)
    {
        gpts /= 2;
        RRTMGP_TRY(make_groups(ngpt, nbnd, band_lims, g, gpts));
    }
    return RRTMGP_OK;
}
}  // namespace rrtmgp_hip
