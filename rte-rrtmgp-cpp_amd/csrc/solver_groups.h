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

// Groups from band limits (2, nbnd), 1-based inclusive; without band limits the g-points are cut
// into consecutive chunks (enough for broadband sums).
inline int make_groups(int64_t ngpt, int64_t nbnd, const int* band_lims, Groups& g)
{
    g.n = 0;
    auto add = [&](int s, int e, int b) {
        for (int x = s; x < e; x += SB_GPTS)
        {
            if (g.n == MAX_GROUPS) return false;
            g.start[g.n] = x;
            g.count[g.n] = std::min(SB_GPTS, e - x);
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
}  // namespace rrtmgp_hip
