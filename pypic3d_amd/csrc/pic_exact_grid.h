// Exact grids: origins and spacings that make every node coordinate an FP32
// number, so the anchor of an FP32 position can be found in FP32 and agrees
// with the FP64 evaluation floor((x - origin)/spacing) bit for bit.
#pragma once
#include <cmath>

#include "pic_common.h"

namespace {

// Grid constants of an exact grid: on every axis the center line has an FP32
// origin and spacing, the vertex line is the center line shifted by half a
// spacing, and every node org + a*sp with a in [lo, hi + 1] (both lines) is an
// FP32 number (checked on the host).  For a position inside [xlo, xhi) the
// anchor of an FP32 position is then found in FP32 by bracketing it between
// exact node coordinates, and x - node is the correctly rounded difference --
// the value the FP64 evaluation rounds to -- so no FP64 arithmetic is needed
// for the old position.
struct ExactGrid {
    float org_c[3], sp_c[3], isp_c[3], half_sp[3];
    float inv_d[3];
    float xlo[3], xhi[3];
};

// Center-line anchor and offset of x (xlo <= x < xhi): the FP32 estimate is
// within one node of the anchor, one bracketing step against the exact nodes
// corrects it.  The vertex line follows from the half-cell test.
__device__ inline void exact_anchors(float x, float org, float sp, float isp, float half_sp, int& ac, float& dc,
                                     float& nodec, int& av, float& dv) {
    float f = floorf((x - org) * isp);
    float nd = fmaf(f, sp, org);
    const bool below = x < nd, above = x >= nd + sp;
    f = below ? f - 1.0f : (above ? f + 1.0f : f);
    nd = below ? nd - sp : (above ? nd + sp : nd);
    ac = (int)f;
    dc = x - nd;
    nodec = nd;
    const float mid = nd + half_sp;          // vertex node of index ac
    const bool upper = x >= mid;
    av = upper ? ac : ac - 1;
    dv = upper ? x - mid : x - (mid - sp);
}

// Grid constants of the tile kernels.  Anchors are found relative to the first
// node of the tile's field box: an FP32 estimate that is never too small
// (isp_up or bias) and at most one too large, corrected by one comparison with
// the node.  On an exact grid node and offset are FP32 (see ExactGrid); on any
// other they are evaluated in FP64 as the reference does, and a position within
// edge of a face, where its division could round either way, is left to the
// rare list.
struct TileGrid {
    float sp[3], isp[3], isp_up[3], half[3], inv_d[3];
    float bias[3], edge[3];
    // a new FP32 offset from the cell's middle below lim stays in the cell: it is within 2^-22 spacings of the FP64
    // one, and FP64 floor((x - org)/sp) differs from the exact bracket only within a few ulps of a quotient below
    // 2^22, so a band of 2^-19 spacings along the faces covers both
    float lim[3];
    double sp64[3], org64[3], half64[3];
    // the rest of cross_axis' arguments, and the time step: scalar kernel arguments, where
    // a division or conversion in the kernel would hold a vector register across its loops
    double inv_d64[3];
    float org32[3], dt32;
};

// False where a grid's vertex line is not the centre line shifted by half a
// spacing up to rounding (no grid of the solver; the slot-ordered kernel takes
// any lines), or an origin so far that the FP32 estimate may be off by two.  An
// exact grid (make_exact_grid) takes every part: its anchors are exact.
bool make_tile_grid(const PicDesc& d, bool exact, TileGrid& t) {
    for (int a = 0; a < 3; ++a) {
        const double org = d.org_c[a], sp = d.sp_c[a];
        if (!exact) {
            if (!(sp > 0.0) || d.dims[a] > (1 << 20) || !(d.d[a] > 0.0)) return false;
            const double off = d.org_v[a] - org - 0.5 * sp;
            if (std::fabs(off) > 1.0e-7 * sp || std::fabs(d.sp_v[a] - sp) * d.dims[a] > 1.0e-7 * sp) return false;
            if (std::fabs(org) > 4.0e6 * sp) return false;
        }
        t.sp[a] = (float)sp;
        t.isp[a] = (float)(1.0 / sp);
        t.isp_up[a] = t.isp[a] * (1.0f + 0x1p-21f);
        t.half[a] = 0.5f * t.sp[a];
        t.inv_d[a] = (float)(1.0 / d.d[a]);
        // FP32 errors of (x - node) * isp: half an ulp of the node and of x, the rounding of the rest
        t.bias[a] = 0x1p-22f * ((float)(std::fabs(org) / sp) + d.dims[a] + 32.0f);
        t.edge[a] = (float)((0.5 - 0x1p-20) * sp);
        t.lim[a] = (float)((0.5 - 0x1p-19) * sp);
        t.sp64[a] = sp;
        t.org64[a] = org;
        t.half64[a] = 0.5 * sp;
        t.inv_d64[a] = 1.0 / d.d[a];
        t.org32[a] = (float)org;
    }
    t.dt32 = (float)d.dt;
    return true;
}

// Node coordinate of the reference (a*sp + org, both roundings) for an index
// held as a float.
__device__ inline double node_at(float a, double sp, double org) {
#pragma clang fp contract(off)
    return (double)a * sp + org;
}

// Cell of x relative to the field box (first node nb, index fo), offset dc from
// its node, offset q from its middle (the vertex node), whether x is in its
// upper half, and offset dv from the vertex node below x.  False: too near a
// face for the FP64 evaluation to be certain.
template <bool kExact>
__device__ inline bool tile_anchor(const TileGrid& tg, int a, float x, float nb, float fo, float& f, float& dc,
                                   float& q, bool& up, float& dv) {
    if constexpr (kExact) {
        f = floorf((x - nb) * tg.isp_up[a]);
        float nd = fmaf(f, tg.sp[a], nb);
        const float b = x < nd ? 1.0f : 0.0f;
        f -= b;
        nd = fmaf(-b, tg.sp[a], nd);
        const float mid = nd + tg.half[a];
        dc = x - nd;
        q = x - mid;
        up = x >= mid;
        dv = x - (up ? mid : mid - tg.sp[a]);
        return true;
    } else {
        f = floorf(fmaf(x - nb, tg.isp[a], tg.bias[a]));
        double dd = (double)x - node_at(f + fo, tg.sp64[a], tg.org64[a]);
        if (dd < 0.0) {
            f -= 1.0f;
            dd = (double)x - node_at(f + fo, tg.sp64[a], tg.org64[a]);
        }
        const double q64 = dd - tg.half64[a];
        dc = (float)dd;
        q = (float)q64;
        up = q64 >= 0.0;
        dv = (float)(up ? q64 : q64 + tg.sp64[a]);
        return fabsf(q) < tg.edge[a];
    }
}

// Host check for ExactGrid (see its comment); false when any axis fails.
bool make_exact_grid(const PicDesc& d, ExactGrid& eg) {
    for (int a = 0; a < 3; ++a) {
        const double org = d.org_c[a], sp = d.sp_c[a];
        const float o32 = (float)org, s32 = (float)sp, h32 = 0.5f * s32;
        if ((double)o32 != org || (double)s32 != sp || !(sp > 0.0)) return false;
        if (d.sp_v[a] != sp || d.org_v[a] != org + 0.5 * sp || (double)(o32 + h32) != d.org_v[a]) return false;
        if (d.dims[a] > (1 << 20)) return false;
        const int lo = -d.dims[a] - 4, hi = 2 * d.dims[a] + 4;
        for (int n = lo - 1; n <= hi + 1; ++n) {
            const double node = (double)n * sp + org;                   // exact: 24-bit operands
            const float n32 = std::fma((float)n, s32, o32);
            if ((double)n32 != node || (double)(n32 + h32) != node + 0.5 * sp) return false;
        }
        eg.org_c[a] = o32;
        eg.sp_c[a] = s32;
        eg.isp_c[a] = (float)(1.0 / sp);
        eg.half_sp[a] = h32;
        eg.inv_d[a] = (float)(1.0 / d.d[a]);
        eg.xlo[a] = std::fma((float)lo, s32, o32);
        eg.xhi[a] = std::fma((float)hi, s32, o32);
    }
    return true;
}

}  // namespace
