// body_geom.hpp -- device geometry of rigid bodies shared by the flow-move
// and the field evaluators.
#pragma once

#include "common.hpp"

namespace vvhd {

// The pre-test of isPointInContour: false when p is outside the body's box or
// disc (a body of non-positive area always takes the contour test).
__device__ inline bool may_be_invalid(const vvhd_body& B, const double* geo, double px, double py) {
    return B.area <= 0 ||
           !(px < geo[1] || py < geo[2] || px > geo[3] || py > geo[4] ||
             (px - B.cofm[0]) * (px - B.cofm[0]) + (py - B.cofm[1]) * (py - B.cofm[1]) > geo[0]);
}

// Does the contour edge a -> b (b the one before a) cross the ray from p?
__device__ inline bool edge_crosses(double vix, double viy, double vjx, double vjy, double px, double py) {
    return ((viy < vjy) && (viy < py) && (py <= vjy) && ((vjy - viy) * (px - vix) > (vjx - vix) * (py - viy))) ||
           ((viy > vjy) && (viy > py) && (py >= vjy) && ((vjy - viy) * (px - vix) < (vjx - vix) * (py - viy)));
}

// Contour test over the points point(k) of a body's segments on one wave,
// lanes sharing the segments (the parity of the crossings and the first
// nearest segment do not depend on the order); all lanes get the result.
template <typename Point>
__device__ inline int wave_in_contour(const vvhd_body& B, const vvhd_seg* segs, const double* geo, double px, double py,
                                      Point point) {
    if (!may_be_invalid(B, geo, px, py)) return -1;
    bool in = B.area <= 0;
    const int f = B.first_seg, n = B.nseg;
    for (int k0 = 0; k0 < n; k0 += kWave) {
        const int i = k0 + lane_id();
        bool cross = false;
        if (i < n) {
            double vix, viy, vjx, vjy;
            point(segs[f + i], vix, viy);
            point(segs[f + (i ? i - 1 : n - 1)], vjx, vjy);
            cross = edge_crosses(vix, viy, vjx, vjy, px, py);
        }
        in ^= (__popcll(__ballot(cross)) & 1) != 0;
    }
    if (!in) return -1;
    int best = INT32_MAX;
    double bd = DBL_MAX;
    for (int k = lane_id(); k < n; k += kWave) {
        const double dx = segs[f + k].x - px, dy = segs[f + k].y - py;
        const double d2 = dx * dx + dy * dy;
        if (d2 < bd) {
            best = f + k;
            bd = d2;
        }
    }
    for (int o = kWave / 2; o > 0; o >>= 1) {
        const double d = __shfl_xor(bd, o, kWave);
        const int k = __shfl_xor(best, o, kWave);
        if (d < bd || (d == bd && k < best)) {
            bd = d;
            best = k;
        }
    }
    return best == INT32_MAX ? -1 : best;
}

// point_invalid on one wave.
__device__ inline int wave_point_invalid(const vvhd_body& B, const vvhd_seg* segs, const double* geo, double px,
                                         double py) {
    return wave_in_contour(B, segs, geo, px, py, [](const vvhd_seg& s, double& x, double& y) {
        x = s.cx;
        y = s.cy;
    });
}

// TBody::isPointInContour over the corners (TBody.cpp:238-281): index of the
// nearest segment when p is inside the body, else -1.
__device__ inline int point_invalid(const vvhd_body& B, const vvhd_seg* segs, const double* geo, double px, double py) {
    if (!may_be_invalid(B, geo, px, py)) return -1;
    bool in = B.area <= 0;
    const int f = B.first_seg, n = B.nseg;
    for (int i = 0, j = n - 1; i < n; j = i++) {
        const double vix = segs[f + i].cx, viy = segs[f + i].cy, vjx = segs[f + j].cx, vjy = segs[f + j].cy;
        if (edge_crosses(vix, viy, vjx, vjy, px, py))
            in = !in;
    }
    if (!in) return -1;
    int best = -1;
    double bd = DBL_MAX;
    for (int k = 0; k < n; k++) {
        const double dx = segs[f + k].x - px, dy = segs[f + k].y - py;
        const double d2 = dx * dx + dy * dy;
        if (d2 < bd) {
            best = f + k;
            bd = d2;
        }
    }
    return best;
}

}  // namespace vvhd
