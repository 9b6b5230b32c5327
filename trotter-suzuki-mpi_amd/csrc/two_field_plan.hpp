// two_field_plan.hpp -- tile shapes of the passes over two fields
// (pair_tile_kernel.hpp, adjoint_tile_kernel.hpp).
#pragma once
#include <algorithm>
#include <cmath>

#include "tile_kernel.hpp"

namespace tsmi {

// Rows per wave and waves per workgroup, tile extents and counts.
struct TwoFieldPlan {
    int r = 0, nw = 0, cols = 0, rows = 0, strips = 0, segs = 0;
    double us = 1e30;                // modelled time per step
};

// us of a row of both fields with several waves per SIMD; planes of the kernel
// precision that a launch moves.
struct TwoFieldCost {
    double row;
    int planes;
    bool wide;                       // 4 rows x 16 waves is compiled (FP32)
};

// The compiled instances: FP32 4 rows x 8 waves, 8 x 8 and (wide) 4 x 16, FP64 4 x 8
// and 4 x 4.
//
// The shape of a pass of `steps` steps is the one with the least modelled time.  A
// launch costs 4.5 us and its bytes (at 6.5 TB/s); a step costs each SIMD its rows
// (more for a wave alone) and 0.5 us of exchanges.  Measured around it, the two
// components of a periodic lattice in real time, us per step: 256^2 FP32 4 rows x
// 8 waves 7.9, 5.6, 4.9 for 1, 2, 3 steps, 8 x 8 12.6, 9.3, 8.1; 1024^2 FP32 4 x 8
// 13.9, 13.0, 19.2, 8 x 8 15.8, 12.2, 17.1 (3 steps: more than one workgroup per
// compute unit); 512^2 FP64 4 x 8 10.9, 8.5, 12.7.  4 rows x 16 waves, the tile of
// 8 x 8 with twice the waves to hide each other's latency, 119 VGPRs at most: 1024^2
// 12.1 -> 11.1, 800^2 10.7 -> 9.7.
inline TwoFieldPlan two_field_plan(int W, int H, int esz, int steps, bool wrap, const TwoFieldCost &cost) {
    static const int shapes[2][3][2] = {{{4, 8}, {8, 8}, {4, 16}}, {{4, 8}, {4, 4}, {0, 0}}};
    TwoFieldPlan best;
    const int a = kApron * steps;
    const double x = 0.5, t0 = 4.5 + (double)W * H * cost.planes * esz / 6.5e6;
    for (const auto &sh : shapes[esz == 4 ? 0 : 1]) {
        if (sh[1] == 0 || (sh[1] == 16 && !cost.wide)) continue;
        TwoFieldPlan p;
        p.r = sh[0];
        p.nw = sh[1];
        p.cols = kTileCols - 2 * a;
        p.rows = p.nw * p.r - 2 * a;
        if (p.cols < 2 || p.rows < 2) continue;
        p.strips = (W + p.cols - 1) / p.cols;
        p.segs = (H + p.rows - 1) / p.rows;
        const double n = p.strips * p.segs / 256.0;                 // workgroups per compute unit
        const double per_cu = n < 6 ? std::ceil(n) : n + 0.5;       // ... on the busiest one
        const double most = p.nw == 16 || (wrap && esz == 4 && p.r == 4) ? 4.0 : 2.0;
        const double waves = std::min(per_cu * p.nw / 4.0, most);   // waves per SIMD
        p.us = t0 / steps + per_cu * p.nw * p.r / 4.0 * cost.row * (1 + 0.6 / waves) + x;
        if (p.us < best.us) best = p;
    }
    return best;
}

// The number of steps per pass, at most `most`, with the least modelled time.
inline int two_field_best_steps(int W, int H, int esz, int most, bool wrap, const TwoFieldCost &cost) {
    int k = 1;
    double us = 1e30;
    for (int s = 1; s <= std::min(most, 6); ++s) {
        const TwoFieldPlan p = two_field_plan(W, H, esz, s, wrap, cost);
        if (p.us < us) {
            us = p.us;
            k = s;
        }
    }
    return k;
}

}  // namespace tsmi
