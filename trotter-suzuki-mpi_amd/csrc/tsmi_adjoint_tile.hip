// tsmi_adjoint_tile.hip -- planning and launching the reverse sweep's tile passes
// (adjoint_tile_kernel.hpp).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstring>
#include <string>

#include "adjoint_tile_kernel.hpp"
#include "common.hpp"
#include "context.hpp"
#include "two_field_plan.hpp"
#include "tsmi_hip.h"

using namespace tsmi;

namespace {

// Modelled us of a row of both fields, and planes moved per launch: two states in
// and out, E, and the FP64 gradient in and out.
TwoFieldCost cost(const tsmi_ctx *c) {
    const bool wide = c->c_nl == 0.0 && c->c_lhy == 0.0 && c->mode >= 0;   // 120 VGPRs; the others need more
    return c->esz == 4 ? TwoFieldCost{0.27, 14, wide} : TwoFieldCost{0.40, 12, false};
}

template <typename T, bool NL, int R, int NW, bool WRAP>
int launch_kernel(tsmi_ctx *c, const AdjTileParams<T> &q, int blocks) {
    const dim3 grid(blocks), block(NW * kWave);
    // tiles with an edge, 8 FP64 waves: as in tsmi_pair_tile.hip
    if constexpr (NW == 16) {
        if (c->mode == 0) hipLaunchKernelGGL((adj_tile_kernel<T, NL, 0, R, NW, WRAP>), grid, block, 0, c->stream, q);
        else hipLaunchKernelGGL((adj_tile_kernel<T, NL, 1, R, NW, WRAP>), grid, block, 0, c->stream, q);
    } else if constexpr (!WRAP && sizeof(T) == 8 && NW == 8) {
        hipLaunchKernelGGL((adj_tile_kernel<T, NL, -1, R, NW, WRAP>), grid, block, 0, c->stream, q);
    } else {
        if (c->mode == 0) hipLaunchKernelGGL((adj_tile_kernel<T, NL, 0, R, NW, WRAP>), grid, block, 0, c->stream, q);
        else if (c->mode == 1) hipLaunchKernelGGL((adj_tile_kernel<T, NL, 1, R, NW, WRAP>), grid, block, 0, c->stream, q);
        else hipLaunchKernelGGL((adj_tile_kernel<T, NL, -1, R, NW, WRAP>), grid, block, 0, c->stream, q);
    }
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) return set_error(TSMI_E_HIP, std::string("adj_tile_kernel: ") + hipGetErrorString(e));
    return TSMI_OK;
}

template <typename T, bool NL, bool WRAP>
int launch(tsmi_ctx *c, const AdjTileParams<T> &q, const TwoFieldPlan &g) {
    const int blocks = g.strips * g.segs;
    if constexpr (sizeof(T) == 4 && !NL) {
        if (g.nw == 16) return launch_kernel<T, NL, 4, 16, WRAP>(c, q, blocks);
    }
    if constexpr (sizeof(T) == 4)
        return g.r == 4 ? launch_kernel<T, NL, 4, 8, WRAP>(c, q, blocks) : launch_kernel<T, NL, 8, 8, WRAP>(c, q, blocks);
    else
        return g.nw == 8 ? launch_kernel<T, NL, 4, 8, WRAP>(c, q, blocks) : launch_kernel<T, NL, 4, 4, WRAP>(c, q, blocks);
}

template <typename T>
int pass(tsmi_ctx *c, int steps, const AdjTileIo &io) {
    AdjTileParams<T> q;
    std::memset(&q, 0, sizeof(q));
    const bool wrap = c->d.periodic_x != 0;
    for (int i = 0; i < 2; ++i) {
        q.in_re[i] = (const T *)io.in[i][0];
        q.in_im[i] = (const T *)io.in[i][1];
        q.out_re[i] = (T *)io.out[i][0];
        q.out_im[i] = (T *)io.out[i][1];
        q.mH[i] = (T)c->amH; q.tH[i] = (T)c->atH; q.mV[i] = (T)c->amV; q.tV[i] = (T)c->atV;
        q.unH[i] = (T)c->aunH; q.unV[i] = (T)c->aunV;
    }
    q.e_re = (const T *)c->e_re;
    q.e_im = (const T *)c->e_im;
    q.grad = c->grad;
    q.W = c->W; q.H = c->H; q.pitch = c->pitch;
    q.nx = wrap ? c->d.dim_x : 0;
    q.ny = wrap ? c->d.dim_y : 0;
    q.steps = steps;
    const TwoFieldPlan g = two_field_plan(c->W, c->H, c->esz, steps, wrap, cost(c));
    if (g.r == 0) return set_error(TSMI_E_INVALID, "reverse tile pass: no tile for this many steps");
    q.n_strips = g.strips; q.cols = g.cols; q.rows = g.rows;
    q.c_nl = (T)c->c_nl_s; q.c_lhy = (T)c->c_lhy_s;
    q.gscale = c->d.delta_t * c->corr_abs;
    if (c->c_nl != 0.0 || c->c_lhy != 0.0)
        return wrap ? launch<T, true, true>(c, q, g) : launch<T, true, false>(c, q, g);
    return wrap ? launch<T, false, true>(c, q, g) : launch<T, false, false>(c, q, g);
}

}  // namespace

namespace tsmi {

// Closed axes or even doubly periodic ones whose E repeats its inner cells on the halo
// (the passes read it there; the streamed steps read the halo itself), no segment height or steps per pass
// asked for, and a lattice where tiles measured faster; us per reverse step,
// streamed against tiles, linear / nonlinear: closed FP32 100^2 20.7 / 29.2 -> 4.3 /
// 5.3, 1024^2 23.7 / 31.7 -> 11.2 / 15.8, 1200^2 25.3 / 32.1 -> 15.3 / 23.0; FP64
// 100^2 15.9 / 21.3 -> 5.3 / 6.7, 800^2 20.7 / 25.4 -> 15.1 / 18.1; periodic ones
// gain the exchanges of both states besides.  Narrow and flat lattices leave most of
// their tiles idle: FP32 2 x 400000 379 / 546, 3 x 300000 the other way round 20 / 59, 20 x
// 15000 42 / 20, FP64 10 x 40000 54 / 73.
bool adjoint_tiles_run(const tsmi_ctx *c) {
    const bool closed = !c->d.periodic_x && !c->d.periodic_y;
    const bool even = c->d.periodic_x && c->d.periodic_y && c->d.dim_x % 2 == 0 && c->d.dim_y % 2 == 0 &&
                      c->e_wraps;
    const long most = c->esz == 4 ? 3L << 19 : 3L << 18;
    return (closed || even) && c->d.tile_rows == 0 && c->d.sweeps == 0 && c->H > 1 &&
           (long)c->W * c->H <= most && tile_area(c->W, c->H) <= most + most / 4 && (long)c->pitch * c->Hd * 8 < (1L << 31);
}

int adjoint_tile_steps(const tsmi_ctx *c, int most) {
    return two_field_best_steps(c->W, c->H, c->esz, most, c->d.periodic_x != 0, cost(c));
}

int adjoint_tile_pass(tsmi_ctx *c, int steps, const AdjTileIo &io) {
    return c->esz == 4 ? pass<float>(c, steps, io) : pass<double>(c, steps, io);
}

}  // namespace tsmi
