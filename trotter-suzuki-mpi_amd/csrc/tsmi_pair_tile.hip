// tsmi_pair_tile.hip -- planning and launching the two-component tile passes
// (pair_tile_kernel.hpp).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstring>
#include <string>

#include "common.hpp"
#include "pair_context.hpp"
#include "pair_tile_kernel.hpp"
#include "two_field_plan.hpp"
#include "tsmi_hip.h"

using namespace tsmi;

namespace {

// One scaled form for both components on both axes.
bool one_form(const tsmi_pair *p) { return p->c[0]->mode == p->c[1]->mode && p->c[0]->mode >= 0; }

// Modelled us of a row of both components, and planes moved per launch.
TwoFieldCost cost(int esz, bool wide) {
    return esz == 4 ? TwoFieldCost{0.27, 10, wide} : TwoFieldCost{0.53, 10, false};
}

template <typename T, bool IMAG, int R, int NW, bool WRAP>
int launch_kernel(tsmi_pair *p, const PairTileParams<T> &q, const TwoFieldPlan &g) {
    // one scaled form for both components on both axes, or both factors
    const int mode = p->c[0]->mode == p->c[1]->mode ? p->c[0]->mode : -1;
    const dim3 grid(g.strips * g.segs), block(NW * kWave);
    hipStream_t s = p->c[0]->stream;
    // FP64 tiles of 8 waves with an edge: the general form for all of them, as both
    // forms in one kernel spill
    if constexpr (!WRAP && sizeof(T) == 8 && NW == 8) {
        hipLaunchKernelGGL((pair_tile_kernel<T, IMAG, -1, R, NW, WRAP>), grid, block, 0, s, q);
    } else if constexpr (IMAG) {   // form A always
        hipLaunchKernelGGL((pair_tile_kernel<T, true, 0, R, NW, WRAP>), grid, block, 0, s, q);
    } else {
        if (mode == 0) hipLaunchKernelGGL((pair_tile_kernel<T, false, 0, R, NW, WRAP>), grid, block, 0, s, q);
        else if (mode == 1) hipLaunchKernelGGL((pair_tile_kernel<T, false, 1, R, NW, WRAP>), grid, block, 0, s, q);
        else hipLaunchKernelGGL((pair_tile_kernel<T, false, -1, R, NW, WRAP>), grid, block, 0, s, q);
    }
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) return set_error(TSMI_E_HIP, std::string("pair_tile_kernel: ") + hipGetErrorString(e));
    return TSMI_OK;
}

template <typename T, bool IMAG, int R, int NW>
int launch(tsmi_pair *p, const PairTileParams<T> &q, const TwoFieldPlan &g) {
    return q.nx ? launch_kernel<T, IMAG, R, NW, true>(p, q, g) : launch_kernel<T, IMAG, R, NW, false>(p, q, g);
}

template <typename T, bool IMAG>
int launch_shape(tsmi_pair *p, const PairTileParams<T> &q, const TwoFieldPlan &g) {
    if constexpr (sizeof(T) == 4) {
        if (g.nw == 16) {   // WRAP and one form only: the other kernels need more registers
            hipStream_t s = p->c[0]->stream;
            const dim3 grid(g.strips * g.segs), block(16 * kWave);
            if constexpr (IMAG) {
                hipLaunchKernelGGL((pair_tile_kernel<T, true, 0, 4, 16, true>), grid, block, 0, s, q);
            } else {
                if (p->c[0]->mode == 0)
                    hipLaunchKernelGGL((pair_tile_kernel<T, false, 0, 4, 16, true>), grid, block, 0, s, q);
                else
                    hipLaunchKernelGGL((pair_tile_kernel<T, false, 1, 4, 16, true>), grid, block, 0, s, q);
            }
            const hipError_t e = hipGetLastError();
            if (e != hipSuccess) return set_error(TSMI_E_HIP, std::string("pair_tile_kernel: ") + hipGetErrorString(e));
            return TSMI_OK;
        }
        return g.r == 4 ? launch<T, IMAG, 4, 8>(p, q, g) : launch<T, IMAG, 8, 8>(p, q, g);
    } else return g.nw == 8 ? launch<T, IMAG, 4, 8>(p, q, g) : launch<T, IMAG, 4, 4>(p, q, g);
}

// What is pending after an imaginary-time step in slot p->slot's partial sums,
// whose rotation is by var.
PairNorm pending(tsmi_pair *p, double var, bool rabi) {
    PairNorm q;
    std::memset(&q, 0, sizeof(q));
    q.part = p->tile_part + (size_t)p->slot * kPairSums * (size_t)p->part_cap;
    q.n = p->tile_n + p->slot;
    q.cap = p->part_cap;
    q.norm_in = norms(p);
    q.norm_out = p->dv + 4 + 2 * (1 - p->norm_slot);
    rabi_coefs(p, var, &q.cc, &q.cs_r, &q.cs_i);
    q.rabi = rabi ? 1 : 0;
    q.dxdy = p->c[0]->d.delta_x * p->c[0]->d.delta_y;
    q.tot_norm = p->tot_norm;
    return q;
}

// How a pass reads the state: the closed tile, the periodic lattice, or the tile
// whose halo exchange has not been run (one step; seam_off).
enum How { kClosed, kWrap, kSeam };

// `steps` steps; the rotation after the last of them is by var (1 after the
// others).  first: nothing pending from a step before (imaginary time).
template <typename T>
int pass(tsmi_pair *p, int steps, How how, double var, bool rabi, bool first) {
    const bool wrap = how == kWrap;
    PairTileParams<T> q;
    std::memset(&q, 0, sizeof(q));
    const int cur = p->c[0]->cur, nb = 1 - cur;
    for (int i = 0; i < 2; ++i) {
        tsmi_ctx *c = p->c[i];
        q.in_re[i] = (const T *)c->psi_re[cur];
        q.in_im[i] = (const T *)c->psi_im[cur];
        q.out_re[i] = (T *)c->psi_re[nb];
        q.out_im[i] = (T *)c->psi_im[nb];
        q.ph[i] = (const T *)c->ph;
        q.mH[i] = (T)c->mH; q.tH[i] = (T)c->tH; q.mV[i] = (T)c->mV; q.tV[i] = (T)c->tV;
        q.unH[i] = (T)c->unH; q.unV[i] = (T)c->unV;
        q.c_self[i] = (T)c->c_nl_s;
        q.mag[i] = p->imag ? 1.0 : c->corr_abs;
    }
    q.c_ab = (T)p->c_ab;
    q.W = p->W; q.H = p->H; q.pitch = p->pitch;
    q.nx = wrap ? p->c[0]->d.dim_x : 0;
    q.ny = wrap ? p->c[0]->d.dim_y : 0;
    q.seam = how == kSeam;
    q.px = p->c[0]->d.periodic_x != 0; q.py = p->c[0]->d.periodic_y != 0;
    q.steps = steps;
    const TwoFieldPlan g = two_field_plan(p->W, p->H, p->esz, steps, wrap, cost(p->esz, wrap && one_form(p)));
    if (g.r == 0) return set_error(TSMI_E_INVALID, "pair tile pass: no tile for this many steps");
    q.n_strips = g.strips; q.cols = g.cols; q.rows = g.rows;
    q.ix0 = p->ix0; q.ix1 = p->ix1; q.iy0 = p->iy0; q.iy1 = p->iy1;
    q.rabi = rabi ? 1 : 0;
    int st;
    if (!p->imag) {
        rabi_coefs(p, 1.0, &q.cc, &q.cs_r, &q.cs_i);
        rabi_coefs(p, var, &q.cc2, &q.cs_r2, &q.cs_i2);
        st = launch_shape<T, false>(p, q, g);
    } else {
        if (!first) {
            q.pend = pending(p, 1.0, rabi);
            p->norm_slot = 1 - p->norm_slot;
        }
        double cc;
        rabi_coefs(p, var, &cc, &q.s_r, &q.s_i);
        p->slot = 1 - p->slot;
        q.part_out = p->tile_part + (size_t)p->slot * kPairSums * (size_t)p->part_cap;
        q.n_out = p->tile_n + p->slot;
        q.cap = p->part_cap;
        st = launch_shape<T, true>(p, q, g);
    }
    if (!st) p->c[0]->cur = p->c[1]->cur = nb;
    return st;
}

int tile_pass(tsmi_pair *p, int steps, How how, double var, bool rabi, bool first) {
    return p->esz == 4 ? pass<float>(p, steps, how, var, rabi, first) : pass<double>(p, steps, how, var, rabi, first);
}

// A call of n steps that runs on the doubly periodic lattice between its first and
// its last step, E read from the inner cells, as FP32 real time always does with two
// steps per pass; elsewhere only when the tables' halos repeat them.
bool wraps(const tsmi_pair *p, int n) {
    const tsmi_desc &d = p->c[0]->d;
    return d.periodic_x && d.periodic_y && d.dim_x % 2 == 0 && d.dim_y % 2 == 0 && n >= 3 &&
           ((p->esz == 4 && !p->imag) || (p->c[0]->e_wraps && p->c[1]->e_wraps));
}

// The renormalisation after the last step.
template <typename T>
int finish(tsmi_pair *p, double var, bool rabi) {
    PairNorm q = pending(p, var, rabi);
    tsmi_ctx *a = p->c[0], *b = p->c[1];
    const int cur = a->cur, blocks = (int)std::min<long>(kFinishBlocks, ((long)p->W * p->H + 1023) / 1024);
    p->slot = 1 - p->slot;
    double *part_out = p->tile_part + (size_t)p->slot * kPairSums * (size_t)p->part_cap;
    int *n_out = p->tile_n + p->slot;
    hipLaunchKernelGGL((pair_finish_kernel<T>), dim3(blocks), dim3(256), 0, a->stream, (T *)a->psi_re[cur],
                       (T *)a->psi_im[cur], (T *)b->psi_re[cur], (T *)b->psi_im[cur], p->W, p->H, p->pitch, p->ix0,
                       p->ix1, p->iy0, p->iy1, q, part_out, n_out);
    hipError_t e = hipGetLastError();
    if (e == hipSuccess && rabi) {
        q.part = part_out;
        q.n = n_out;
        hipLaunchKernelGGL(pair_targets_kernel<>, dim3(1), dim3(kWave), 0, a->stream, q);
        e = hipGetLastError();
    }
    if (e != hipSuccess) return set_error(TSMI_E_HIP, std::string("pair_finish_kernel: ") + hipGetErrorString(e));
    p->norm_slot = 1 - p->norm_slot;
    return TSMI_OK;
}

}  // namespace

namespace tsmi {

int pair_tile_blocks(const tsmi_pair *p) {
    const TwoFieldPlan a = two_field_plan(p->W, p->H, p->esz, 1, false, cost(p->esz, false)),
                       b = two_field_plan(p->W, p->H, p->esz, 1, true, cost(p->esz, one_form(p)));
    return std::max({a.strips * a.segs, b.strips * b.segs, kFinishBlocks});
}

// No segment height or steps per pass asked for, offsets within 31 bits, and a
// lattice small enough that the row latency (real time) or the ticketed
// reductions (imaginary time) bound the streaming passes; us per step, streamed
// against tiles, doubly periodic / closed: real FP32 100^2 36 / 33 -> 5.5 / 5.8,
// 512^2 37 / 33 -> 7.8 / 8.0, 1240^2 38 / 35 -> 22 / 29; FP64 100^2 61 / 55 -> 7.7 /
// 8.6, 1240^2 64 / 59 -> 40 / 43; imaginary FP32 100^2 63 / 58 -> 11 / 12, 1240^2
// 263 / 257 -> 26 / 33, FP64 1240^2 279 / 275 -> 54 / 54.
// Narrow and flat lattices leave most of their tiles idle: real FP32 2 x 400000 204 /
// 563, 8 x 10^5 the other way round 15 / 22, 20 x 15000 29 / 22; imaginary FP64 2 x
// 400000 811 / 5884, 10 x 40000 289 / 143, FP32 3 x 300000 291 / 177.
bool pair_tiles_fit(const tsmi_pair *p, int tile_rows, int sweeps) {
    const long most = p->imag ? 5L << 20 : 3L << 19, area = p->imag ? 2 * most : most + most / 4;
    return tile_rows == 0 && sweeps == 0 && p->H > 1 && (long)p->W * p->H <= most && tile_area(p->W, p->H) <= area &&
           (long)p->pitch * p->c[0]->Hd * p->esz < (1L << 31);
}

// FP64 in real time where tiles have an edge gives out earlier: closed 1100^2 36.4 /
// 31.9, 1200^2 37.5 / 39.6; periodic in x 1100^2 41.9 / 32.9, 1200^2 42.4 / 42.4.
bool pair_tiles_run(const tsmi_pair *p, int n) {
    return p->tiles && (p->imag || p->esz == 4 || wraps(p, n) || (long)p->W * p->H <= 19L << 16);
}

int pair_tile_evolve(tsmi_pair *p, int n, bool rabi) {
    if (n <= 0) return TSMI_OK;
    const tsmi_desc &d = p->c[0]->d;
    const bool closed = !d.periodic_x && !d.periodic_y;
    const bool wrap = wraps(p, n);
    const int most = p->imag || !(closed || wrap) ? 1 : n;
    int i = 0, st = TSMI_OK;
    // n steps from step i on; the call's last rotation is by 1/2 (src/solver.cpp:222-225)
    auto passes = [&](int m, How how) {
        const int k = two_field_best_steps(p->W, p->H, p->esz, std::min(m, most), how == kWrap,
                                           cost(p->esz, how == kWrap && one_form(p)));
        const int q = (m + k - 1) / k;
        for (int j = 0; j < q && !st; ++j) {
            const int s = m / q + (j < m % q ? 1 : 0);
            i += s;
            st = tile_pass(p, s, how, i == n ? 0.5 : 1.0, rabi, i == s);
        }
    };
    if (closed) {
        passes(n, kClosed);
    } else if (wrap) {
        passes(1, kClosed);
        passes(n - 2, kWrap);
        if (!st) passes(1, kClosed);
    } else {
        // mixed axes; odd periodic extents, where the pair pattern of a halo cell
        // differs from that of the cell it mirrors; a call of two steps
        for (int j = 0; j < n && !st; ++j) passes(1, j == 0 ? kClosed : kSeam);
    }
    if (!st && p->imag) st = p->esz == 4 ? finish<float>(p, 0.5, rabi) : finish<double>(p, 0.5, rabi);
    return st;
}

}  // namespace tsmi
