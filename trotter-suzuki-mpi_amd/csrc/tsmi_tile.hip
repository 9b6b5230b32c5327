// tsmi_tile.hip -- planning and launching the tile passes (tile_kernel.hpp):
// several real-time steps of a small or medium lattice per launch.
#include "tsmi_hip.h"

#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <complex>
#include <cstring>
#include <string>

#include "common.hpp"
#include "context.hpp"
#include "frame.hpp"
#include "tile_kernel.hpp"
#include "tile_plan.hpp"

using namespace tsmi;

namespace {

// Rows per wave of the compiled instances, of 4 or 8 waves each; FP32 with 4 rows
// also of 16 (80 VGPRs).  No 8 rows in FP32: their tiles, 32 and 64 rows high, are
// those of 4 rows with twice the waves, which hide each other's latency.
constexpr int kRows32[] = {4, 12}, kRows64[] = {4, 6, 8};

// The tile shape of a pass of `steps` steps: the one with the least modelled time.
// A launch costs about 5 us whatever it does; a step costs each SIMD its rows
// (about 0.17 us a row in FP32, 0.27 in FP64 with several waves per SIMD, up to
// 60% more for a wave alone) and 0.35 us of exchanges.  Measured around it, us
// per step: 256^2 FP64 4 rows x 8 waves 6.9, 4.9, 4.4 for 1, 2, 3 steps, 8 x 8
// 10.7, 7.9, 7.1; 1100^2 FP32 4 x 16 9.8, 6.7, 8.7 (3 steps: more than one
// workgroup per compute unit), 12 x 8 12.3, 8.7, 7.4, 7.2, 9.5 (5 steps).
TilePlan plan(const std::pair<int, int> *size, size_t count, int esz, int steps) {
    TilePlan best;
    const int a = kApron * steps;
    const int *rr = esz == 4 ? kRows32 : kRows64, n_rr = esz == 4 ? 2 : 3;
    const double c_row = esz == 4 ? 0.17 : 0.27, x = 0.35, t0 = 5.0;
    for (int i = 0; i < n_rr; ++i)
        for (int nw : {4, 8, 16}) {
            if (nw == 16 && (esz != 4 || i != 0)) continue;
            TilePlan p;
            p.r = rr[i];
            p.nw = nw;
            const int cols = kTileCols - 2 * a, rows = nw * p.r - 2 * a;
            if (cols < 2 || rows < 2) continue;
            long tiles = 0;
            for (size_t j = 0; j < count; ++j)
                tiles += (long)((size[j].first + cols - 1) / cols) * ((size[j].second + rows - 1) / rows);
            const double n = tiles / 256.0;                          // workgroups per compute unit
            const double per_cu = n < 6 ? std::ceil(n) : n + 0.5;    // ... on the busiest one
            const double waves = std::min(per_cu * nw / 4.0, nw == 16 ? 4.0 : 3.0);   // waves per SIMD
            p.us = t0 / steps + per_cu * nw * p.r / 4.0 * c_row * (1 + 0.6 / waves) + x;
            if (p.us < best.us) best = p;
        }
    return best;
}

int best_steps(const std::pair<int, int> *size, size_t count, int esz, int most) {
    int k = 1;
    double us = 1e30;
    for (int s = 1; s <= std::min(most, 8); ++s) {
        const TilePlan p = plan(size, count, esz, s);
        if (p.us < us) {
            us = p.us;
            k = s;
        }
    }
    return k;
}

// Launches tile_kernel, or (items) tile_batch_kernel.
template <typename T, bool LHY, int MODE, int R, int NW>
void launch(const TilePlan &g, int blocks, const TileParams<T> *p, const int2 *items, hipStream_t s) {
    if constexpr (MODE != kTileImag)
        if (items) {
            hipLaunchKernelGGL((tile_batch_kernel<T, LHY, MODE, R, NW>), dim3(blocks), dim3(g.nw * kWave), 0, s, p, items);
            return;
        }
    hipLaunchKernelGGL((tile_kernel<T, LHY, MODE, R, NW>), dim3(blocks), dim3(g.nw * kWave), 0, s, *p);
}

template <typename T, bool LHY, int R, int NW>
void launch_mode(int mode, const TilePlan &g, int blocks, const TileParams<T> *p, const int2 *items, hipStream_t s) {
    if (mode == kTileImag) launch<T, LHY, kTileImag, R, NW>(g, blocks, p, items, s);
    else if (mode == 0) launch<T, LHY, 0, R, NW>(g, blocks, p, items, s);
    else if (mode == 1) launch<T, LHY, 1, R, NW>(g, blocks, p, items, s);
    else launch<T, LHY, -1, R, NW>(g, blocks, p, items, s);
}

template <typename T, bool LHY>
int launch_rows(int mode, const TilePlan &g, int blocks, const TileParams<T> *p, const int2 *items, hipStream_t s) {
    constexpr int N = kTileWaves;
    if constexpr (sizeof(T) == 4) {
        if (g.nw == 16) launch_mode<T, LHY, 4, 16>(mode, g, blocks, p, items, s);
        else if (g.r == 4) launch_mode<T, LHY, 4, N>(mode, g, blocks, p, items, s);
        else launch_mode<T, LHY, 12, N>(mode, g, blocks, p, items, s);
    } else {
        if (g.r == 4) launch_mode<T, LHY, 4, N>(mode, g, blocks, p, items, s);
        else if (g.r == 6) launch_mode<T, LHY, 6, N>(mode, g, blocks, p, items, s);
        else launch_mode<T, LHY, 8, N>(mode, g, blocks, p, items, s);
    }
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) return set_error(TSMI_E_HIP, std::string("tile_kernel: ") + hipGetErrorString(e));
    return TSMI_OK;
}

template <typename T>
int launch_any(bool lhy, int mode, const TilePlan &g, int blocks, const TileParams<T> *p, const int2 *items,
               hipStream_t s) {
    return lhy ? launch_rows<T, true>(mode, g, blocks, p, items, s)
               : launch_rows<T, false>(mode, g, blocks, p, items, s);
}

// One pass of context c.  how: kClosed, kWrap, kSeam.
enum How { kClosed, kWrap, kSeam };

template <typename T>
int pass(tsmi_ctx *c, int steps, How how, long double &drift) {
    TileParams<T> p;
    std::memset(&p, 0, sizeof(p));
    const int nb = 1 - c->cur;
    const std::pair<int, int> size(c->W, c->H);
    const TilePlan g = plan(&size, 1, c->esz, steps);
    if (g.r == 0) return set_error(TSMI_E_INVALID, "tile pass: no tile for this many steps");
    const TileFactors f = {c->mH, c->tH, c->mV, c->tV, c->unH, c->unV, c->c_nl_s, c->c_lhy_s, c->corr_abs,
                           c->d.delta_t / (4. * c->d.mass * c->d.delta_y * c->d.delta_y)};
    const bool wrap = how == kWrap;
    tile_params<T>(p, f, g, c->W, c->H, c->pitch, wrap ? c->d.dim_x : 0, wrap ? c->d.dim_y : 0, steps, drift);
    p.seam = how == kSeam;
    p.px = c->d.periodic_x != 0; p.py = c->d.periodic_y != 0;
    p.in_re = (const T *)c->psi_re[c->cur];
    p.in_im = (const T *)c->psi_im[c->cur];
    p.out_re = (T *)c->psi_re[nb];
    p.out_im = (T *)c->psi_im[nb];
    p.ph = (const T *)c->ph;
    const int blocks = p.n_strips * ((c->H + p.rows - 1) / p.rows);
    const bool imag = c->d.imag_time != 0;
    if (imag) {
        if (blocks > c->part_cap) return set_error(TSMI_E_INVALID, "tile pass: more workgroups than partial sums");
        p.part_in = c->div_pending ? c->partials + (size_t)c->div_slot * c->part_cap : nullptr;
        p.n_in = c->part_n + c->div_slot;
        p.part_out = c->partials + (size_t)(1 - c->div_slot) * c->part_cap;
        p.n_out = c->part_n + (1 - c->div_slot);
        p.norm_target = c->d.norm_target;
        p.dxdy = c->d.delta_x * c->d.delta_y;
        p.ix0 = c->ix0; p.ix1 = c->ix1; p.iy0 = c->iy0; p.iy1 = c->iy1;
    }
    if (int st = ctx_time_mark(c, steps > 1, 0)) return st;
    if (int st = launch_any<T>(c->c_lhy != 0.0, imag ? kTileImag : c->mode, g, blocks, &p, nullptr, c->stream)) return st;
    c->cur = nb;
    if (imag) {
        c->div_slot = 1 - c->div_slot;
        c->div_pending = true;
    }
    return ctx_time_mark(c, steps > 1, 1);
}

}  // namespace

namespace tsmi {

TilePlan tile_plan(const std::vector<std::pair<int, int>> &sizes, int esz, int steps) {
    return plan(sizes.data(), sizes.size(), esz, steps);
}

int tile_best_steps(const std::vector<std::pair<int, int>> &sizes, int esz, int most) {
    return best_steps(sizes.data(), sizes.size(), esz, most);
}

template <typename T>
void tile_params(TileParams<T> &p, const TileFactors &f, const TilePlan &g, int W, int H, int pitch, int nx, int ny,
                 int steps, long double &drift) {
    p.W = W; p.H = H; p.pitch = pitch;
    p.nx = nx;
    p.ny = ny;
    p.steps = steps;
    p.cols = kTileCols - 2 * kApron * steps;
    p.rows = g.nw * g.r - 2 * kApron * steps;
    p.n_strips = (W + p.cols - 1) / p.cols;
    p.mH = (T)f.mH; p.tH = (T)f.tH; p.mV = (T)f.mV; p.tV = (T)f.tV;
    p.unH = (T)f.unH; p.unV = (T)f.unV;
    p.c_nl = (T)f.c_nl_s; p.c_lhy = (T)f.c_lhy_s;
    // The merged V0 V0 pass (factors m2, t2) stands for the square of V0's (m, t):
    // its eigenvalue is 1/q of the exact one, q = (m + i t)^2 / (m2 + i t2), so a
    // step followed by it applies |q| with |corr|.  The sign of q goes into the
    // modulus (a phase near pi would leave the small-angle forms); what is left of
    // its phase, an effect of the rounded coefficients, commutes with every pass
    // and is spread over the k steps.  The moduli are rounded to FP64: a rounding
    // that repeats every step would be a drift of the norm (1.8e-16 per step at
    // 64^2), so the last step of a pass takes back what the pass's and the
    // call's earlier ones left (drift: the log of what was applied over what was
    // meant).
    typedef std::complex<long double> zl;
    const Axis two = frame_axis(std::cos(2 * f.by), std::sin(2 * f.by), false, (int)sizeof(T));
    const zl v1(f.mV, f.tV), v2(two.m, two.t);
    zl q = v1 * v1 / v2;
    const long double sign = q.real() < 0 ? -1.0L : 1.0L;
    q *= sign;
    p.m2 = (T)two.m; p.t2 = (T)two.t; p.un2 = (T)two.un;
    p.mode2 = two.form;
    const long double mid = f.corr_abs * std::abs(q);
    p.mag_mid = (double)(sign * mid);
    drift += (steps - 1) * std::log(std::fabs((long double)p.mag_mid) / mid);
    p.mag = (double)(f.corr_abs * (1.0L - drift));
    drift += std::log((long double)p.mag / f.corr_abs);
    p.dphi = (T)(-(steps - 1.0L) / steps * std::arg(q));
}

template void tile_params<float>(TileParams<float> &, const TileFactors &, const TilePlan &, int, int, int, int, int,
                                 int, long double &);
template void tile_params<double>(TileParams<double> &, const TileFactors &, const TilePlan &, int, int, int, int, int,
                                  int, long double &);

int tile_batch_launch(int esz, bool lhy, int mode, const TilePlan &g, const void *params, const int2 *items,
                      int n_items, hipStream_t stream) {
    return esz == 4 ? launch_any<float>(lhy, mode, g, n_items, (const TileParams<float> *)params, items, stream)
                    : launch_any<double>(lhy, mode, g, n_items, (const TileParams<double> *)params, items, stream);
}

bool tile_wraps(const tsmi_ctx *c) {
    return c->d.periodic_x && c->d.periodic_y && c->d.dim_x % 2 == 0 && c->d.dim_y % 2 == 0;
}

// The one-plane form of E, no segment height or steps per pass asked
// for, offsets within 31 bits, and a lattice small enough that a wave's row
// latency bounds the streaming passes: us per step, streamed against tiles, 64^2
// FP64 17.3 / 2.8, 256^2 FP64 23.1 / 4.4, FP32 16.6 / 3.2, 512^2 FP32 14.5 / 3.9,
// 1024^2 FP32 17.0 / 6.6, FP64 23.6 / 10.5, 1600^2 FP64 36.0 / 19.6, 1700^2 FP64
// 35.8 / 30.0, 1800^2 37.1 / 32.6, 2000^2 FP32 23.7 / 18.3, 2200^2 FP32 24.7 / 31.3,
// 2048^2 FP64 33.6 / 43.4.  Imaginary time, one step per pass, gives out earlier: closed FP32 100^2
// 12.4 / 6.9, 1200^2 15.0 / 13.1, 2048^2 23.1 / 28.8, FP64 100^2 14.7 / 6.8, 1024^2
// 20.7 / 14.8, 1200^2 21.3 / 22.6.
bool tile_runs(const tsmi_ctx *c) {
    const bool imag = c->d.imag_time != 0;
    const long most = imag ? (c->esz == 4 ? 3L << 19 : 9L << 17) : (c->esz == 4 ? 9L << 19 : 5L << 19);
    return c->ph_mode && c->d.sweeps == 0 && c->d.tile_rows == 0 && c->H > 1 && (long)c->W * c->H <= most &&
           (long)c->pitch * c->Hd * c->esz < (1L << 31);
}

int tile_blocks(const tsmi_ctx *c) {
    const std::pair<int, int> size(c->W, c->H);
    const TilePlan g = plan(&size, 1, c->esz, 1);
    const int cols = kTileCols - 2 * kApron, rows = g.nw * g.r - 2 * kApron;
    return ((c->W + cols - 1) / cols) * ((c->H + rows - 1) / rows);
}

static int tile_pass(tsmi_ctx *c, int steps, How how, long double &drift) {
    return c->esz == 4 ? pass<float>(c, steps, how, drift) : pass<double>(c, steps, how, drift);
}

int tile_passes(tsmi_ctx *c, int n, bool wrap) {
    if (n <= 0) return TSMI_OK;
    const std::pair<int, int> size(c->W, c->H);
    const int k = c->d.imag_time ? 1 : best_steps(&size, 1, c->esz, n), passes = (n + k - 1) / k;
    long double drift = 0.0L;
    int st = TSMI_OK;
    for (int i = 0; i < passes && !st; ++i)
        st = tile_pass(c, n / passes + (i < n % passes ? 1 : 0), wrap ? kWrap : kClosed, drift);
    return st;
}

int tile_seam_steps(tsmi_ctx *c, int n) {
    long double drift = 0.0L;
    int st = TSMI_OK;
    for (int i = 0; i < n && !st; ++i) st = tile_pass(c, 1, kSeam, drift);
    return st;
}

}  // namespace tsmi
