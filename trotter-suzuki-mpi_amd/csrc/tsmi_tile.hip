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

// The modelled time of a step, fitted to 800 timings (200^2 to 2400^2, every
// shape, 1 to 6 steps per pass; 8 % rms in FP64, 12 % in FP32): a launch costs
// t0 and its planes at bw TB/s (3 in, 2 out; a part h of that when a compute unit
// holds several workgroups, one computing while another loads), a step costs each
// SIMD its rows (row us, more for a wave alone) and x of exchanges and passes.
struct TileCost {
    double row, alone, x, t0, bw, h;
};
constexpr TileCost kCost32 = {0.117, 0.8, 1.9, 2.0, 5.8, 0.8}, kCost64 = {0.207, 0.37, 1.0, 3.3, 6.5, 0.85};

// Waves per SIMD that the registers of an instance leave.
int tile_waves(int esz, int r) { return esz == 4 ? (r == 4 ? 4 : 2) : (r == 4 ? 3 : 2); }

// The tile shape of a pass of `steps` steps: the one with the least modelled time.
// Without the planes' time the model took one step per pass at 1800^2 and 2100^2
// FP32 (21.5 and 28.7 us per step; three and four steps 15.5 and 20.1) and 4 rows
// x 8 waves for single FP64 steps of 1200^2 (18.7; 8 x 4 15.3).  In imaginary time
// every wave adds the partial sums of all workgroups: 4 ns each.
TilePlan plan(const std::pair<int, int> *size, size_t count, int esz, int steps, bool imag) {
    TilePlan best;
    const int a = kApron * steps;
    const int *rr = esz == 4 ? kRows32 : kRows64, n_rr = esz == 4 ? 2 : 3;
    const TileCost &m = esz == 4 ? kCost32 : kCost64;
    double cells = 0;
    for (size_t j = 0; j < count; ++j) cells += (double)size[j].first * size[j].second;
    const double planes = cells * 5 * esz / (m.bw * 1e6);
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
            const int held = std::max(1, tile_waves(esz, p.r) * 4 / nw);   // ... that it holds at a time
            const double waves = std::min(per_cu, (double)held) * nw / 4;  // waves per SIMD
            p.us = (m.t0 + planes * (std::min(per_cu, (double)held) > 1 ? m.h : 1.0)) / steps +
                   per_cu * nw * p.r / 4 * m.row * (1 + m.alone / waves) + m.x + (imag ? 0.004 * tiles : 0.0);
            if (p.us < best.us) best = p;
        }
    return best;
}

int best_steps(const std::pair<int, int> *size, size_t count, int esz, int most) {
    int k = 1;
    double us = 1e30;
    for (int s = 1; s <= std::min(most, 8); ++s) {
        const TilePlan p = plan(size, count, esz, s, false);
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
int pass(tsmi_ctx *c, const TilePlan &g, int steps, How how, long double &drift) {
    TileParams<T> p;
    std::memset(&p, 0, sizeof(p));
    const int nb = 1 - c->cur;
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
    return plan(sizes.data(), sizes.size(), esz, steps, false);
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

long tile_area(int W, int H) { return (W + 119L) / 120 * 120 * ((H + 23L) / 24 * 24); }

// Cells, and cells of whole tiles (tile_area), up to which a pass of one step, or of
// several, takes tiles.  us per step, streamed / tiles, closed and doubly periodic
// alike unless said.
// Several steps per pass (against two streamed): 64^2 FP64 17.3 / 2.8, FP32 256^2
// 16.6 / 3.2, 512^2 14.5 / 3.9, 1000^2 14.0 / 5.6, 1800^2 19.0 / 15.5, 2100^2 22.6 /
// 20.1, 2200^2 22.6 / 22.4; FP64 1000^2 15.4 / 8.0, 1600^2 24.2 / 18.7, 2000^2 29.1 /
// 27.9, 2100^2 31.0 / 32.9 (the FP64 line is drawn at 1620^2).
// One step per pass (single steps, short calls, mixed axes, odd periodic extents):
// FP32 1000^2 17.9 / 9.0, 1800^2 22.9 / 18.9, 2000^2 24.2 / 22.5, 2100^2 25.7 / 24.6
// before the halo exchange of a periodic step, mixed or odd periodic axes 2001^2 26.2 /
// 22.5 with it; FP64 1000^2 15.8 / 12.0, 1200^2 17.2 / 15.3, 1400^2 22.8 / 20.7,
// 1500^2 23.3 / 24.7.
// Imaginary time: FP32 100^2 12.4 / 6.9, 1200^2 14.5 / 13.1, 1300^2 16.9 / 16.7, 1400^2
// 17.4 / 17.9; FP64 100^2 14.7 / 6.8, 1050^2 18.3 / 15.2, 1200^2 19.4 / 17.7, 1300^2 24.5 /
// 24.7 (the line is drawn at 1080^2).
// Narrow and flat lattices leave most of their tiles idle: several FP32 steps 2 x 10^6
// 202 / 479, 61 x 30000 19 / 12, 30 x 10^5 the other way round 14.8 / 14.5, 9 x 300000
// 12.7 / 17; single FP32 steps 30 x 10^5 18.4 / 21; FP64 125 x 19000 30 / 40, 30 x 30000
// 24.3 / 23.8; imaginary time FP32 20 x 20000 15.7 / 12.9, 30 x 30000 20.1 / 20.9, FP64
// 22.4 / 20.3, 28.1 / 32.1.
struct TileLimit {
    long cells, area;
};
static bool within(const TileLimit &l, int W, int H) { return (long)W * H <= l.cells && tile_area(W, H) <= l.area; }
static TileLimit limit_one(int esz, bool imag) {
    if (imag) return {esz == 4 ? 3L << 19 : 9L << 17, 5L << 19};
    return esz == 4 ? TileLimit{8L << 19, 9L << 19} : TileLimit{15L << 17, 7L << 19};
}
static TileLimit limit_several(int esz) {
    return esz == 4 ? TileLimit{9L << 19, 10L << 19} : TileLimit{5L << 19, 7L << 19};
}

// No segment height or steps per pass asked for, and a lattice small enough that a wave's row latency bounds the
// streaming passes.
TileRoute tile_route(const tsmi_desc &d, int W, int H, int n, bool e_wraps) {
    if (n <= 0 || d.sweeps != 0 || d.tile_rows != 0 || H <= 1) return kRouteStream;
    const int esz = d.precision == 32 ? 4 : 8;
    const bool imag = d.imag_time != 0, closed = !d.periodic_x && !d.periodic_y;
    const bool even = d.periodic_x && d.periodic_y && d.dim_x % 2 == 0 && d.dim_y % 2 == 0;
    const bool one = within(limit_one(esz, imag), W, H);
    const bool several = imag ? one : within(limit_several(esz), W, H);
    if (closed && (n == 1 ? one : several)) return kRouteClosed;
    if (even && (!imag || e_wraps) && n >= 3 && several) return kRouteWrap;
    return !closed && one ? kRouteSeam : kRouteStream;
}

TileRoute tile_route(const tsmi_ctx *c, int n) {
    return c->ph_mode ? tile_route(c->d, c->W, c->H, n, c->e_wraps) : kRouteStream;
}

void tile_geometry(const tsmi_desc &d, int W, int H, int n, int32_t out[4]) {
    const TileRoute route = tile_route(d, W, H, n, true);
    for (int i = 0; i < 4; ++i) out[i] = 0;
    if (route == kRouteStream) return;
    const std::pair<int, int> size(W, H);
    const int esz = d.precision == 32 ? 4 : 8;
    int k = 1;
    if (!d.imag_time && route != kRouteSeam) {
        const int m = route == kRouteWrap ? n - 2 : n, q = (m + best_steps(&size, 1, esz, m) - 1) / best_steps(&size, 1, esz, m);
        k = (m + q - 1) / q;
    }
    const TilePlan g = plan(&size, 1, esz, k, d.imag_time != 0);
    const int cols = kTileCols - 2 * kApron * k, rows = g.nw * g.r - 2 * kApron * k;
    out[0] = g.r;
    out[1] = g.nw;
    out[2] = k;
    out[3] = ((W + cols - 1) / cols) * ((H + rows - 1) / rows);
}

static TilePlan plan_of(const tsmi_ctx *c, int steps) {
    const std::pair<int, int> size(c->W, c->H);
    return plan(&size, 1, c->esz, steps, c->d.imag_time != 0);
}

int tile_blocks(const tsmi_ctx *c) {
    const TilePlan g = plan_of(c, 1);
    const int cols = kTileCols - 2 * kApron, rows = g.nw * g.r - 2 * kApron;
    return ((c->W + cols - 1) / cols) * ((c->H + rows - 1) / rows);
}

static int tile_pass(tsmi_ctx *c, const TilePlan &g, int steps, How how, long double &drift) {
    return c->esz == 4 ? pass<float>(c, g, steps, how, drift) : pass<double>(c, g, steps, how, drift);
}

int tile_passes(tsmi_ctx *c, int n, bool wrap) {
    if (n <= 0) return TSMI_OK;
    const std::pair<int, int> size(c->W, c->H);
    const int k = c->d.imag_time ? 1 : best_steps(&size, 1, c->esz, n), passes = (n + k - 1) / k;
    const int steps = n / passes, longer = n % passes;   // the first `longer` passes take a step more
    long double drift = 0.0L;
    int st = TSMI_OK;
    TilePlan g = plan_of(c, steps + (longer > 0));
    for (int i = 0; i < passes && !st; ++i) {
        if (i == longer && longer > 0) g = plan_of(c, steps);
        st = tile_pass(c, g, steps + (i < longer), wrap ? kWrap : kClosed, drift);
    }
    return st;
}

int tile_seam_steps(tsmi_ctx *c, int n) {
    const TilePlan g = plan_of(c, 1);
    long double drift = 0.0L;
    int st = TSMI_OK;
    for (int i = 0; i < n && !st; ++i) st = tile_pass(c, g, 1, kSeam, drift);
    return st;
}

}  // namespace tsmi
