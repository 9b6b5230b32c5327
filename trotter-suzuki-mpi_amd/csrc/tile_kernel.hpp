// tile_kernel.hpp -- several real-time steps of a small or medium lattice per
// launch, the tile held in registers.
//
// What bounds a small lattice is not memory but each wave's chain of dependent
// row updates: step_kernel and step2_kernel stream rows through a pipeline, one
// row per beat, and a 256^2 lattice gives them a few dozen waves, each alone on
// its SIMD, whose beats wait for one another (FP64 54 us per two-step launch).
// Here a workgroup of NW waves holds a tile of 128 columns x (NW R) rows, R rows
// x 2 columns per lane in registers, and runs k whole steps on it: every pass is
// R independent row updates per wave, so a wave alone on its SIMD issues back to
// back, the rows are loaded at once, and one launch serves k steps.  The tile
// carries an apron of 4k cells on each side (the dependency cone of k steps).
//
// Vertical pairs inside a wave's rows are register operations.  A vertical pass
// pairs rows (y, y+1) where x + y + s is even, so at the border between two
// waves one of a lane's two columns pairs across it: the waves exchange that
// column of their first and last rows through LDS (double-buffered, one barrier
// per vertical pass; the border rows are computed first, so that the other rows'
// work lies between the write and the barrier).  The last V0 of a step and the
// first of the next are one pass of twice the angle (coefficients m2, t2 of
// that angle), which saves one of the four exchanges.
//
// Measured against the streaming passes, us per step: 64^2 periodic FP64 17.3 ->
// 2.8, 256^2 FP64 23.1 -> 4.4, 1024^2 FP32 17.0 -> 6.6, FP64 23.6 -> 10.5.  Now
// bound by instruction issue (and by the launch, some 4 us of a pass).
//
// Imaginary time (kTileImag) takes one step per pass, as every step ends in a
// renormalisation by the whole lattice's norm: the partial sums of a step's
// workgroups are added by every wave of the next, which scales its rows as it
// loads them (256^2 closed FP32 12.8 -> 7.0 us per step, FP64 15.3 -> 7.0).
//
// Two uses, by p.nx: 0: the tile W x H is closed at its edges (closed axes, or
// one step on the reference tile of a periodic lattice, its halo as it is).
// Otherwise W and H are the tile of a doubly periodic lattice of nx x ny inner
// cells, both even (the pair pattern then is periodic too): rows and columns are
// read from the inner cells they mirror, every cell of the tile is written, and
// the halo is left as the exchange would leave it.  Mixed axes and odd periodic
// extents run one step per pass on the closed tile, the state's halo cells read
// from the cells they mirror (seam): no exchange runs between the steps.
#pragma once
#include "step_kernel.hpp"

namespace tsmi {

constexpr int kTileWaves = 8;        // most waves per workgroup of a tile (the 16 waves of 4 FP32 rows apart)
constexpr int kTileCols = 2 * kWave; // columns of a tile
constexpr int kTileImag = 2;         // MODE of imaginary time

template <typename T>
struct TileParams {
    const T *in_re, *in_im;
    T *out_re, *out_im;
    const T *ph;                     // phase plane (StepParams::ph)
    int W, H, pitch;
    int nx, ny;                      // inner extents of a doubly periodic lattice, or 0
    int steps;                       // k
    int seam, px, py;                // 1: one step on the reference tile, the state's halo read through seam_off
    int n_strips, cols, rows;        // output columns and rows per tile
    T mH, tH, mV, tV, unH, unV;      // scaled-frame pair factors (StepParams)
    T m2, t2, un2;                   // the merged V0 V0 pass
    int mode2;                       // its scaled form
    T c_nl, c_lhy;
    double mag, mag_mid;             // |corr| of the last step and of the steps before it
    T dphi;                          // phase of the merged frame, added to every phase
    // imaginary time, as StepParams; one partial sum per workgroup
    const double *part_in;
    const int *n_in;
    double *part_out;
    int *n_out;
    double norm_target, dxdy;
    int ix0, ix1, iy0, iy1;
};

// A cell of the reference tile whose halo exchange has not run: where its value
// is (a byte offset), as exchange_cell would have copied it.  The copy's own
// quirk is kept: with a closed y axis the x halo of the last 2 halo rows stays.
struct SeamTile {
    int W, H, px, py;
};
__device__ __forceinline__ unsigned seam_off(const SeamTile &q, int x, int y, unsigned row_bytes, unsigned esz) {
    if (x < 0 || x >= q.W || y < 0 || y >= q.H) return kOffNone;
    const int lo = q.py ? kApron : 0, hi = lo + max(0, q.H - 2 * kApron);   // rows whose x halo is refreshed
    int sx = x, sy = y;
    if (q.py && y < kApron) sy = y + q.H - 2 * kApron;
    if (q.py && y >= q.H - kApron) sy = y - (q.H - 2 * kApron);
    if (q.px && sy >= lo && sy < hi) {
        if (x < kApron) sx = x + q.W - 2 * kApron;
        if (x >= q.W - kApron) sx = x - (q.W - 2 * kApron);
    }
    return (unsigned)sx * esz + (unsigned)sy * row_bytes;
}
__device__ __forceinline__ float buf_load1(__amdgpu_buffer_rsrc_t r, unsigned off, float) {
    return __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(r, off, 0u, 0));
}
__device__ __forceinline__ double buf_load1(__amdgpu_buffer_rsrc_t r, unsigned off, double) {
    return __builtin_bit_cast(double, __builtin_amdgcn_raw_buffer_load_b64(r, off, 0u, 0));
}
// Two cells of a row, each from where it is.
template <typename T>
__device__ __forceinline__ void seam_load(const SeamTile &q, __amdgpu_buffer_rsrc_t re, __amdgpu_buffer_rsrc_t im, int x,
                                          int y, unsigned row_bytes, Row<T, 2> &s) {
#pragma unroll
    for (int k = 0; k < 2; ++k) {
        const unsigned off = seam_off(q, x + k, y, row_bytes, (unsigned)sizeof(T));
        s.re[k] = buf_load1(re, off, T(0));
        s.im[k] = buf_load1(im, off, T(0));
    }
}

// The barrier of the step loops.  Waves of one workgroup may meet at it from
// different instances of a loop: the instance is chosen by a wave's own rows (with or
// without the edges' factors; for the whole workgroup the edge's instance, closed
// 256^2 FP64 measured 4.39 -> 4.46 us per step, 1000^2 8.2 -> 8.6).  __syncthreads is
// defined for one and the same barrier only; s_barrier counts the arrivals of waves,
// whatever the instruction's place.  So two things must hold: the choice is uniform in
// a wave (its index comes through readfirstlane), and every instance runs the same
// number of vertical passes, which depends on the number of steps alone.
__device__ __forceinline__ void tile_barrier() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
}

template <typename T, int NW>
struct TileXch {
    typedef T __attribute__((ext_vector_type(2))) T2;
    // [buffer][first / last row of a wave][wave + 1][lane]; the slots of waves -1
    // and NW hold zeros (no row there)
    T2 v[2][2][NW + 2][kWave];
};

// The potential pass of two rows: one wave-uniform test and straight-line code
// for the four values per lane.
template <typename T, bool LHY, bool IMAG = false, int NEAR = 1>
__device__ __forceinline__ void tile_ppass(Row<T, 2> &a, Row<T, 2> &b, const T (&pa)[2], const T (&pb)[2], T c, T cl,
                                           double mag) {
    T ang[4], sn[4], cs[4];
    auto angle = [&](const Row<T, 2> &r, int k, T ph) {
        const T n2 = r.re[k] * r.re[k] + r.im[k] * r.im[k];
        return (LHY ? c * n2 + cl * (n2 * sqrt_t(n2)) : c * n2) + ph;
    };
    ang[0] = angle(a, 0, pa[0]);
    ang[1] = angle(a, 1, pa[1]);
    ang[2] = angle(b, 0, pb[0]);
    ang[3] = angle(b, 1, pb[1]);
    if constexpr (IMAG) {
        T f[4];
        expneg_row<T, 4>(ang, f);
#pragma unroll
        for (int k = 0; k < 2; ++k) {
            a.re[k] *= f[k];
            a.im[k] *= f[k];
            b.re[k] *= f[2 + k];
            b.im[k] *= f[2 + k];
        }
        return;
    }
    sincos_row<T, 4, NEAR>(ang, sn, cs);
    const T ca[2] = {cs[0], cs[1]}, sa[2] = {sn[0], sn[1]}, cb[2] = {cs[2], cs[3]}, sb[2] = {sn[2], sn[3]};
    rotate_row_ph<T, 2>(a, ca, sa, mag);
    rotate_row_ph<T, 2>(b, cb, sb, mag);
}

// EH: the strip reaches past the tile's left or right edge (per-lane pair
// coefficients); EV: so do the wave's rows at the top or bottom (bit r + 1 of ok:
// rows r and r + 1 of the wave are both inside the tile).
// MODE: kTileImag is one step in imaginary time (form A).
template <typename T, bool LHY, int MODE, int R, bool EH, bool EV, int NW>
__device__ __forceinline__ void tile_steps(const TileParams<T> &p, Row<T, 2> (&s)[R], const T (&ph)[R][2],
                                           TileXch<T, NW> &x, int w, int lane, int xl,
                                           unsigned ok) {
    static_assert(R % 2 == 0 && R >= 4, "row parities are fixed per register");
    typedef typename TileXch<T, NW>::T2 T2;
    constexpr bool IMAG = MODE == kTileImag;
    constexpr int M = MODE < 0 || IMAG ? 0 : MODE;
    const T kH = M == 0 ? p.tH : p.mH;
    HCoef<T, 2> hc = {};
    // a periodic lattice has no edge: every column far from one
    if constexpr (EH)
        hc = make_hcoef<T, 2>(p.nx ? 2 * lane + 2 : xl, lane, p.nx ? 1 << 30 : p.W, p.mH, p.tH, p.unH);
    int buf = 0;

    auto hrow = [&](auto ss, Row<T, 2> &r, auto rr) {
        constexpr int PAR = (decltype(ss)::value + decltype(rr)::value) & 1;
        if constexpr (EH) hpass<PAR, IMAG>(r, hc);
        else hpass_fast<PAR, IMAG, M>(r, kH);
    };
    // the vertical pass V(S), factors (m, t) in the scaled form FM (-1: both
    // factors) and un for unpaired cells; `first` has run on the border rows and
    // `rest` runs on the others between the exchange's write and its barrier
    auto vpass = [&](auto ss, auto fm, T m, T t, T un, auto &&rest) {
        constexpr int S = decltype(ss)::value, FM = decltype(fm)::value;
        constexpr int CX = 1 - S;                    // the column that pairs across the border
        T2 top, bot;
        top[0] = s[0].re[CX];
        top[1] = s[0].im[CX];
        bot[0] = s[R - 1].re[CX];
        bot[1] = s[R - 1].im[CX];
        x.v[buf][0][w + 1][lane] = top;
        x.v[buf][1][w + 1][lane] = bot;
        rest();
        tile_barrier();
        const T2 up = x.v[buf][1][w][lane], dn = x.v[buf][0][w + 2][lane];
        buf ^= 1;
        // cells without a partner only exist at the tile's edges (EV): the test of
        // their bit is uniform
        auto pair = [&](int c, int r) {
            if (EV && __builtin_expect(!(ok >> (r + 1) & 1u), 0)) {
                s[r].re[c] *= un;
                s[r].im[c] *= un;
                s[r + 1].re[c] *= un;
                s[r + 1].im[c] *= un;
            } else if constexpr (FM < 0) {
                rot<IMAG>(m, t, s[r].re[c], s[r].im[c], s[r + 1].re[c], s[r + 1].im[c]);
            } else {
                fpair<IMAG, FM>(FM == 0 ? t : m, s[r].re[c], s[r].im[c], s[r + 1].re[c], s[r + 1].im[c]);
            }
        };
#pragma unroll
        for (int r = 0; r + 1 < R; r += 2) pair(S, r);
#pragma unroll
        for (int r = 1; r + 1 < R; r += 2) pair(CX, r);
        Row<T, 2> &f = s[0], &l = s[R - 1];
        if (EV && __builtin_expect(!(ok & 1u), 0)) {
            f.re[CX] *= un;
            f.im[CX] *= un;
        } else if constexpr (FM < 0) {
            rot_q<IMAG>(m, t, up[0], up[1], f.re[CX], f.im[CX]);
        } else {
            fpair_q<IMAG, FM>(FM == 0 ? t : m, up[0], up[1], f.re[CX], f.im[CX]);
        }
        if (EV && __builtin_expect(!(ok >> R & 1u), 0)) {
            l.re[CX] *= un;
            l.im[CX] *= un;
        } else if constexpr (FM < 0) {
            rot_p<IMAG>(m, t, l.re[CX], l.im[CX], dn[0], dn[1]);
        } else {
            fpair_p<IMAG, FM>(FM == 0 ? t : m, l.re[CX], l.im[CX], dn[0], dn[1]);
        }
    };
    using I0 = std::integral_constant<int, 0>;
    using I1 = std::integral_constant<int, 1>;
    using IM = std::integral_constant<int, IMAG ? 0 : MODE>;
    auto h_border = [&](auto ss) {
        hrow(ss, s[0], I0());
        hrow(ss, s[R - 1], I1());                    // R - 1 is odd
    };
    auto h_rest = [&](auto ss) {
#pragma unroll
        for (int r = 1; r + 1 < R; r += 2) {
            hrow(ss, s[r], I1());
            hrow(ss, s[r + 1], I0());
        }
    };

    vpass(I0(), IM(), p.mV, p.tV, p.unV, [] {});
    for (int st = 0;; ++st) {
        const bool last = st == p.steps - 1;
        const double mag = last ? p.mag : p.mag_mid;
        h_border(I0());
        vpass(I1(), IM(), p.mV, p.tV, p.unV, [&] { h_rest(I0()); });
        h_border(I1());
        h_rest(I1());
        // the potential pass, border rows first
        tile_ppass<T, LHY, IMAG>(s[0], s[R - 1], ph[0], ph[R - 1], p.c_nl, p.c_lhy, mag);
        h_border(I1());
        vpass(I1(), IM(), p.mV, p.tV, p.unV, [&] {
#pragma unroll
            for (int r = 1; r + 1 < R; r += 2)
                tile_ppass<T, LHY, IMAG>(s[r], s[r + 1], ph[r], ph[r + 1], p.c_nl, p.c_lhy, mag);
            h_rest(I1());
        });
        h_border(I0());
        if (IMAG || last) break;
        if (p.mode2 == 0)
            vpass(I0(), I0(), p.m2, p.t2, p.un2, [&] { h_rest(I0()); });
        else
            vpass(I0(), I1(), p.m2, p.t2, p.un2, [&] { h_rest(I0()); });
    }
    vpass(I0(), IM(), p.mV, p.tV, p.unV, [&] { h_rest(I0()); });
}

// Tile `tile` of the pass p by a workgroup of nw waves, at most NW.
template <typename T, bool LHY, int MODE, int R, int NW>
__device__ __forceinline__ void tile_group(const TileParams<T> &p, int tile, TileXch<T, NW> &xch) {
    const int lane = threadIdx.x & (kWave - 1);
    const int w = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
    const int nw = blockDim.x / kWave;
    const int strip = tile % p.n_strips, seg = tile / p.n_strips;
    const int A = kApron * p.steps;
    const bool wrap = p.nx != 0;
    const int X0 = strip * p.cols - A;                            // even
    const int xl = X0 + 2 * lane;
    // a closed tile's first rows need no apron above them
    const int y_tile = wrap ? seg * p.rows - A : max(0, seg * p.rows - A);
    const int y0 = y_tile + w * R;                                // even: first row of this wave

    // slots of the rows above the first and below the last wave
    if (w == 0) {
        typename TileXch<T, NW>::T2 z = {T(0), T(0)};
        xch.v[0][1][0][lane] = xch.v[1][1][0][lane] = z;
        xch.v[0][0][nw + 1][lane] = xch.v[1][0][nw + 1][lane] = z;
    }

    const unsigned bytes = (unsigned)p.pitch * (unsigned)p.H * (unsigned)sizeof(T);
    const __amdgpu_buffer_rsrc_t r_in_re = make_rsrc(p.in_re, bytes), r_in_im = make_rsrc(p.in_im, bytes);
    const __amdgpu_buffer_rsrc_t r_ph = make_rsrc(p.ph, bytes);
    const __amdgpu_buffer_rsrc_t r_out_re = make_rsrc(p.out_re, bytes), r_out_im = make_rsrc(p.out_im, bytes);
    const unsigned row_bytes = (unsigned)p.pitch * (unsigned)sizeof(T);
    auto mod = [](int a, int n) {
        const int r = a % n;
        return r < 0 ? r + n : r;
    };
    int xs = xl;
    bool ld_ok = xl >= 0 && xl + 2 <= p.pitch;
    if (wrap) {
        xs = kApron + mod(xl - kApron, p.nx);                     // even, nx even: the pair stays together
        ld_ok = true;
    }
    const unsigned v_ld = ld_ok ? (unsigned)xs * (unsigned)sizeof(T) : kOffNone;

    Row<T, 2> s[R];
    T ph[R][2];
    auto load = [&](auto seam) {
        const SeamTile q = {p.W, p.H, p.px, p.py};
        int ys = wrap ? mod(y0 - kApron, p.ny) : y0;              // one division, then row by row
#pragma unroll
        for (int r = 0; r < R; ++r) {
            const bool in = wrap || (ys >= 0 && ys < p.H);
            const unsigned off = in ? v_ld + (unsigned)(wrap ? ys + kApron : ys) * row_bytes : kOffNone;
            ys = wrap && ys + 1 == p.ny ? 0 : ys + 1;
            if constexpr (decltype(seam)::value) {
                seam_load<T>(q, r_in_re, r_in_im, xl, y0 + r, row_bytes, s[r]);
            } else {
                buf_load<T, 2>(r_in_re, off, 0u, s[r].re);
                buf_load<T, 2>(r_in_im, off, 0u, s[r].im);
            }
            buf_load<T, 2>(r_ph, off, 0u, ph[r]);
        }
    };
    if (p.seam) load(std::true_type());
    else load(std::false_type());
    if constexpr (MODE == kTileImag) {
        // the pending renormalisation, as step_kernel applies it
        if (p.part_in) {
            const int n = __builtin_amdgcn_readfirstlane(*p.n_in);
            const double inv = 1.0 / renorm_divisor(p.part_in, n, p.dxdy, p.norm_target, lane);
#pragma unroll
            for (int r = 0; r < R; ++r) scale_row<T, 2>(s[r], inv);
        }
    }
#pragma unroll
    for (int r = 0; r < R; ++r) {
        ph[r][0] += p.dphi;
        ph[r][1] += p.dphi;
    }
    __syncthreads();

    // per wave: see tile_barrier
    const bool eh = MODE < 0 || (!wrap && (X0 < 0 || X0 + kTileCols > p.W));
    const bool ev = MODE < 0 || (!wrap && (y0 <= 0 || y0 + R >= p.H));
    unsigned ok = 0;
#pragma unroll
    for (int r = -1; r < R; ++r)
        if (wrap || (y0 + r >= 0 && y0 + r + 1 < p.H)) ok |= 1u << (r + 1);
    if constexpr (MODE < 0) {
        tile_steps<T, LHY, MODE, R, true, true, NW>(p, s, ph, xch, w, lane, xl, ok);
    } else {
        if (ev) tile_steps<T, LHY, MODE, R, true, true, NW>(p, s, ph, xch, w, lane, xl, ok);
        else if (eh) tile_steps<T, LHY, MODE, R, true, false, NW>(p, s, ph, xch, w, lane, xl, ok);
        else tile_steps<T, LHY, MODE, R, false, false, NW>(p, s, ph, xch, w, lane, xl, ok);
    }

    // columns in [W, pitch) are padding and are written back as the zeros they hold
    const bool own = lane >= A / 2 && lane < A / 2 + p.cols / 2 && xl < p.W;
    const int y_lo = seg * p.rows, y_hi = min(p.H, y_lo + p.rows);
#pragma unroll
    for (int r = 0; r < R; ++r) {
        const int y = y0 + r;
        const unsigned off =
            own && y >= y_lo && y < y_hi ? (unsigned)xl * (unsigned)sizeof(T) + (unsigned)y * row_bytes : kOffNone;
        buf_store<T, 2>(r_out_re, off, 0u, s[r].re);
        buf_store<T, 2>(r_out_im, off, 0u, s[r].im);
    }
    if constexpr (MODE == kTileImag) {
        double q = 0.0, e = 0.0;
#pragma unroll
        for (int r = 0; r < R; ++r) {
            const int y = y0 + r;
            if (!(y >= y_lo && y < y_hi && y >= p.iy0 && y < p.iy1)) continue;   // uniform
            double v = 0.0;
#pragma unroll
            for (int k = 0; k < 2; ++k) {
                const double re = s[r].re[k], im = s[r].im[k];
                v += own && xl + k >= p.ix0 && xl + k < p.ix1 ? re * re + im * im : 0.0;
            }
            const double t = q + v;
            e += fabs(q) >= fabs(v) ? (q - t) + v : (v - t) + q;
            q = t;
        }
        double t = q + e;
        for (int o = kWave / 2; o > 0; o >>= 1) t += __shfl_xor(t, o, kWave);
        __shared__ double red[NW];
        if (lane == 0) red[w] = t;
        __syncthreads();
        if (threadIdx.x == 0) {
            double a = 0.0, c = 0.0;
            for (int i = 0; i < nw; ++i) {
                const double u = a + red[i];
                c += fabs(a) >= fabs(red[i]) ? (a - u) + red[i] : (red[i] - u) + a;
                a = u;
            }
            p.part_out[tile] = a + c;
            if (tile == 0) *p.n_out = gridDim.x;
        }
    }
}

template <typename T, bool LHY, int MODE, int R, int NW>
__global__ void __launch_bounds__(NW * kWave) tile_kernel(TileParams<T> p) {
    __shared__ TileXch<T, NW> xch;
    tile_group<T, LHY, MODE, R, NW>(p, blockIdx.x, xch);
}

// One pass of many lattices: a workgroup per item (lattice, tile).
template <typename T, bool LHY, int MODE, int R, int NW>
__global__ void __launch_bounds__(NW * kWave) tile_batch_kernel(const TileParams<T> *__restrict__ params,
                                                                           const int2 *__restrict__ items) {
    __shared__ TileXch<T, NW> xch;
    const int2 it = items[blockIdx.x];
    const int i = __builtin_amdgcn_readfirstlane(it.x), tile = __builtin_amdgcn_readfirstlane(it.y);
    const TileParams<T> p = params[i];
    tile_group<T, LHY, MODE, R, NW>(p, tile, xch);
}

}  // namespace tsmi
