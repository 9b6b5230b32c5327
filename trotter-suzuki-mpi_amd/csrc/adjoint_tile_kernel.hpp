// adjoint_tile_kernel.hpp -- several reverse steps per launch (adjoint_kernel.hpp
// says what a reverse step is) on register tiles.
//
// adjoint_kernel streams the state and the adjoint state through one row pipeline
// per strip, a step per launch: 1024^2 FP32 puts 5 x 12 strips of waves on the
// chip, whose beats wait for one another.  Here the two states are the two fields
// of pair_tile_kernel's tiles, E's rows stay in registers, and the gradient of
// the tile's own rows is summed over the pass's steps in FP64 registers and added
// to the plane once.
//
// Closed axes, or doubly periodic ones with even extents (WRAP: every plane is
// read from the inner cells, and the halo is written as an exchange would leave it).
#pragma once
#include "adjoint_kernel.hpp"
#include "pair_tile_kernel.hpp"

namespace tsmi {

template <typename T>
struct AdjTileParams {
    const T *in_re[2], *in_im[2];    // psi_{n+1}, G_{n+1}
    T *out_re[2], *out_im[2];        // psi_{n+1-k}, G_{n+1-k}
    const T *e_re, *e_im;
    double *grad;
    int W, H, pitch, nx, ny;
    int steps, n_strips, cols, rows;
    T mH[2], tH[2], mV[2], tV[2], unH[2], unV[2];   // of the step at -dt, the same for both
    T c_nl, c_lhy;
    double gscale;
};

template <typename T, bool NL, int MODE, int R, bool EDGE, int NW>
__device__ __forceinline__ void adj_tile_steps(const AdjTileParams<T> &p, Row<T, 2> (&s)[2][R], const Row<T, 2> (&e)[R],
                                               double (&gr)[R][2], PairXch<T, NW> &x, int w, int lane, int xl,
                                               unsigned ok) {
    two_field_steps<T, false, MODE, R, EDGE, EDGE, NW>(
        p, s, x, w, lane, xl, ok, [](int) {},
        [&](int r0, int r1) {
            auto row = [&](int r) {
                Row<T, 2> &y = s[0][r], &mu = s[1][r];
#pragma unroll
                for (int k = 0; k < 2; ++k)
                    gr[r][k] = fma(p.gscale, double(mu.re[k]) * double(y.im[k]) - double(mu.im[k]) * double(y.re[k]),
                                   gr[r][k]);
                if constexpr (NL) {
                    nl_reverse<T, 2>(y, mu, e[r], p.c_nl, p.c_lhy);
                } else {
                    conj_e_mul(y, e[r]);
                    conj_e_mul(mu, e[r]);
                }
            };
            row(r0);
            row(r1);
            __builtin_amdgcn_sched_barrier(0);
        },
        [](int) {}, [](int) {});
}

template <typename T, bool NL, int MODE, int R, int NW, bool WRAP>
__global__ void __launch_bounds__(NW * kWave, (kPairWaves<T, R, NW, WRAP && MODE >= 0 && !NL>))
adj_tile_kernel(AdjTileParams<T> p) {
    __shared__ PairXch<T, NW> xch;
    typedef typename PairXch<T, NW>::T4 T4;
    const int lane = threadIdx.x & (kWave - 1);
    const int w = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
    const int strip = blockIdx.x % p.n_strips, seg = blockIdx.x / p.n_strips;
    const int A = kApron * p.steps;
    const int X0 = strip * p.cols - A;                            // even
    const int xl = X0 + 2 * lane;
    const int y_tile = WRAP ? seg * p.rows - A : max(0, seg * p.rows - A);
    const int y0 = y_tile + w * R;                                // even

    if (w == 0) {
        const T4 z = {T(0), T(0), T(0), T(0)};
        xch.v[0][1][0][lane] = xch.v[1][1][0][lane] = z;
        xch.v[0][0][NW + 1][lane] = xch.v[1][0][NW + 1][lane] = z;
    }

    const unsigned bytes = (unsigned)p.pitch * (unsigned)p.H * (unsigned)sizeof(T);
    const unsigned row_bytes = (unsigned)p.pitch * (unsigned)sizeof(T);
    auto mod = [](int a, int n) {
        const int r = a % n;
        return r < 0 ? r + n : r;
    };
    int xs = xl;
    bool ld_ok = xl >= 0 && xl + 2 <= p.pitch;
    if (WRAP) {
        xs = kApron + mod(xl - kApron, p.nx);                     // even, nx even: the pair stays together
        ld_ok = true;
    }
    const unsigned v_ld = ld_ok ? (unsigned)xs * (unsigned)sizeof(T) : kOffNone;

    Row<T, 2> s[2][R], e[R];
    double gr[R][2];
    int ys = WRAP ? mod(y0 - kApron, p.ny) : y0;
#pragma unroll
    for (int r = 0; r < R; ++r) {
        const bool in = WRAP || (ys >= 0 && ys < p.H);
        const unsigned off = in ? v_ld + (unsigned)(WRAP ? ys + kApron : ys) * row_bytes : kOffNone;
        ys = WRAP && ys + 1 == p.ny ? 0 : ys + 1;
#pragma unroll
        for (int c = 0; c < 2; ++c) {
            buf_load<T, 2>(make_rsrc(p.in_re[c], bytes), off, 0u, s[c][r].re);
            buf_load<T, 2>(make_rsrc(p.in_im[c], bytes), off, 0u, s[c][r].im);
        }
        buf_load<T, 2>(make_rsrc(p.e_re, bytes), off, 0u, e[r].re);
        buf_load<T, 2>(make_rsrc(p.e_im, bytes), off, 0u, e[r].im);
        gr[r][0] = gr[r][1] = 0.0;
    }
    __syncthreads();

    if constexpr (WRAP && MODE >= 0) {
        adj_tile_steps<T, NL, MODE, R, false>(p, s, e, gr, xch, w, lane, xl, 0u);
    } else {
        unsigned ok = 0;
#pragma unroll
        for (int r = -1; r < R; ++r)
            if (WRAP || (y0 + r >= 0 && y0 + r + 1 < p.H)) ok |= 1u << (r + 1);
        // per wave: see tile_barrier
        const bool edge = X0 < 0 || X0 + kTileCols > p.W || y0 <= 0 || y0 + R >= p.H;
        if (MODE < 0 || edge) {
            adj_tile_steps<T, NL, MODE, R, true>(p, s, e, gr, xch, w, lane, xl, ok);
        } else if constexpr (MODE >= 0) {
            adj_tile_steps<T, NL, MODE, R, false>(p, s, e, gr, xch, w, lane, xl, ok);
        }
    }

    const bool own = lane >= A / 2 && lane < A / 2 + p.cols / 2 && xl < p.W;
    const int y_lo = seg * p.rows, y_hi = min(p.H, y_lo + p.rows);
    const __amdgpu_buffer_rsrc_t r_grad = make_rsrc(p.grad, (unsigned)p.pitch * (unsigned)p.H * 8u);
#pragma unroll
    for (int r = 0; r < R; ++r) {
        const int y = y0 + r;
        const bool mine = own && y >= y_lo && y < y_hi;
        const unsigned off = mine ? (unsigned)xl * (unsigned)sizeof(T) + (unsigned)y * row_bytes : kOffNone;
        const unsigned off_d = mine ? (unsigned)xl * 8u + (unsigned)y * (unsigned)p.pitch * 8u : kOffNone;
        double g[2];
        buf_load_f64<T, 2>(r_grad, off_d, 0u, g);
        g[0] += gr[r][0];
        g[1] += gr[r][1];
        buf_store_f64<T, 2>(r_grad, off_d, 0u, g);
#pragma unroll
        for (int c = 0; c < 2; ++c) {
            buf_store<T, 2>(make_rsrc(p.out_re[c], bytes), off, 0u, s[c][r].re);
            buf_store<T, 2>(make_rsrc(p.out_im[c], bytes), off, 0u, s[c][r].im);
        }
    }
}

}  // namespace tsmi
