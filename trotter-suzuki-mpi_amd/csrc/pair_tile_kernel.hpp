// pair_tile_kernel.hpp -- both components of a small or medium two-component
// lattice in register tiles: several real-time steps per launch, or one
// imaginary-time step with everything between two steps folded into its loads.
//
// The streaming passes (pair_kernel, pair2_kernel) run such a lattice as a few
// dozen waves, each alone on its SIMD, whose row updates wait for one another,
// and imaginary time adds a pass and two ticketed reductions per step.  This is
// tile_kernel's layout for two components: a workgroup holds 128 columns x
// (NW R) rows of both in registers, one LDS exchange per vertical pass carries a
// border column of both, and the apron is 4 cells per step.  Each potential pass
// sees the other component's density at the start of the step, so neighbouring
// V0 passes stay apart (four exchanges per step); the angle's constant part
// (phase plane + that density) is formed while the first exchange is on its way.
//
// Real time: the Rabi rotation runs on the rows in registers between steps.
// Imaginary time: a step divides each component by its norm, rotates, and
// divides both by the joint norm (src/cpukernel.cpp:551-563, :581-667).  All
// three are one 2 x 2 matrix for every cell, which follows from three sums over
// the step's output -- sum |a|^2, sum |b|^2 and the cross term Re(s conj(a) b) of
// the rotation -- so a step stores its raw output and its workgroups' partial
// sums, and every wave of the next launch adds the partials in order and applies
// the matrix (in FP64, one rounding) as it loads.  pair_finish_kernel does the
// same after the last step.  The norms after the rotation, the next step's targets,
// follow from the same sums, unless the rotation cancels most of a component (a state
// on its way to the antiphase ground state passes there): then the launch that applied
// the matrix sums what it loaded, and that sum is the target.
//
// The edges of a closed tile take per-lane and per-row pair factors; a periodic
// lattice has none, and its kernels (WRAP) are compiled without that code, which
// leaves FP32 tiles of 4 rows 119 VGPRs (two workgroups per CU) instead of 153,
// and those of 8 rows 231 instead of spilling (1024^2 FP32 17.1 -> 12.2 us per step).
//
// Measured, us per step, streamed -> tiles: 1024^2 periodic real FP32 29.5 -> 11.1
// (its 3 planes in and 2 out of both components, 43 MB, and 4.5 us per launch of
// two steps, then instruction issue), 512^2 FP64 62 -> 8.3, 250^2 closed
// imaginary FP64 101 -> 11.0 (launch, partial sums and three rows' latency).
#pragma once
#include "pair_kernel.hpp"
#include "tile_kernel.hpp"

namespace tsmi {

// Partial sums of an imaginary-time launch: of its output sum |a|^2, sum |b|^2 and
// sum Re(s conj(a) b); of its input, the pending matrix applied, sum |a|^2, sum |b|^2
// (only where the matrix asks for them).
constexpr int kPairSums = 5, kPairOut = 3;

// Waves per SIMD asked of the compiler for a workgroup of NW waves.  FP32 with 4
// rows: two workgroups of 8 waves on a CU, so that one loads or stores while the
// other computes.
template <typename T, int R, int NW, bool PLAIN>
constexpr int kPairWaves = PLAIN && sizeof(T) == 4 && R == 4 && NW == 8 ? 4 : NW / 4;

// What follows from the sums of an imaginary-time step (see the top).
struct PairNorm {
    const double *part;              // partial sums [kPairSums][cap] of the step before (nullptr: none)
    const int *n;                    // their count
    int cap;
    const double *norm_in;           // squared-norm targets of that step (0: no division, < 0: the input's sum)
    double *norm_out;                // targets after it
    double cc, cs_r, cs_i;           // its rotation
    int rabi;
    double dxdy, tot_norm;
};

// a <- aa a + ab b, b <- bb b + ba a; off-diagonals (x, y) = x + i y.
struct PairMatrix {
    double aa, bb, ab_r, ab_i, ba_r, ba_i;
    bool sums;                       // a target is the sum over what the matrix gives
};

// Partial sums j0 .. j0 + N - 1 added up in order, the same bits in every wave.
template <int N>
__device__ __forceinline__ void pair_add(const PairNorm &q, int j0, int lane, double (&s)[N]) {
    const int n = __builtin_amdgcn_readfirstlane(*q.n);
    double e[N];
#pragma unroll
    for (int j = 0; j < N; ++j) s[j] = e[j] = 0.0;
    for (int i = lane; i < n; i += kWave)
#pragma unroll
        for (int j = 0; j < N; ++j) neumaier(s[j], e[j], q.part[(long)(j0 + j) * q.cap + i]);
#pragma unroll
    for (int j = 0; j < N; ++j) {
        s[j] += e[j];
        for (int o = kWave / 2; o > 0; o >>= 1) s[j] += __shfl_xor(s[j], o, kWave);
    }
}

// A norm after a rotation, of the terms it is made of: relative to the total, or -1
// where they cancel to less than a quarter and its relative error would exceed 1e-15.
__device__ __forceinline__ double pair_target(double q, double terms, double total, double tot_norm) {
    return q >= 0.25 * terms && q > 0.0 ? q / total * tot_norm : -1.0;
}

// The matrix of a pending renormalisation, the same bits in every wave; the
// wave with `store` also leaves the new targets.
__device__ __forceinline__ PairMatrix pair_matrix(const PairNorm &q, int lane, bool store) {
    PairMatrix m = {1.0, 1.0, 0.0, 0.0, 0.0, 0.0, false};
    if (!q.part) return m;
    double s[kPairOut];
    pair_add(q, 0, lane, s);
    double na = q.norm_in[0], nb = q.norm_in[1];
    if (na < 0.0 || nb < 0.0) {
        double t[2];
        pair_add(q, kPairOut, lane, t);
        if (na < 0.0) na = t[0] * q.dxdy;
        if (nb < 0.0) nb = t[1] * q.dxdy;
    }
    const double ia = na != 0.0 ? 1.0 / sqrt(s[0] * q.dxdy / na) : 1.0;
    const double ib = nb != 0.0 ? 1.0 / sqrt(s[1] * q.dxdy / nb) : 1.0;
    if (!q.rabi) {
        m.aa = ia;
        m.bb = ib;
        if (store) {
            q.norm_out[0] = na;
            q.norm_out[1] = nb;
        }
        return m;
    }
    const double c2 = q.cc * q.cc, s2 = q.cs_r * q.cs_r + q.cs_i * q.cs_i;
    // a divided component's norm is its target itself: recomputed from the sum, its
    // rounding would repeat as the state converges and drift the targets' ratio
    // (5.6e-14 after 1000 steps)
    const double va = na != 0.0 ? na : s[0] * q.dxdy, vb = nb != 0.0 ? nb : s[1] * q.dxdy;
    const double x = 2.0 * q.cc * (s[2] * q.dxdy) * ia * ib;
    const double qa = c2 * va + s2 * vb + x, qb = c2 * vb + s2 * va + x;
    const double f = 1.0 / sqrt((qa + qb) / q.tot_norm);
    m.aa = q.cc * ia * f;
    m.bb = q.cc * ib * f;
    m.ab_r = q.cs_r * ib * f;
    m.ab_i = q.cs_i * ib * f;
    m.ba_r = q.cs_r * ia * f;
    m.ba_i = -q.cs_i * ia * f;
    const double ta = pair_target(qa, c2 * va + s2 * vb, qa + qb, q.tot_norm);
    const double tb = pair_target(qb, c2 * vb + s2 * va, qa + qb, q.tot_norm);
    m.sums = ta < 0.0 || tb < 0.0;
    if (store) {
        q.norm_out[0] = ta;
        q.norm_out[1] = tb;
    }
    return m;
}

template <typename T>
__device__ __forceinline__ void pair_apply(const PairMatrix &m, T &ar, T &ai, T &br, T &bi) {
    const double xr = ar, xi = ai, yr = br, yi = bi;
    ar = T(m.aa * xr + (m.ab_r * yr - m.ab_i * yi));
    ai = T(m.aa * xi + (m.ab_r * yi + m.ab_i * yr));
    br = T(m.bb * yr + (m.ba_r * xr - m.ba_i * xi));
    bi = T(m.bb * yi + (m.ba_r * xi + m.ba_i * xr));
}

template <typename T>
struct PairTileParams {
    const T *in_re[2], *in_im[2];
    T *out_re[2], *out_im[2];
    const T *ph[2];
    int W, H, pitch;
    int nx, ny;                      // as TileParams
    int seam, px, py;                // as TileParams
    int steps;
    int n_strips, cols, rows;
    T mH[2], tH[2], mV[2], tV[2], unH[2], unV[2];
    T c_self[2], c_ab;
    double mag[2];
    // real time: the rotation after every step but the last of the pass, and after that one
    double cc, cs_r, cs_i, cc2, cs_r2, cs_i2;
    int rabi;
    // imaginary time
    PairNorm pend;                   // of the step before
    double s_r, s_i;                 // s of the rotation after this step
    double *part_out;                // this step's partial sums, one set per workgroup
    int *n_out;
    int cap;
    int ix0, ix1, iy0, iy1;
};

template <typename T, int NW>
struct PairXch {
    typedef T __attribute__((ext_vector_type(4))) T4;
    T4 v[2][2][NW + 2][kWave];   // as TileXch: (a re, a im, b re, b im)
};

// p.steps steps of two fields on a tile held in registers (p: pair factors per
// field, extents).  EH: the strip reaches past the tile's left or right edge
// (per-lane factors); EV: so do the wave's rows at the top or bottom (bit r + 1 of
// ok: rows r and r + 1 of the wave are both inside).  begin(st) runs before a step
// changes the state, mid(r0, r1) is the potential stage of two rows, used(st) runs
// after the last of them, end(st) after the step.
template <typename T, bool IMAG, int MODE, int R, bool EH, bool EV, int NW, typename P, typename Begin, typename Mid,
          typename Used, typename End>
__device__ __forceinline__ void two_field_steps(const P &p, Row<T, 2> (&s)[2][R], PairXch<T, NW> &x, int w, int lane,
                                                int xl, unsigned ok, Begin &&begin, Mid &&mid, Used &&used, End &&end) {
    static_assert(R % 2 == 0 && R >= 4, "row parities are fixed per register");
    typedef typename PairXch<T, NW>::T4 T4;
    constexpr int M = MODE < 0 ? 0 : MODE;
    // a periodic lattice has no edge: every column far from one
    HCoef<T, 2> hc0 = {}, hc1 = {};
    if constexpr (EH) {
        const int xe = p.nx ? 2 * lane + 2 : xl, We = p.nx ? 1 << 30 : p.W;
        hc0 = make_hcoef<T, 2>(xe, lane, We, p.mH[0], p.tH[0], p.unH[0]);
        hc1 = make_hcoef<T, 2>(xe, lane, We, p.mH[1], p.tH[1], p.unH[1]);
    }
    const T kH[2] = {M == 0 ? p.tH[0] : p.mH[0], M == 0 ? p.tH[1] : p.mH[1]};
    int buf = 0;

    auto hrow = [&](auto ss, auto rr, int r) {
        constexpr int PAR = (decltype(ss)::value + decltype(rr)::value) & 1;
        if constexpr (EH) {
            hpass<PAR, IMAG>(s[0][r], hc0);
            hpass<PAR, IMAG>(s[1][r], hc1);
        } else {
            hpass_fast<PAR, IMAG, M>(s[0][r], kH[0]);
            hpass_fast<PAR, IMAG, M>(s[1][r], kH[1]);
        }
    };
    // V(S); `rest` runs between the exchange's write and its barrier
    auto vpass = [&](auto ss, auto &&rest) {
        constexpr int S = decltype(ss)::value, CX = 1 - S;
        T4 top, bot;
        top[0] = s[0][0].re[CX]; top[1] = s[0][0].im[CX]; top[2] = s[1][0].re[CX]; top[3] = s[1][0].im[CX];
        bot[0] = s[0][R - 1].re[CX]; bot[1] = s[0][R - 1].im[CX];
        bot[2] = s[1][R - 1].re[CX]; bot[3] = s[1][R - 1].im[CX];
        x.v[buf][0][w + 1][lane] = top;
        x.v[buf][1][w + 1][lane] = bot;
        rest();
        tile_barrier();
        const T4 up = x.v[buf][1][w][lane], dn = x.v[buf][0][w + 2][lane];
        buf ^= 1;
#pragma unroll
        for (int c = 0; c < 2; ++c) {
            const T m = p.mV[c], t = p.tV[c], un = p.unV[c], k = M == 0 ? t : m;
            // bit r + 1 of ok: rows r and r + 1 are both inside; a cell without a
            // partner is multiplied by un
            auto pair = [&](int col, int r) {
                Row<T, 2> &u = s[c][r], &l = s[c][r + 1];
                if constexpr (EV) {
                    const bool in = ok >> (r + 1) & 1u;
                    rot<IMAG>(in ? m : un, in ? t : T(0), u.re[col], u.im[col], l.re[col], l.im[col]);
                } else {
                    fpair<IMAG, M>(k, u.re[col], u.im[col], l.re[col], l.im[col]);
                }
            };
#pragma unroll
            for (int r = 0; r + 1 < R; r += 2) pair(S, r);
#pragma unroll
            for (int r = 1; r + 1 < R; r += 2) pair(CX, r);
            Row<T, 2> &f = s[c][0], &l = s[c][R - 1];
            const T ur = up[2 * c], ui = up[2 * c + 1], dr = dn[2 * c], di = dn[2 * c + 1];
            if constexpr (EV) {
                const bool in0 = ok & 1u, in1 = ok >> R & 1u;
                rot_q<IMAG>(in0 ? m : un, in0 ? t : T(0), ur, ui, f.re[CX], f.im[CX]);
                rot_p<IMAG>(in1 ? m : un, in1 ? t : T(0), l.re[CX], l.im[CX], dr, di);
            } else {
                fpair_q<IMAG, M>(k, ur, ui, f.re[CX], f.im[CX]);
                fpair_p<IMAG, M>(k, l.re[CX], l.im[CX], dr, di);
            }
        }
    };
    using I0 = std::integral_constant<int, 0>;
    using I1 = std::integral_constant<int, 1>;
    auto h_border = [&](auto ss) {
        hrow(ss, I0(), 0);
        hrow(ss, I1(), R - 1);
    };
    auto h_rest = [&](auto ss) {
#pragma unroll
        for (int r = 1; r + 1 < R; r += 2) {
            hrow(ss, I1(), r);
            hrow(ss, I0(), r + 1);
        }
    };
    for (int st = 0; st < p.steps; ++st) {
        vpass(I0(), [&] { begin(st); });
        h_border(I0());
        vpass(I1(), [&] { h_rest(I0()); });
        h_border(I1());
        h_rest(I1());
        mid(0, R - 1);
        h_border(I1());
        vpass(I1(), [&] {
#pragma unroll
            for (int r = 1; r + 1 < R; r += 2) mid(r, r + 1);
            used(st);
            h_rest(I1());
        });
        h_border(I0());
        vpass(I0(), [&] { h_rest(I0()); });
        end(st);
    }
}

// The steps of the two components.
template <typename T, bool IMAG, int MODE, int R, bool EDGE, int NW, typename LoadPh>
__device__ __forceinline__ void pair_tile_steps(const PairTileParams<T> &p, Row<T, 2> (&s)[2][R],
                                                PairXch<T, NW> &x, int w, int lane, int xl, unsigned ok,
                                                LoadPh &&load_ph) {
    // phase plane, plus the other component's start-of-step density; the plane is
    // read anew for each step as soon as the potential pass of the one before has
    // used it (it stays in the L2), which holds one set of registers, not two
    T base[2][R][2];
    load_ph(base);
    two_field_steps<T, IMAG, MODE, R, EDGE, EDGE, NW>(
        p, s, x, w, lane, xl, ok,
        [&](int) {
#pragma unroll
            for (int r = 0; r < R; ++r) {
                T na[2], nb[2];
                density(s[0][r], na);
                density(s[1][r], nb);
#pragma unroll
                for (int k = 0; k < 2; ++k) {
                    base[0][r][k] += p.c_ab * nb[k];
                    base[1][r][k] += p.c_ab * na[k];
                }
            }
        },
        [&](int r0, int r1) {
#pragma unroll
            for (int c = 0; c < 2; ++c)
                tile_ppass<T, false, IMAG, 2>(s[c][r0], s[c][r1], base[c][r0], base[c][r1], p.c_self[c], T(0), p.mag[c]);
            __builtin_amdgcn_sched_barrier(0);   // one group of rows at a time: fewer registers at once
        },
        [&](int st) {
            if (st + 1 < p.steps) load_ph(base);
        },
        [&](int st) {
            // always, by the identity when there is no coupling: a branch would merge
            // two versions of the state, and did so in copies of every register
            if constexpr (!IMAG) {
                const bool last = st == p.steps - 1;
                const double cc = last ? p.cc2 : p.cc, sr = last ? p.cs_r2 : p.cs_r, si = last ? p.cs_i2 : p.cs_i;
#pragma unroll
                for (int r = 0; r < R; ++r) {
                    rabi_rows<T, 2>(s[0][r], s[1][r], cc, sr, si);
                    __builtin_amdgcn_sched_barrier(0);
                }
            }
        });
}

template <typename T, bool IMAG, int MODE, int R, int NW, bool WRAP>
__global__ void __launch_bounds__(NW * kWave, (kPairWaves<T, R, NW, WRAP && MODE >= 0>)) pair_tile_kernel(PairTileParams<T> p) {
    __shared__ PairXch<T, NW> xch;
    typedef typename PairXch<T, NW>::T4 T4;
    const int lane = threadIdx.x & (kWave - 1);
    const int w = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
    constexpr int nw = NW;
    const int strip = blockIdx.x % p.n_strips, seg = blockIdx.x / p.n_strips;
    const int A = kApron * p.steps;
    constexpr bool wrap = WRAP;
    const int X0 = strip * p.cols - A;                            // even
    const int xl = X0 + 2 * lane;
    const int y_tile = wrap ? seg * p.rows - A : max(0, seg * p.rows - A);
    const int y0 = y_tile + w * R;                                // even

    if (w == 0) {
        const T4 z = {T(0), T(0), T(0), T(0)};
        xch.v[0][1][0][lane] = xch.v[1][1][0][lane] = z;
        xch.v[0][0][nw + 1][lane] = xch.v[1][0][nw + 1][lane] = z;
    }

    const unsigned bytes = (unsigned)p.pitch * (unsigned)p.H * (unsigned)sizeof(T);
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
    // row offsets; rows outside a closed tile (zeros that never meet it) take the
    // nearest row's phases
    unsigned so[R];
    int ys = wrap ? mod(y0 - kApron, p.ny) : y0;
#pragma unroll
    for (int r = 0; r < R; ++r) {
        so[r] = (unsigned)(wrap ? ys + kApron : min(max(ys, 0), p.H - 1)) * row_bytes;
        ys = wrap && ys + 1 == p.ny ? 0 : ys + 1;
    }
    auto load_ph = [&](T (&b)[2][R][2]) {
#pragma unroll
        for (int r = 0; r < R; ++r)
#pragma unroll
            for (int c = 0; c < 2; ++c) buf_load<T, 2>(make_rsrc(p.ph[c], bytes), v_ld, so[r], b[c][r]);
    };

    Row<T, 2> s[2][R];
#pragma unroll
    for (int r = 0; r < R; ++r) {
        const bool in = wrap || (y0 + r >= 0 && y0 + r < p.H);
        const unsigned off = in ? v_ld + so[r] : kOffNone;
#pragma unroll
        for (int c = 0; c < 2; ++c) {
            if (!WRAP && p.seam) continue;
            buf_load<T, 2>(make_rsrc(p.in_re[c], bytes), off, 0u, s[c][r].re);
            buf_load<T, 2>(make_rsrc(p.in_im[c], bytes), off, 0u, s[c][r].im);
        }
    }
    if (!WRAP && p.seam) {
        const SeamTile q = {p.W, p.H, p.px, p.py};
#pragma unroll
        for (int r = 0; r < R; ++r)
#pragma unroll
            for (int c = 0; c < 2; ++c)
                seam_load<T>(q, make_rsrc(p.in_re[c], bytes), make_rsrc(p.in_im[c], bytes), xl, y0 + r, row_bytes,
                             s[c][r]);
    }
    const bool own = lane >= A / 2 && lane < A / 2 + p.cols / 2 && xl < p.W;
    const int y_lo = seg * p.rows, y_hi = min(p.H, y_lo + p.rows);
    __shared__ double red[IMAG ? kPairSums : 1][NW];
    if constexpr (IMAG) {
        if (lane == 0) red[kPairOut][w] = red[kPairOut + 1][w] = 0.0;
        if (p.pend.part) {
            const PairMatrix m = pair_matrix(p.pend, lane, blockIdx.x == 0 && threadIdx.x == 0);
#pragma unroll
            for (int r = 0; r < R; ++r)
#pragma unroll
                for (int k = 0; k < 2; ++k)
                    pair_apply(m, s[0][r].re[k], s[0][r].im[k], s[1][r].re[k], s[1][r].im[k]);
            if (__builtin_expect(m.sums, 0)) {
                for (int c = 0; c < 2; ++c) {
                    double q = 0.0, e = 0.0;
#pragma unroll
                    for (int r = 0; r < R; ++r)
#pragma unroll
                        for (int k = 0; k < 2; ++k) {
                            const int y = y0 + r, x = xl + k;
                            const double re = c ? s[1][r].re[k] : s[0][r].re[k], im = c ? s[1][r].im[k] : s[0][r].im[k];
                            const bool in = own && y >= y_lo && y < y_hi && y >= p.iy0 && y < p.iy1 && x >= p.ix0 &&
                                            x < p.ix1;
                            neumaier(q, e, in ? re * re + im * im : 0.0);
                        }
                    double t = q + e;
                    for (int o = kWave / 2; o > 0; o >>= 1) t += __shfl_xor(t, o, kWave);
                    if (lane == 0) red[kPairOut + c][w] = t;
                }
            }
        }
    }
    __syncthreads();

    if constexpr (WRAP && MODE >= 0) {
        pair_tile_steps<T, IMAG, MODE, R, false>(p, s, xch, w, lane, xl, 0u, load_ph);
    } else {
        unsigned ok = 0;
#pragma unroll
        for (int r = -1; r < R; ++r)
            if (wrap || (y0 + r >= 0 && y0 + r + 1 < p.H)) ok |= 1u << (r + 1);
        // per wave: see tile_barrier
        const bool edge = X0 < 0 || X0 + kTileCols > p.W || y0 <= 0 || y0 + R >= p.H;
        if (MODE < 0 || edge) {
            pair_tile_steps<T, IMAG, MODE, R, true>(p, s, xch, w, lane, xl, ok, load_ph);
        } else if constexpr (MODE >= 0) {
            pair_tile_steps<T, IMAG, MODE, R, false>(p, s, xch, w, lane, xl, ok, load_ph);
        }
    }

#pragma unroll
    for (int r = 0; r < R; ++r) {
        const int y = y0 + r;
        const unsigned off =
            own && y >= y_lo && y < y_hi ? (unsigned)xl * (unsigned)sizeof(T) + (unsigned)y * row_bytes : kOffNone;
#pragma unroll
        for (int c = 0; c < 2; ++c) {
            buf_store<T, 2>(make_rsrc(p.out_re[c], bytes), off, 0u, s[c][r].re);
            buf_store<T, 2>(make_rsrc(p.out_im[c], bytes), off, 0u, s[c][r].im);
        }
    }
    if constexpr (IMAG) {
        double q[kPairOut], e[kPairOut];
#pragma unroll
        for (int j = 0; j < kPairOut; ++j) q[j] = e[j] = 0.0;
#pragma unroll
        for (int r = 0; r < R; ++r) {
            const int y = y0 + r;
            if (!(y >= y_lo && y < y_hi && y >= p.iy0 && y < p.iy1)) continue;   // uniform
            double v[kPairOut] = {0.0, 0.0, 0.0};
#pragma unroll
            for (int k = 0; k < 2; ++k) {
                const bool in = own && xl + k >= p.ix0 && xl + k < p.ix1;
                const double ar = s[0][r].re[k], ai = s[0][r].im[k], br = s[1][r].re[k], bi = s[1][r].im[k];
                v[0] += in ? ar * ar + ai * ai : 0.0;
                v[1] += in ? br * br + bi * bi : 0.0;
                v[2] += in ? p.s_r * (ar * br + ai * bi) - p.s_i * (ar * bi - ai * br) : 0.0;
            }
#pragma unroll
            for (int j = 0; j < kPairOut; ++j) neumaier(q[j], e[j], v[j]);
        }
#pragma unroll
        for (int j = 0; j < kPairOut; ++j) {
            double t = q[j] + e[j];
            for (int o = kWave / 2; o > 0; o >>= 1) t += __shfl_xor(t, o, kWave);
            if (lane == 0) red[j][w] = t;
        }
        __syncthreads();
        if (threadIdx.x < kPairSums) {
            double a = 0.0, c = 0.0;
            for (int i = 0; i < nw; ++i) neumaier(a, c, red[threadIdx.x][i]);
            p.part_out[(long)threadIdx.x * p.cap + blockIdx.x] = a + c;
        }
        if (blockIdx.x == 0 && threadIdx.x == 0) *p.n_out = gridDim.x;
    }
}

// The pending matrix applied to both tiles in place, the new targets stored, and the
// sums they may stand for (sums 3 and 4 of part_out, as an imaginary-time launch's).
constexpr int kFinishBlocks = 256;
template <typename T>
__global__ void __launch_bounds__(256) pair_finish_kernel(T *ar, T *ai, T *br, T *bi, int W, int H, int pitch, int ix0,
                                                          int ix1, int iy0, int iy1, PairNorm q, double *part_out,
                                                          int *n_out) {
    const int lane = threadIdx.x & (kWave - 1);
    const PairMatrix m = pair_matrix(q, lane, blockIdx.x == 0 && threadIdx.x == 0);
    const long n = (long)W * H;
    double t[2] = {0.0, 0.0}, e[2] = {0.0, 0.0};
    for (long i = blockIdx.x * 256L + threadIdx.x; i < n; i += gridDim.x * 256L) {
        const long y = i / W, x = i - y * W, k = y * pitch + x;
        T xr = ar[k], xi = ai[k], yr = br[k], yi = bi[k];
        pair_apply(m, xr, xi, yr, yi);
        ar[k] = xr;
        ai[k] = xi;
        br[k] = yr;
        bi[k] = yi;
        if (m.sums && x >= ix0 && x < ix1 && y >= iy0 && y < iy1) {
            neumaier(t[0], e[0], double(xr) * double(xr) + double(xi) * double(xi));
            neumaier(t[1], e[1], double(yr) * double(yr) + double(yi) * double(yi));
        }
    }
    __shared__ double red[2][256 / kWave];
#pragma unroll
    for (int c = 0; c < 2; ++c) {
        t[c] += e[c];
        for (int o = kWave / 2; o > 0; o >>= 1) t[c] += __shfl_xor(t[c], o, kWave);
        if (lane == 0) red[c][threadIdx.x / kWave] = t[c];
    }
    __syncthreads();
    if (threadIdx.x < 2) {
        double a = 0.0, c = 0.0;
        for (int i = 0; i < 256 / kWave; ++i) neumaier(a, c, red[threadIdx.x][i]);
        part_out[(long)(kPairOut + threadIdx.x) * q.cap + blockIdx.x] = a + c;
    }
    if (blockIdx.x == 0 && threadIdx.x == 0) *n_out = gridDim.x;
}

// The targets a finished call leaves: those of its last rotation, or the sums.
template <typename = void>
__global__ void __launch_bounds__(kWave) pair_targets_kernel(PairNorm q) {
    double t[2];
    pair_add(q, kPairOut, threadIdx.x, t);
    if (threadIdx.x < 2 && q.norm_out[threadIdx.x] < 0.0) q.norm_out[threadIdx.x] = t[threadIdx.x] * q.dxdy;
}

}  // namespace tsmi
