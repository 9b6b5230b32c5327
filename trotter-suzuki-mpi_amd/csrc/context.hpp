// context.hpp -- the single-component context (tsmi_ctx) shared by the
// library's translation units.
//
// A context owns two device copies of the tile (ping-pong: a step reads one and
// writes the other, as CPUBlock does with its two buffers,
// src/cpukernel.cpp:244-247), the E planes, the raw potential and the
// coordinate tables.  The two-component context (tsmi_pair.hip) is built from
// two of them, one per component, on one stream.
#pragma once
#include <hip/hip_runtime.h>

#include <vector>

#include "stage.hpp"
#include "tsmi_hip.h"

struct tsmi_ctx {
    tsmi_desc d;
    int W = 0, H = 0, pitch = 0, esz = 0, vec = 0;
    int n_strips = 0, n_segs = 0, seg_rows = 0, n_waves = 0;
    // Views at the origin of the reference tile (W x H, row pitch `pitch`).  With
    // the 8-wide halo layout they sit 4 rows and 4 columns inside allocations of
    // Wd x Hd = (W + 8) x (H + 8); otherwise view and allocation coincide.
    void *psi_re[2] = {nullptr, nullptr}, *psi_im[2] = {nullptr, nullptr};
    void *e_re = nullptr, *e_im = nullptr;
    void *psi_base[2][2] = {{nullptr, nullptr}, {nullptr, nullptr}};
    void *e_base[2] = {nullptr, nullptr};
    void *e8[2] = {nullptr, nullptr};     // E wrapped over the whole 8-wide halo (fused passes)
    // E corr as one plane (phase in real time, exponent in imaginary time): the
    // steps read it instead of E when ph_mode (every |E| = 1, or every E > 0)
    void *ph_base = nullptr, *ph = nullptr, *ph8 = nullptr;
    bool ph_mode = false;
    bool e_wraps = false;                // doubly periodic: E's halo is known to repeat the inner cells
    unsigned *flag = nullptr;             // set by the E import when E has no phase form
    double *v_base = nullptr;
    int Wd = 0, Hd = 0;
    size_t off_el = 0;                    // elements from allocation to view origin
    bool halo8 = false;
    bool nt_out = false;                  // FP64 real time: output rows stored non-temporal
    // kernel timing (tsmi_kernel_timing): one event pair per step-kernel launch
    bool timing = false;
    std::vector<hipEvent_t> ev[2][2];     // [fused?][start/end]
    size_t ev_used[2] = {0, 0};
    // fused two-step passes (fused_kernel.hpp)
    int sweeps = 1;
    int n_strips2 = 0, n_segs2 = 0, seg_rows2 = 0, n_waves2 = 0;
    int geo2_key = -1;                    // (form, E form) the segments were sized for; -1: none
    double *v = nullptr, *xc = nullptr, *yc = nullptr;
    // imaginary time: two slots of per-wave partial sums (one per step parity),
    // their counts, and one divisor for host-side readers (divisor_kernel)
    double *div = nullptr;
    double *partials = nullptr;
    int *part_n = nullptr;
    int part_cap = 0;                    // partial sums per slot
    double *obs_partials = nullptr;      // kObsBlocksMax * OBS_COUNT block partials
    double *obs_out = nullptr;           // kObsOut results of the last observables pass
    int obs_blocks = 0;
    int cur = 0, div_slot = 0;
    bool div_pending = false, has_state = false, has_e = false, has_v = false;
    hipStream_t own = nullptr, stream = nullptr;
    double aH = 0, bH = 0, aV = 0, bV = 0, c_nl = 0, c_lhy = 0;   // FP64, as the reference
    // scaled-frame factors actually used by the kernel (values of the kernel precision)
    double mH = 1, tH = 0, mV = 1, tV = 0, unH = 1, unV = 1;
    double corr_re = 1.0, corr_im = 0.0;   // folded into E
    double c_nl_s = 0, c_lhy_s = 0;        // couplings rescaled to the mid-step frame
    int mode = 0;                          // 0 / 1: both axes in form A / B; -1: mixed
    int ix0 = 0, ix1 = 0, iy0 = 0, iy1 = 0;
    // reverse sweep (real time, closed axes, no nonlinearity)
    bool adj_ok = false;
    double amH = 1, atH = 0, amV = 1, atV = 0, aunH = 1, aunV = 1;   // frame of the step at -dt
    double corr_abs = 1.0;                                         // |corr| = |kappa|^2
    void *ck = nullptr;               // checkpoints: 2 planes each
    size_t ck_cap = 0;
    int ck_every = 0, ck_steps = 0, ck_count = 0;
    bool ck_valid = false;
    void *adj = nullptr;              // 8 planes: adjoint re/im x2, reversed state re/im x2
    double *grad = nullptr;           // FP64, pitched
    tsmi::HostStage stage;            // pinned chunks of the host transfers
};

namespace tsmi {

// The periodic halo refresh of one state allocation of c (re/im planes in the
// context precision), asynchronous on c's stream.
int ctx_exchange(tsmi_ctx *c, void *re, void *im);

// One event of the pair around a step-kernel launch when timing is on (kind 1:
// several steps per launch; which 0: before, 1: after).
int ctx_time_mark(tsmi_ctx *c, int kind, int which);

// Tile passes (tsmi_tile.hip), asynchronous on c's stream.
// How a call of n steps runs: streamed; on the tile closed at its edges, several
// steps per launch; on the doubly periodic lattice, several steps per launch
// between a first and a last step of their own, E read from the inner cells; step by
// step, the state's halo read from the cells it mirrors and E's as it is.  E's halo
// may differ from the inner cells: real time reads those in the streamed two-step
// passes too, imaginary time (one step per launch) does only when e_wraps.
enum TileRoute { kRouteStream, kRouteClosed, kRouteWrap, kRouteSeam };
TileRoute tile_route(const tsmi_desc &d, int W, int H, int n, bool e_wraps);   // E in one plane
TileRoute tile_route(const tsmi_ctx *c, int n);
// The cells of the tiles that cover W x H cells: columns in whole tile widths, rows in
// whole heights of the lowest common tile.
long tile_area(int W, int H);
// Rows per wave, waves, steps and workgroups of the longest pass of such a call (0s:
// streamed).
void tile_geometry(const tsmi_desc &d, int W, int H, int n, int32_t out[4]);
// n steps as one or several passes, on the tile closed at its edges or (wrap) on the
// periodic lattice, the halo refreshed.
int tile_passes(tsmi_ctx *c, int n, bool wrap);
// n steps, each starting with the halo exchange that has not been run yet (the
// state's halo cells are read from the cells they mirror).
int tile_seam_steps(tsmi_ctx *c, int n);
// Workgroups of a pass of one step.
int tile_blocks(const tsmi_ctx *c);

// Reverse sweep as tile passes (tsmi_adjoint_tile.hip): whether it runs so; the
// steps of a pass, at most `most`; one pass of that many reverse steps, field 0 the
// state, field 1 the adjoint state, planes (re, im) of the reference tile.
struct AdjTileIo {
    const void *in[2][2];
    void *out[2][2];
};
bool adjoint_tiles_run(const tsmi_ctx *c);
int adjoint_tile_steps(const tsmi_ctx *c, int most);
int adjoint_tile_pass(tsmi_ctx *c, int steps, const AdjTileIo &io);

}  // namespace tsmi
