// pair_context.hpp -- the two-component context (tsmi_pair) shared by the
// library's translation units.
#pragma once
#include "context.hpp"

struct tsmi_pair {
    tsmi_ctx *c[2] = {nullptr, nullptr};
    int esz = 0, vec = 0;
    bool imag = false;
    double dt = 0, c_ab = 0, omega_r = 0, omega_i = 0, g_ab = 0, tot_norm = 0;
    int W = 0, H = 0, pitch = 0;
    int n_strips = 0, seg_rows = 0, n_segs = 0, n_waves = 0, rabi_blocks = 0;
    // two steps per pass (pair2_kernel) over the whole allocation, Wd x Hd
    bool fused = false, halo8 = false;
    int Wd = 0, Hd = 0, n_strips2 = 0, seg_rows2 = 0, n_segs2 = 0, n_waves2 = 0;
    int ix0 = 0, ix1 = 0, iy0 = 0, iy1 = 0;
    // device scalars: divisor pairs [2][2] (a pending pair is read while the
    // next one is written), norm targets [2][2] (the same, in the tile passes)
    double *dv = nullptr;
    double *partials = nullptr;
    unsigned *counter = nullptr;
    int slot = 0, norm_slot = 0;
    bool pending = false;
    // tile passes (pair_tile_kernel.hpp): taken at all; imaginary time's partial
    // sums, two slots of kPairSums x part_cap doubles, and their two counts
    bool tiles = false;
    double *tile_part = nullptr;
    int *tile_n = nullptr;
    int part_cap = 0;
};

namespace tsmi {

// The rotation constants of CPUBlock::rabi_coupling(var, dt) (src/cpukernel.cpp:581-608).
void rabi_coefs(const tsmi_pair *p, double var, double *cc, double *cs_r, double *cs_i);
inline bool rabi_on(const tsmi_pair *p) { return p->omega_r != 0.0 || p->omega_i != 0.0; }
inline double *norms(tsmi_pair *p) { return p->dv + 4 + 2 * p->norm_slot; }
// The periodic exchange of both components' current tiles.
int exchange_both(tsmi_pair *p);

// Tile passes (tsmi_pair_tile.hip): whether the lattice takes them (set at
// creation), whether a call of n steps does (the E tables must have the phase form
// besides), the most workgroups of an imaginary-time pass, and an evolve of n steps as them (no
// renormalisation pending before; every cell renormalised after).
bool pair_tiles_fit(const tsmi_pair *p, int tile_rows, int sweeps);
bool pair_tiles_run(const tsmi_pair *p, int n);
int pair_tile_blocks(const tsmi_pair *p);
int pair_tile_evolve(tsmi_pair *p, int n, bool rabi);

}  // namespace tsmi
