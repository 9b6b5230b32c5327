// tile_plan.hpp -- what a tile pass (tile_kernel.hpp) of one lattice or of many
// needs from the host: its tile shape, its parameters, its launch.
#pragma once
#include <hip/hip_runtime.h>

#include <utility>
#include <vector>

#include "tile_kernel.hpp"

namespace tsmi {

// Rows per wave and waves per workgroup; us: modelled time per step.
struct TilePlan {
    int r = 0, nw = 0;
    double us = 1e30;
};

// The shape of a pass of `steps` steps over lattices of these tile extents
// (W, H); r = 0 when no tile fits the apron of so many steps.
TilePlan tile_plan(const std::vector<std::pair<int, int>> &sizes, int esz, int steps);
// The number of steps per pass, at most `most`, with the least modelled time.
int tile_best_steps(const std::vector<std::pair<int, int>> &sizes, int esz, int most);

// A lattice's constants, as StepCoefs or the context hold them.
struct TileFactors {
    double mH, tH, mV, tV, unH, unV, c_nl_s, c_lhy_s, corr_abs;
    double by;                      // the vertical pair angle
};

// Fills everything but the planes: extents, tile counts, factors.  wrap: a doubly
// periodic lattice of nx x ny inner cells (0: closed).  drift: see tsmi_tile.hip.
template <typename T>
void tile_params(TileParams<T> &p, const TileFactors &f, const TilePlan &g, int W, int H, int pitch, int nx, int ny,
                 int steps, long double &drift);
extern template void tile_params<float>(TileParams<float> &, const TileFactors &, const TilePlan &, int, int, int, int,
                                        int, int, long double &);
extern template void tile_params<double>(TileParams<double> &, const TileFactors &, const TilePlan &, int, int, int,
                                         int, int, int, long double &);

// One launch over many lattices (device arrays of TileParams<T> and of items
// (lattice, tile)), all of shape g and scaled form `mode`.
int tile_batch_launch(int esz, bool lhy, int mode, const TilePlan &g, const void *params, const int2 *items,
                      int n_items, hipStream_t stream);

}  // namespace tsmi
