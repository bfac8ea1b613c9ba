// How a run's time steps are launched: which lattices take several steps per
// launch, and how those launches deal the lattice to waves and work-groups.
// Host only and without the HIP runtime.  Internal.
#pragma once

#include <cstdint>
#include <vector>

namespace lbm {

enum Storage : int32_t { kF64 = 0, kF32 = 1, kF16 = 2 };

// What the rules look at.
struct LatticeShape {
    int32_t storage;
    bool psbb;                  // partially saturated bounce-back
    int64_t nr, nc;
    bool wet_top, wet_bottom;   // row 0 / row NR-1 holds a wet node
    int32_t cus;                // compute units of the device
    int64_t wet, wet_segments;  // wet nodes, and 64-row segments of columns that hold one
};

// Lattices below these node counts take tiles, FP64 and FP32 lattices from
// there on marching waves; ensembles take marching waves from kMarchMinNodes
// nodes in all.
constexpr int64_t kTileMaxNodes = 300000, kTileMaxNodesF16 = (int64_t)3 << 19;
constexpr int64_t kMarchMinNodes = (int64_t)1 << 17, kBatchFusedNodes = (int64_t)1 << 20;
// Lattices whose waves keep the SIMDs full.
constexpr int64_t kMarchLargeNodes = (int64_t)1 << 22;

// How a launch of the marching kernel deals its waves (march_kernel).
struct MarchPlan {
    int32_t stripes;         // stripes of rows
    int32_t top, bottom;     // of these, the first / last ones, whose windows hold wet nodes of row 0 / NR-1
    int32_t cols;            // columns per wave
    int32_t edge_cols;       // columns per wave of the edge stripes
    int32_t edge_chunks;     // waves per edge stripe
    int32_t edge_row_waves;  // waves of the edge stripes
    int32_t edge_waves;      // and with the first and last columns of the others, rounded up to whole work-groups
};
// Waves of a launch of K steps of a lattice of nc columns.
inline int64_t march_launch_waves(const MarchPlan &m, int64_t nc, int32_t K)
{
    const int64_t inner = m.stripes - m.top - m.bottom;
    return m.edge_waves + (inner > 0 ? inner * ((nc - 2 * (K + 1) + m.cols - 1) / m.cols) : 0);
}

// Steps per launch of the marching kernel for this lattice (0: not for it),
// and the deal of a launch of K of them.
int32_t march_steps(const LatticeShape &a);
MarchPlan march_plan(const LatticeShape &a, int32_t K);
// Whether such launches are faster than the one-step kernels, by shape and
// wet nodes.
bool march_pays(const LatticeShape &a);

// Waves of an ensemble's marching launch of K steps, the columns of the
// windows without perimeter nodes in chunks of `cols`, or in chunks chosen
// here: per wave, 4 int32 -- sample, first row of the window, columns
// [j0, j1) (sign bit of j1: perimeter window).
void march_table(const LatticeShape *a, int64_t samples, int32_t K, std::vector<int32_t> &table);
void march_table(const LatticeShape *a, int64_t samples, int32_t K, int32_t cols, std::vector<int32_t> &table);
// Whether an ensemble's launches of that table are faster than its one-step
// kernels, by the samples' wet nodes.
bool ensemble_pays(const LatticeShape *a, int64_t samples, int32_t K, const std::vector<int32_t> &table);

// Region of a tile, and the steps per launch it holds (halo 0: no tiles for
// this lattice).
struct TileShape {
    int32_t rows, cols, halo;
};
TileShape tile_shape(const LatticeShape &a);
int64_t tiles_of(const LatticeShape &a, TileShape t);
// Whether launches of many steps in tiles are faster than the one-step
// kernels, and the fewest steps for which one launch is; waiting: with new
// prescribed values that the one-step kernels would wait for a copy of.
bool tiles_pay(const LatticeShape &a, TileShape t);
int32_t tile_min_steps(const LatticeShape &a, TileShape t, bool waiting);

}  // namespace lbm
