// Launch rules (lbm_plan.h).
#include "lbm_plan.h"

#include <algorithm>

namespace lbm {

namespace {

// Waves per SIMD that the columns are dealt for.  The kernels' registers allow
// as many or more: FP64 two at 5 steps (197 VGPRs) and 4 unfused (194), three
// at 2, 3 and 4 fused (138, 166, 164); FP32 three at 4 (132 fused, 148), four at 3
// (119), five at 2 (90).  The chunk lengths below were measured with these.
int64_t march_waves(int32_t storage) { return storage == kF64 ? 2 : 3; }

// Deals the columns to waves.  A wave computes cols + 2 K columns' levels
// for cols columns of results, so long chunks waste less, but the waves
// should fill the chip a whole number of times (every wave takes about the
// same time): the longest chunk of at most kMarchCols columns that does.
// Small lattices: as many chunks as fit on the chip at once, of at least
// kMarchMinCols columns.  Measured at K = 4, us a step by cols: FP64
// 4096^2 open 141.8 (40), 143.6 (56, 2.6 fills), 136.0 (78, 2 fills), 169
// (146, 1 fill); porous 8192^2 FP32 278 (32), 271 (64), 273 (128); FP64
// 512 x 2048 16.0 (8), 14.3 (12), 17.2 (16).  A fill that the edge waves
// leave less than a fifth of is no reason for a long chunk: its few waves
// would run on alone for most of the launch (FP64, first row wet, 200 x 5000:
// 27.0 with one of 40 columns, 22.7 with the next fill's 9).
constexpr int64_t kMarchCols = 80, kMarchMinCols = 6;

// Waves the device holds at once.
int64_t march_chip(const LatticeShape &a) { return (int64_t)a.cus * 4 * march_waves(a.storage); }

// Columns per wave of the stripes with perimeter windows, `columns` of them in
// all.  Edge waves are slower than the others and start first, so in a short
// launch they are short: 2 columns, of 2 + 2 K that they compute.  Once they
// fill the chip by themselves that is wasted work, and they take as many
// columns as leave seven eighths of a fill, up to 8.  us a step of lattices
// with a wet first row, one step a launch / 2 columns / this: 50 x 20000 FP64
// 39.7 / 48.7 / 35.3, FP32 28.1 / 29.8 / 21.4; 16 x 62500 FP64 94.7 / 143.6 /
// 80.9, FP32 67.1 / 84.1 / 49.8; both rows wet, 160 x 2000 FP64 18.6 / 27.2 /
// 13.1.  Lattices of 2^21 nodes and more take 8.
constexpr int64_t kEdgeLongNodes = (int64_t)1 << 21;
constexpr int32_t kEdgeMaxCols = 8;
int32_t edge_columns_per_wave(int64_t columns, int64_t chip)
{
    const int64_t waves = std::max<int64_t>(chip * 7 / 8, 1);
    return (int32_t)std::clamp<int64_t>((columns + waves - 1) / waves, 2, kEdgeMaxCols);
}

// Stripes of rows of K-step windows, and which of them hold wet nodes of
// the first or last row.
MarchPlan march_stripes(const LatticeShape &a, int32_t K)
{
    const int32_t rows = 64 - 2 * K;
    MarchPlan m{};
    m.stripes = (int32_t)((a.nr + rows - 1) / rows);
    if (a.nc < 2 * (K + 1) + 1) {  // no column is free of the first and last columns' influence
        m.top = m.stripes;
    } else {
        m.top = a.wet_top ? 1 : 0;
        if (a.wet_bottom)
            for (int32_t q = m.stripes - 1; q >= m.top && (int64_t)q * rows - K + 64 >= a.nr; --q) ++m.bottom;
    }
    return m;
}

}  // namespace

// A launch of marching waves takes at least the time one wave needs for its
// columns (30 us at K = 4 in FP64, half of it in FP32; more where the top
// or bottom row is wet): small lattices take tiles (tile_shape).  FP64 at
// K = 5 against K = 4, us a step (columns dealt for two waves per SIMD in both):
// porous 4096^2 104.4 / 113.5, TRT cavity 4096^2 141.4 / 150.3, open 3001 x 5003
// 122.0 / 125.3, 8192^2 523 / 613, 2100^2 40.1 / 40.7; slower on small lattices.
int32_t march_steps(const LatticeShape &a)
{
    const int64_t nodes = a.nr * a.nc;
    if (a.storage == kF16 || a.psbb || nodes < kTileMaxNodes) return 0;
    return a.storage == kF64 && nodes >= kMarchLargeNodes ? 5 : 4;
}

// A marching launch walks every window of the lattice, wet or not, and its
// waves at the perimeter store few of the columns that they compute.  The
// one-step kernels leave dry segments at once.  us a step, one step a launch /
// marching:
//  * Mostly dry lattices, single steps below 2^20 nodes where less than half
//    of the segments hold a wet node: FP64 600^2, fluid in one rectangle of 5 /
//    20 / 40 % 4.6 / 6.7, 5.2 / 6.9, 6.7 / 7.1, squares of fluid 3 / 10 / 30 %
//    (10 / 32 / 73 % of the segments) 5.1 / 6.7, 5.7 / 6.8, 7.4 / 7.2; 2000 x
//    200 FP32 5 % 4.1 / 5.0.  At 1100^2 5 % FP64 the two meet (9.6 / 10.0) and
//    above marching wins: the one-step kernel's dry waves cost what it saves.
//  * All windows at the perimeter because the first and the last row are wet:
//    single steps where the windows are more than the segments (57 to 64 rows,
//    or K = 5 and 109 to 128): 64 x 15625 FP64 36.7 / 42.4, FP32 24.6 / 28.3, 112
//    x 44642 FP64 181.9 / 193.2; but 80 x 12500 FP64 44.2 / 41.6.
//  * Fewer than 2 K + 5 columns, so that no window, or hardly one, is free of
//    the first and last column: single steps with many solid nodes.  440000 x
//    10 FP32, 30 % solid 31.7 / 37.1, open 61.9 / 52.1; 400000 x 11 30 % solid
//    31.9 / 35.8.
bool march_pays(const LatticeShape &a)
{
    const int64_t nodes = a.nr * a.nc, rows = (a.nr + 63) / 64;
    if (nodes < ((int64_t)1 << 20) && 2 * a.wet_segments < rows * a.nc) return false;
    const int32_t K = march_steps(a);
    if (a.nc < 2 * K + 5) return 4 * a.wet >= 3 * nodes;
    const MarchPlan m = march_stripes(a, K);
    return m.top + m.bottom < m.stripes || m.stripes <= rows;
}

MarchPlan march_plan(const LatticeShape &a, int32_t K)
{
    MarchPlan m = march_stripes(a, K);
    const int64_t inner = m.stripes - m.top - m.bottom, free_cols = a.nc - 2 * (K + 1), chip = march_chip(a);
    m.edge_cols = a.nr * a.nc < kEdgeLongNodes ? edge_columns_per_wave((m.top + m.bottom) * a.nc, chip) : kEdgeMaxCols;
    m.edge_chunks = (int32_t)((a.nc + m.edge_cols - 1) / m.edge_cols);
    m.edge_row_waves = (m.top + m.bottom) * m.edge_chunks;
    m.edge_waves = (int32_t)((m.edge_row_waves + 2 * inner + 3) & ~(int64_t)3);
    m.cols = kMarchMinCols;
    if (inner > 0) {
        for (int64_t fills = 1;; ++fills) {
            const int64_t slots = fills * chip - m.edge_waves, chunks = slots / inner;
            if (chunks < 1) continue;
            const int64_t cols = (free_cols + chunks - 1) / chunks;
            if (cols > kMarchCols || (cols > kMarchCols / 2 && slots < chip / 5)) continue;
            m.cols = (int32_t)std::max(cols, kMarchMinCols);
            break;
        }
    }
    return m;
}

namespace {

// Columns that a marching wave computes, weighted by how long one takes: the
// perimeter's closures wait for loads of their own at every level.
double march_work(const int32_t *wave, int32_t K)
{
    const bool edge = wave[3] < 0;
    return ((wave[3] & 0x7fffffff) - wave[2] + 2 * K) * (edge ? 1.75 : 1.0);
}

}  // namespace

// Chunks of columns: the longest of these whose waves keep three quarters of
// the chip busy for as long as one of them takes (each wave recomputes the 2 K
// columns at its ends), and the shortest for ensembles that never do.  us a
// step by columns (64 / 32 / 16 / 8): 32 lattices of up to 1024^2 FP32 48.6 /
// 47.6 / 50.9 / 57.6; 20 of up to 512^2 24.1 / 18.4 / 14.8 / 15.4; 60 of up to
// 256^2 FP64 35.0 / 26.6 / 27.2 / 26.2.  It is the work that counts and not the
// number of waves: perimeter waves are many and short.  Counted alike they
// made the others long, single steps / counted alike / this: 20 lattices of
// 129^2 with a wet first row FP64 18.1 / 23.9 / 13.3, and last row 20.9 / 47.1
// / 16.0; 60 of 64^2 17.2 / 41.6 / 14.3; 16 porous ones of 512^2 92.1 / 47.4 /
// 35.5.
void march_table(const LatticeShape *a, int64_t samples, int32_t K, std::vector<int32_t> &table)
{
    for (int32_t cols : {64, 32, 16, 12, 8, 6}) {
        march_table(a, samples, K, cols, table);
        double work = 0.0;
        for (size_t k = 0; k < table.size(); k += 4) work += march_work(&table[k], K);
        if (samples == 0 || work >= 0.75 * (double)march_chip(a[0]) * (cols + 2 * K)) return;
    }
}

void march_table(const LatticeShape *a, int64_t samples, int32_t K, int32_t cols, std::vector<int32_t> &table)
{
    const int32_t rows = 64 - 2 * K;
    int64_t edge = 0;
    for (int64_t s = 0; s < samples; ++s) {
        const MarchPlan m = march_stripes(a[s], K);
        edge += (m.top + m.bottom) * a[s].nc;
    }
    const int32_t edge_cols = samples ? edge_columns_per_wave(edge, march_chip(a[0])) : 0;
    table.clear();
    auto add = [&](int64_t s, int32_t stripe, int32_t j0, int32_t j1, bool edge) {
        table.insert(table.end(), {(int32_t)s, stripe * rows - K, j0, edge ? (int32_t)(j1 | (1u << 31)) : j1});
    };
    for (int64_t s = 0; s < samples; ++s) {
        const MarchPlan m = march_stripes(a[s], K);
        const int32_t nc = (int32_t)a[s].nc, ec = a[s].nr * nc < kEdgeLongNodes ? edge_cols : kEdgeMaxCols;
        for (int32_t q = 0; q < m.stripes; ++q) {
            if (q < m.top || q >= m.stripes - m.bottom) {
                for (int32_t j = 0; j < nc; j += ec) add(s, q, j, std::min(j + ec, nc), true);
            } else {
                add(s, q, 0, K + 1, true);
                add(s, q, nc - (K + 1), nc, true);
            }
        }
    }
    for (int64_t s = 0; s < samples; ++s) {
        const MarchPlan m = march_stripes(a[s], K);
        const int32_t end = (int32_t)a[s].nc - (K + 1);
        for (int32_t j = K + 1; j < end; j += cols)
            for (int32_t q = m.top; q < m.stripes - m.bottom; ++q) add(s, q, j, std::min(j + cols, end), false);
    }
}

// A marching launch walks every window, wet or not; an ensemble's one-step
// kernels have a table of the segments that hold a wet node and take only
// those.  The launch takes as long as the columns that fall to one slot of the
// chip (march_waves a SIMD, edge columns a quarter more); four single steps
// cost a fixed time, one per segment and one per wet node, in the same unit of
// about 2.5 us.  Fitted to 90 ensembles per format: 131072 to 12 million nodes,
// lattices of 16 x 16 to 1024^2, 2 to 1000 of them, channels, cavities, porous
// and mostly dry media, wet first and last rows.  Single steps were up to 6 times
// faster on 27 of them, and marching up to 2.8 on the others; the rule errs by up
// to 17 %, where the two are close.  us a step, one step a launch /
// marching: 16 lattices of 512^2, 5 / 20 / 50 % of each wet, FP64 7.8 / 33.5,
// 24.5 / 34.1, 50.7 / 34.4; FP32 5.9 / 22.4, 13.6 / 23.2, 26.8 / 23.3.
bool ensemble_pays(const LatticeShape *a, int64_t samples, int32_t K, const std::vector<int32_t> &table)
{
    if (table.empty()) return false;
    double segments = 0.0, wet = 0.0, columns = 0.0;
    for (int64_t s = 0; s < samples; ++s) {
        segments += (double)a[s].wet_segments;
        wet += (double)a[s].wet;
    }
    for (size_t k = 0; k < table.size(); k += 4)
        columns += ((table[k + 3] & 0x7fffffff) - table[k + 2] + 2 * K) * (table[k + 3] < 0 ? 1.25 : 1.0);
    const double slots = std::min((double)table.size() / 4, (double)march_chip(a[0]));
    const double per_cu = 256.0 / a[0].cus;
    const double single = a[0].storage == kF64 ? 10.0 + (0.8e-3 * segments + 8e-6 * wet) * per_cu
                                               : 11.0 + (0.3e-3 * segments + 12e-6 * wet) * per_cu;
    return columns / slots < single;
}

int64_t tiles_of(const LatticeShape &a, TileShape t)
{
    const int64_t r = t.rows - 2 * t.halo, c = t.cols - 2 * t.halo;
    return ((a.nr + r - 1) / r) * ((a.nc + c - 1) / c);
}

// As many steps a launch as leave one tile per CU: more steps share a
// launch's fixed cost, and a second tile on a CU costs what it saves.  Smaller
// regions step faster (waves per SIMD: 24 x 24 two to three, 32 x 24 three, 32
// x 32 four) but hold fewer steps: the shapes are tried from the fastest per
// step on.  Beyond one tile
// per CU 8- and 4-byte elements part: two 32 x 24 tiles of FP32 or FP16 run
// on a CU side by side.  Measured, us a step (steps a launch): 129^2 FP64
// 32 x 24 1.85 (9), 32 x 20 1.84 (7), 32 x 16 1.95 (6), 24 x 24 2.05 (7), 32 x
// 32 2.15 (10), FP32 1.45, 1.53, -, 1.60, 1.65; 65^2 FP64 24 x 24 1.75 (8), 32
// x 24 1.86 (9); 160^2 24 x 24 1.92 (7), 32 x 24 2.01 (8); 200^2 FP64 32 x 24 2.27 (7), 32
// x 32 2.50 (7); 300^2 FP64 32 x 32 3.26 (6), 32 x 24 3.71 (4); 251 x 1003 FP32
// 32 x 24 4.63 (5), 4.88 (6), 32 x 32 5.14 (4), FP64 7.97 (4), 7.23 (4).  From
// about 300000 nodes the marching waves are as fast (FP64 / FP32: 1400 x 200
// march 7.8 / 5.6, porous 500 x 700 7.6 / 5.7); FP16, which has none, stays
// until single steps are: 700^2 6.7 against 12.4, 1000^2 11.0 against 16.3,
// 1500^2 about 24 either way.
TileShape tile_shape(const LatticeShape &a)
{
    const int64_t nodes = a.nr * a.nc;
    if (nodes >= (a.storage == kF16 ? kTileMaxNodesF16 : kTileMaxNodes)) return {0, 0, 0};
    constexpr TileShape kOnePerCu[] = {{24, 24, 8}, {32, 24, 9}, {24, 24, 7}, {32, 24, 8}, {32, 24, 7}, {32, 32, 9},
                                       {32, 32, 8}, {32, 32, 7}, {32, 32, 6}, {32, 32, 5}, {32, 32, 4}};
    for (const TileShape &t : kOnePerCu)
        if ((t.halo > 4 || a.storage == kF64) && tiles_of(a, t) <= a.cus) return t;
    if (a.storage != kF64) {
        if (tiles_of(a, {32, 24, 6}) <= 3 * (int64_t)a.cus) return {32, 24, 6};
        return {32, 24, a.storage == kF16 && tiles_of(a, {32, 24, 5}) > 4 * (int64_t)a.cus ? 4 : 5};
    }
    for (int32_t halo = 7; halo > 4; --halo)
        if (tiles_of(a, {32, 32, halo}) <= 2 * (int64_t)a.cus) return {32, 32, halo};
    return {32, 32, 4};
}

// Lattices of a few columns leave most of each tile outside.  us a step, one
// step a launch / tiles: 3 columns, 40000 rows FP64 9.5 / 12.0, 96666 rows 14.1
// / 26.8, FP32 10.0 / 14.1, FP16 10.4 / 15.4; 5 columns, 58000 rows FP64 14.4 /
// 17.7; but 5 columns, 24000 rows FP32 8.4 / 4.9.
bool tiles_pay(const LatticeShape &a, TileShape t)
{
    return a.nc > 5 || tiles_of(a, t) <= (a.storage == kF64 ? 6 : 10) * (int64_t)a.cus;
}

namespace {

// us of one step by the one-step kernels, and of a tile launch of one, of
// lattices below kTileMaxNodes (FP16: kTileMaxNodesF16), as fitted to 230 of
// them per format (calls of one step; to 5 % and to 15 to 20 %).
struct StepCost {
    double base, segments, wet_segments, perimeter, wet;  // the last four per million
    double tile_base, tile;                               // per round of one tile per CU
};
constexpr StepCost kStepCost[3] = {{8.4, 0, 590, 730, 9.4, 2.9, 5.25},
                                   {7.0, 430, 0, 450, 5.3, 4.0, 2.47},
                                   {7.6, 580, 0, 650, 0, 3.9, 2.33}};

double one_step_us(const LatticeShape &a)
{
    const StepCost &c = kStepCost[a.storage];
    const int64_t rows = (a.nr + 63) / 64;
    const int64_t perimeter = (a.wet_top ? a.nc : 0) + (a.wet_bottom && rows > 1 ? a.nc : 0) + 2 * rows;
    return c.base + 1e-6 * (c.segments * (double)(rows * a.nc) + c.wet_segments * (double)a.wet_segments +
                            c.perimeter * (double)perimeter + c.wet * (double)a.wet);
}

double tile_us(const LatticeShape &a, int64_t tiles)
{
    const StepCost &c = kStepCost[a.storage];
    return c.tile_base + c.tile * std::max(1.0, (double)tiles / a.cus);
}

}  // namespace

// A launch in tiles loads and stores its halo whatever its steps, so one of a
// single step, or two, is slower than one-step launches except on the smallest
// lattices, and on shallow ones, whose perimeter segments are slow in one-step
// launches.  us a step by calls of one step, one-step kernels / tiles: FP64 129^2
// 8.5 / 7.4, 200^2 8.8 / 9.4, 545^2 15.2 / 20.7; FP32 250^2 7.9 / 8.1, 545^2 10.7
// / 14.3; FP16 320^2 9.2 / 9.1, 1240^2 19.6 / 37.4; first row wet, 3 x 20000 FP64
// 34.9 / 25.1; FP64 with partially saturated obstacles (one kernel a step) 60^2
// 4.7 / 6.3, 545^2 11.0 / 19.9.  Of two: FP16 1100^2 the same, 1240^2 19.7 / 21.8;
// 50000 x 4 FP64 12.8 / 18.2; partially saturated 200^2 5.5 / 5.7, 400^2 8.5 / 10.0.
// Where new values wait, a one-step launch takes their copy, of about 10 us, with
// it: one step with new values FP16 500^2 32.7 / 14.5, 600^2 31.1 / 14.2 (they
// wait up to nr + nc = 1365).
int32_t tile_min_steps(const LatticeShape &a, TileShape t, bool waiting)
{
    if (waiting) return 1;
    const int64_t nodes = a.nr * a.nc, tiles = tiles_of(a, t), cus = a.cus;
    if (a.psbb) return tiles <= cus ? 2 : 3;
    const int64_t small = a.storage == kF64 ? 32768 : a.storage == kF32 ? 65000 : 110000;
    const double margin = a.storage == kF64 ? 0.78 : 0.9, single = one_step_us(a), tile = tile_us(a, tiles);
    if (nodes < small && tiles <= (a.storage == kF64 ? 1 : 2) * cus) return 1;
    if (tiles > cus && tile < margin * single) return 1;
    return tiles <= (a.nc < 8 ? 5 : 14) * cus || 1.3 * tile < margin * 2.0 * single ? 2 : 3;
}

}  // namespace lbm
