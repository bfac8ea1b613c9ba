// Tiles in LDS: several time steps of a small lattice per launch.
// Included by lbm_kernels.hip inside its anonymous namespace.
//
// A small lattice's step is bound by its launches, not by its work: two
// kernels of 3-5 us each on 129^2 nodes.  Here a work-group keeps a region
// of S x S nodes in LDS, one node per thread, and takes up to `halo` steps
// between one load and one store of the state; each step spoils one more
// ring of the region, so the work-group stores the (S - 2 halo)^2 nodes in
// the middle.  Perimeter nodes (frozen slots, Zou-He, prescribed
// velocities), new prescribed values and the macro fields are handled here
// too, so one launch does all a lattice needs.  New prescribed values are
// read from the page-locked memory they wait in, and kept in the device copy
// for the steps after (bc_new).
//
// Slots whose source lies outside the domain keep their value (the
// reference never writes them): the region's positions just outside the
// domain hold those values in LDS and are never overwritten, so the gather
// needs no case for them.
//
// What bounds it: latency.  A launch costs about 5 us and a step 1.2 us in
// FP64 (a gather from LDS, a barrier, the collision's dependent chain, a
// store, a barrier); the vector ALUs are busy for 18 % of a launch on the
// 129^2 cavity in FP64 (40 % on 251 x 1003 in FP32), the waves wait for 58 %
// (50 %) of their cycles, and bank conflicts take below 1 % of the LDS's.  us
// a step in long runs, single steps -> tiles: 129^2 cavity FP64 7.7 -> 1.85,
// FP32 7.1 -> 1.45, FP16 7.9 -> 1.7; channel 40 x 96 FP64 7.0 -> 1.7; 300^2 FP64
// 9.1 -> 3.3; 251 x 1003 FP32 9.6 -> 4.6.  Launches of one step or two are
// another matter (tile_min_steps).
//
// Same arithmetic per node as the step kernels, same bits.
// PS: partially saturated obstacles (FP64).  A node keeps the populations
// that enter it through its obstacle slots, and their weights, in registers
// (psbb_gather, psbb_update); its carried values alternate between two
// buffers like the state, since the tiles around it read the old ones.  At 32
// x 32 two of its registers spill (12 bytes a lane of scratch memory).
template <typename T, int kRows, int kCols, bool PS = false>
__global__ __launch_bounds__(kRows * kCols) void tile_kernel(StepArgs a, int32_t steps, int32_t halo, int32_t tiles_i)
{
    constexpr int kTileNodes = kRows * kCols;
    __shared__ T F[9 * kTileNodes];
    __shared__ uint8_t kind[kTileNodes];  // 0 dry, 1 wet, 2 outside the domain
    const int32_t nr = a.g.nr, nc = a.g.nc;
    const int32_t tj = (int32_t)blockIdx.x / tiles_i, ti = (int32_t)blockIdx.x - tj * tiles_i;
    const int32_t pos = threadIdx.x;
    const int32_t rj = pos / kRows, ri = pos - rj * kRows;
    const int32_t i = ti * (kRows - 2 * halo) - halo + ri, j = tj * (kCols - 2 * halo) - halo + rj;
    const bool inside = (uint32_t)i < (uint32_t)nr && (uint32_t)j < (uint32_t)nc;
    // distance from the region's border: the node is valid for that many steps
    const int32_t depth = min(min(ri, kRows - 1 - ri), min(rj, kCols - 1 - rj));

    bool wet = false;
    int32_t own = 0;
    if (inside) {
        const uint32_t k = (uint32_t)(j + 1) * (uint32_t)a.g.wl + (uint32_t)(i >> 6) + 1u;
        const uint64_t word = ((const LBM_GLOBAL uint64_t *)a.g.wet)[k];
        const int32_t base = ((const LBM_GLOBAL int32_t *)a.g.sb)[k];
        wet = (word >> (i & 63)) & 1;
        own = base + (int32_t)__builtin_popcountll(word & ((1ull << (i & 63)) - 1ull));
    }
    kind[pos] = inside ? (wet ? 1 : 0) : 2;
    T raw[9];
    if (wet) {
        const uint32_t off = slot_bytes<T>(a, (uint32_t)own);
#pragma unroll
        for (int d = 0; d < 9; ++d) raw[d] = ld((const T *)a.fin_plane[d], off);
#pragma unroll
        for (int d = 0; d < 9; ++d) F[d * kTileNodes + pos] = raw[d];
    } else if (!inside) {
#pragma unroll
        for (int d = 1; d < 9; ++d) {
            const int32_t xi = i + kOffI[d], xj = j + kOffJ[d];  // the node this slot streams into
            if ((uint32_t)xi < (uint32_t)nr && (uint32_t)xj < (uint32_t)nc)
                F[d * kTileNodes + pos] = ((const LBM_GLOBAL T *)a.frozen)[d * a.g.E + edge_slot(xi, xj, nr, nc)];
        }
    }
    uint32_t ps_mask = 0;
    double ps_val[9], ps_b[9];
    if constexpr (PS) {
        if (wet) ps_mask = ((const LBM_GLOBAL uint16_t *)a.ps_mask)[own];
#pragma unroll
        for (int d = 1; d < 9; ++d) {
            ps_val[d] = ps_b[d] = 0.0;
            if ((ps_mask >> d) & 1u) {
                const int64_t k = (int64_t)d * a.g.plane + own;
                ps_val[d] = ((const LBM_GLOBAL double *)a.ps_val)[k];
                ps_b[d] = ((const LBM_GLOBAL double *)a.ps_b)[k];
            }
        }
    }
    // perimeter node: its policy and prescribed values (prev: those of the
    // step before the launch, which close its first gather)
    int policy = -1, bt = BT_NONE;
    Prescribed v{}, prev{};
    double rho = 0.0, rho_prev = 0.0;
    const bool edge = i == 0 || i == nr - 1 || j == 0 || j == nc - 1;
    if (wet && edge) {
        const int64_t e = edge_slot(i, j, nr, nc);
        const int k = ((const LBM_GLOBAL uint8_t *)a.g.edge_kind)[e];
        const LBM_GLOBAL double *bc = (const LBM_GLOBAL double *)a.bc_cur + e;
        const LBM_GLOBAL double *bp = (const LBM_GLOBAL double *)a.bc_prev + e;
        v = {bc[0], bc[a.g.E]};
        rho = bc[2 * a.g.E];
        prev = {bp[0], bp[a.g.E]};
        rho_prev = bp[2 * a.g.E];
        if (a.bc_new && depth >= halo) {  // this tile stores the node: it also keeps its new values
            LBM_GLOBAL double *bn = (LBM_GLOBAL double *)a.bc_new + e;
            bn[0] = v.ux;
            bn[a.g.E] = v.uy;
            bn[2 * a.g.E] = rho;
        }
        if (k != kEdgePlain) policy = k == kEdgeInlet ? a.inlet_policy : a.outlet_policy;
        bt = edge_btype(i, j, nr, nc);
    }
    __syncthreads();
    // where each direction's population comes from: the source's slot, or
    // the node's own opposite one
    int32_t src[9];
    src[0] = pos;
#pragma unroll
    for (int d = 1; d < 9; ++d) {
        const int32_t si = ri - kOffI[d], sj = rj - kOffJ[d];
        const bool in = (uint32_t)si < (uint32_t)kRows && (uint32_t)sj < (uint32_t)kCols;
        const int32_t sp = in ? sj * kRows + si : pos;
        src[d] = kind[sp] != 0 ? d * kTileNodes + sp : kOpp[d] * kTileNodes + pos;
    }
#pragma unroll 1
    for (int32_t t = 1; t <= steps; ++t) {
        const bool last = t == steps;
        // nodes whose result still counts
        const bool act = wet && depth >= (last ? halo : t);
        if (act) {
#pragma unroll
            for (int d = 0; d < 9; ++d) raw[d] = F[src[d]];
        }
        if (!last) __syncthreads();
        if (act) {
            if constexpr (PS) {
#pragma unroll
                for (int d = 1; d < 9; ++d)
                    if ((ps_mask >> d) & 1u) raw[d] = ps_val[d];
            }
            if constexpr (sizeof(T) == 8) {
                if (policy == kVelocity) zouhe_velocity64(bt, raw, prev.ux, prev.uy);
                else if (policy == kPressure) zouhe_pressure64(bt, raw, rho_prev);
                T o[9], eq[9];
                if (last) collide_f64<true>(a, raw, policy, v, i, j, o, eq);
                else collide_f64<false>(a, raw, policy, v, i, j, o, eq);
                if constexpr (PS) {
#pragma unroll
                    for (int d = 1; d < 9; ++d)
                        if ((ps_mask >> d) & 1u) ps_val[d] = psbb_value(a, d, ps_b[d], raw, eq, o);
                }
#pragma unroll
                for (int d = 0; d < 9; ++d) raw[d] = o[d];
            } else {
                float g[9];
#pragma unroll
                for (int d = 0; d < 9; ++d) g[d] = (float)raw[d];
                if (policy >= 0 && policy != kNoop) {
                    // the closures work on f - w
#pragma unroll
                    for (int d = 0; d < 9; ++d) g[d] = to_g<T>(raw[d], a.inv_scale);
                    if (policy == kVelocity) zouhe_velocity32(bt, g, (float)prev.ux, (float)prev.uy);
                    else zouhe_pressure32(bt, g, (float)rho_prev, (float)(rho_prev - 1.0));
                    if constexpr (sizeof(T) == 2)
#pragma unroll
                        for (int d = 0; d < 9; ++d) g[d] *= a.scale;
                }
                float o[9];
                if (last) collide_shifted<sizeof(T) == 2, true>(a, g, policy, v, i, j, o);
                else collide_shifted<sizeof(T) == 2, false>(a, g, policy, v, i, j, o);
                encode(a, own, o, raw);
            }
            if (last) {
                store9(a, own, raw);
                if constexpr (PS) {
#pragma unroll
                    for (int d = 1; d < 9; ++d)
                        if ((ps_mask >> d) & 1u) a.ps_next[(int64_t)d * a.g.plane + own] = ps_val[d];
                }
            } else {
#pragma unroll
                for (int d = 0; d < 9; ++d) F[d * kTileNodes + pos] = raw[d];
            }
        }
        prev = v;
        rho_prev = rho;
        if (!last) __syncthreads();
    }
}
