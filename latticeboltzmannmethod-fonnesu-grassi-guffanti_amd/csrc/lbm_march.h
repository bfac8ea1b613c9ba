// Marching waves: several time steps of a lattice per launch.
// Included by lbm_kernels.hip inside its anonymous namespace.
//
// A step reads and writes every population once, and a launch of one step
// is bound by that traffic (72 GB/s per GLUPS in FP32).  A marching wave
// takes K steps in registers instead, so a launch reads and writes the
// state once for K steps.  It holds a window of 64 rows and walks along the
// columns.  Per column it loads the nine stored populations of its rows
// (level 0), and each level q = 1 .. K streams and collides the column
// that level q - 1 has completed the neighbours of: level q runs one column
// behind level q - 1.  Sources one row up or down are the neighbouring
// lanes (one DPP move), sources in the neighbouring columns are what the
// level kept of the column before (Level) or is fed now: no LDS and no
// barrier, and every population is loaded once instead of gathered.  The
// outermost lanes lack their neighbours, so a level loses one valid row at
// each end and a wave stores 64 - 2 K rows; at the ends of its columns it
// recomputes K columns of the neighbouring waves.
//
// The arithmetic is that of the one-step kernels, node for node, so the
// results are the same bits.  Frozen slots, Zou-He nodes and prescribed
// velocities are taken at every level by the waves whose windows hold
// perimeter nodes (EDGE); the prescribed values are those of the current
// step throughout, so the launch is for steps without new values.
//
// What bounds it: in FP32 the VALU (busy throughout on porous media, 0.85 on
// unobstructed ones, which load at 4.5 TB/s meanwhile; 122 instructions per
// level and lane, of which the collision takes 110), in FP64 the VALU at 0.8
// and latency.  FP64 at K = 5 takes 197 registers, so two waves per SIMD; at
// K = 4 the fused moves take 164 and three fit, but the columns are dealt for
// two.  FP32 at K = 4 takes 132 and three waves fit; its copy for planes keeps
// 68 bytes a lane in scratch memory besides.  us a step, before (one step a
// launch) -> K = 4 (FP32), 5 (FP64): porous 8192^2 FP32 549 (tuned; 602
// untuned) -> 252; open 4096^2 FP64 419 -> 121; TRT cavity 4096^2 FP32 194 ->
// 77, FP64 416 -> 157; porous 4096^2 FP64 303 -> 112.  K = 2 / 3 / 4 / 5 on the
// porous 4096^2 (without FUSED): FP64 211 / 146 / 119 / 114, FP32 121 / 78 / 71
// / 74.  In FP64 a launch grows from 420 us at K = 2 to 475 at K = 4, its
// traffic alike, and to 570 at K = 5: from there on the levels cost what the
// traffic saves, and the lanes and columns lost to the window's ends more.
// FP16 keeps one step a launch: its rounding takes another 50 instructions
// per node, and it was at the VALU limit with one step; marching FP16 has not
// been built.

// One column's 64-row window of a marching wave (rows i0 .. i0 + 63), all
// wave-uniform: bit l of mid / up / dn is the wet bit of row i0 + l, of the
// row above and of the row below; base is the compact index of the first
// wet row of the column at or below row i0.
struct Win {
    uint64_t mid, up, dn;
    int32_t base;
};

// The words a window is formed from: words w, w + 1, w + 2 of the column,
// w holding row i0 - 1 (the guard word above the column when i0 <= 0; its
// segment base is the column's first compact index).
struct WinWords {
    uint64_t a, b, c;
    int32_t base;
};

__device__ __forceinline__ WinWords load_words(const Geometry &g, int j, int32_t i0)
{
    const uint32_t k = (uint32_t)(j + 1) * (uint32_t)g.wl + (uint32_t)(((i0 - 1) >> 6) + 1);
    const LBM_CONST uint64_t *col = (const LBM_CONST uint64_t *)g.wet + k;
    WinWords w;
    w.a = col[0];
    w.b = col[1];
    w.c = col[2];
    w.base = ((const LBM_CONST int32_t *)g.sb)[k];
    return w;
}

__device__ __forceinline__ Win window(const WinWords &w, int32_t i0)
{
    const uint32_t b = (uint32_t)(i0 - 1) & 63u;
    Win x;
    x.up = (w.a >> b) | ((w.b << 1) << (63u - b));
    const uint64_t hi = (w.b >> b) | ((w.c << 1) << (63u - b));  // rows i0 + 63 ..
    x.mid = (x.up >> 1) | (hi << 63);
    x.dn = (x.up >> 2) | (hi << 62);
    x.base = w.base + (int32_t)__builtin_popcountll(w.a & ((2ull << b) - 1ull));
    return x;
}

// The value of the lane one row below (+1) / above (-1); lanes past the
// wave's ends read 0 (their results are not used).
template <int CTRL>
__device__ __forceinline__ uint32_t lane_move(uint32_t v)
{
    return (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, CTRL, 0xf, 0xf, true);
}

template <int CTRL, typename T>
__device__ __forceinline__ T lane_shift(T v)
{
    if constexpr (sizeof(T) == 8) {
        uint2 u = __builtin_bit_cast(uint2, v);
        u.x = lane_move<CTRL>(u.x);
        u.y = lane_move<CTRL>(u.y);
        return __builtin_bit_cast(T, u);
    } else {
        return __builtin_bit_cast(T, lane_move<CTRL>(__builtin_bit_cast(uint32_t, v)));
    }
}

// A move from the neighbouring lane and the choice against y in one
// instruction: lanes of m take the neighbour's x (the lane below's or
// above's), the others y.  v_cndmask has a DPP form only with its condition
// in VCC and picks its moved operand where the bit is clear, which the
// compiler does not form from a mask in other scalar registers; keep: the
// complement of m.  s_mov leaves SCC alone.  A DPP read must stay two wait
// states behind the write of its register (s_mov, s_nop).
#define LBM_BELOW "wave_shl:1 row_mask:0xf bank_mask:0xf bound_ctrl:0"
#define LBM_ABOVE "wave_shr:1 row_mask:0xf bank_mask:0xf bound_ctrl:0"
#define LBM_MOVED(DIR)                                                                                         \
    asm("s_mov_b64 vcc, %6\n\ts_nop 0\n\tv_cndmask_b32_dpp %0, %2, %4, vcc " DIR                              \
        "\n\tv_cndmask_b32_dpp %1, %3, %5, vcc " DIR                                                            \
        : "=&v"(r0), "=&v"(r1)                                                                                 \
        : "v"(x0), "v"(x1), "v"(y0), "v"(y1), "s"(keep)                                                        \
        : "vcc")

template <bool BELOW>
__device__ __forceinline__ void moved2(uint64_t keep, uint32_t x0, uint32_t y0, uint32_t x1, uint32_t y1, uint32_t &r0,
                                       uint32_t &r1)
{
    if constexpr (BELOW) LBM_MOVED(LBM_BELOW);
    else LBM_MOVED(LBM_ABOVE);
}

template <bool BELOW>
__device__ __forceinline__ uint32_t moved1(uint64_t keep, uint32_t x, uint32_t y)
{
    uint32_t r;
    if constexpr (BELOW)
        asm("s_mov_b64 vcc, %3\n\ts_nop 0\n\tv_cndmask_b32_dpp %0, %1, %2, vcc " LBM_BELOW
            : "=v"(r)
            : "v"(x), "v"(y), "s"(keep)
            : "vcc");
    else
        asm("s_mov_b64 vcc, %3\n\ts_nop 0\n\tv_cndmask_b32_dpp %0, %1, %2, vcc " LBM_ABOVE
            : "=v"(r)
            : "v"(x), "v"(y), "s"(keep)
            : "vcc");
    return r;
}

// FUSED: the form above; otherwise a move and a choice.
template <bool BELOW, bool FUSED, typename T>
__device__ __forceinline__ T moved(uint64_t m, T x, T y)
{
    if constexpr (!FUSED) {
        const T z = lane_shift<BELOW ? 0x130 : 0x138>(x);  // wave_shl:1 (lane l + 1), wave_shr:1 (lane l - 1)
        return __builtin_amdgcn_inverse_ballot_w64(m) ? z : y;
    } else if constexpr (sizeof(T) == 8) {
        const uint2 a = __builtin_bit_cast(uint2, x), b = __builtin_bit_cast(uint2, y);
        uint2 r;
        moved2<BELOW>(~m, a.x, b.x, a.y, b.y, r.x, r.y);
        return __builtin_bit_cast(T, r);
    } else {
        return __builtin_bit_cast(T, moved1<BELOW>(~m, __builtin_bit_cast(uint32_t, x), __builtin_bit_cast(uint32_t, y)));
    }
}

// Two values under one mask (FP32: one asm for both).
template <bool BELOW, bool FUSED, typename T>
__device__ __forceinline__ void moved_pair(uint64_t m, T x0, T y0, T x1, T y1, T &r0, T &r1)
{
    if constexpr (FUSED && sizeof(T) == 4) {
        uint32_t u0, u1;
        moved2<BELOW>(~m, __builtin_bit_cast(uint32_t, x0), __builtin_bit_cast(uint32_t, y0),
                      __builtin_bit_cast(uint32_t, x1), __builtin_bit_cast(uint32_t, y1), u0, u1);
        r0 = __builtin_bit_cast(T, u0);
        r1 = __builtin_bit_cast(T, u1);
    } else {
        r0 = moved<BELOW, FUSED>(m, x0, y0);
        r1 = moved<BELOW, FUSED>(m, x1, y1);
    }
}

// What one level of a marching wave keeps of the last column it was fed:
// the six pre-collision populations that are complete, and the three
// post-collision populations that leave to the next column (which are also
// the bounce-back values of the three slots still open).
template <typename T>
struct Level {
    T p0, p1, p2, p4, p5, p8;
    T e1, e5, e8;
};

// Streams column c's post-collision populations o into a level that holds
// column c - 1: p receives the complete pre-collision populations of column
// c - 1.  wc, wp: the windows of columns c and c - 1.
template <bool FUSED, typename T>
__device__ __forceinline__ void feed(Level<T> &s, const T *o, const Win &wc, const Win &wp, T *p)
{
    auto sel = [](uint64_t m, T x, T y) { return __builtin_amdgcn_inverse_ballot_w64(m) ? x : y; };
    p[0] = s.p0;
    p[1] = s.p1;
    p[2] = s.p2;
    p[4] = s.p4;
    p[5] = s.p5;
    p[8] = s.p8;
    p[3] = sel(wc.mid, o[3], s.e1);
    s.p0 = o[0];
    s.p1 = sel(wp.mid, s.e1, o[3]);
    s.p5 = moved<true, FUSED>(wp.dn, s.e5, o[7]);
    s.p8 = moved<false, FUSED>(wp.up, s.e8, o[6]);
    moved_pair<true, FUSED>(wc.dn, o[6], s.e8, o[2], o[4], p[6], s.p2);
    moved_pair<false, FUSED>(wc.up, o[7], s.e5, o[4], o[2], p[7], s.p4);
    s.e1 = o[1];
    s.e5 = o[5];
    s.e8 = o[8];
}

// Frozen slots and Zou-He closure of a perimeter node whose interior slots
// are in p; returns the node's policy.  The prescribed values do not change
// within the launch.  All loads issue together: the levels of an edge wave
// follow each other, so their round trips to memory add up.
template <typename T>
__device__ __forceinline__ int close_edge(const StepArgs &a, int i, int j, T *p, Prescribed &v)
{
    const int64_t e = edge_slot(i, j, a.g.nr, a.g.nc);
    T frozen[9];
#pragma unroll
    for (int d = 1; d < 9; ++d) frozen[d] = ((const LBM_GLOBAL T *)a.frozen)[d * a.g.E + e];
    const int kind = ((const LBM_GLOBAL uint8_t *)a.g.edge_kind)[e];
    const LBM_GLOBAL double *bc = (const LBM_GLOBAL double *)a.bc_cur + e;
    v.ux = bc[0];
    v.uy = bc[a.g.E];
    const double rho = bc[2 * a.g.E];
#pragma unroll
    for (int d = 1; d < 9; ++d) {
        const int si = i - kOffI[d], sj = j - kOffJ[d];
        if (si < 0 || si >= a.g.nr || sj < 0 || sj >= a.g.nc) p[d] = frozen[d];
    }
    if (kind == kEdgePlain) return -1;
    const int policy = kind == kEdgeInlet ? a.inlet_policy : a.outlet_policy;
    const int bt = edge_btype(i, j, a.g.nr, a.g.nc);
    if constexpr (sizeof(T) == 8) {
        if (policy == kVelocity) zouhe_velocity64(bt, p, v.ux, v.uy);
        else if (policy == kPressure) zouhe_pressure64(bt, p, rho);
    } else {
        if (policy == kVelocity) zouhe_velocity32(bt, p, (float)v.ux, (float)v.uy);
        else if (policy == kPressure) zouhe_pressure32(bt, p, (float)rho, (float)(rho - 1.0));
    }
    return policy;
}

// One 64-row window's elements in memory: a scalar base at the 64-node block
// of the window's first wet row, and the byte offset of this lane's node from
// it (the window's nodes fall in two blocks at most).  The directions lie 64
// elements apart (blocked) or, PLANES, a plane apart: a scalar base each,
// formed by adding.  Lattices of 4 GiB and more a buffer lie in planes.  us a
// step, one step a launch (tuned) -> this: open 8192^2 FP64 1583 -> 484 (420
// would be blocked FP64's time per node); 2100^2 FP64 36.2 against 35.5
// blocked, FP32 23.7 against 22.6.
template <typename T, bool PLANES>
__device__ __forceinline__ int64_t win_base(const Win &w)
{
    return (int64_t)(w.base >> 6) * (int64_t)((PLANES ? 1 : 9) * 64 * sizeof(T));
}

template <typename T, bool PLANES>
__device__ __forceinline__ uint32_t win_offset(const Win &w)
{
    const uint32_t r = __builtin_amdgcn_mbcnt_hi((uint32_t)(w.mid >> 32),
                                                 __builtin_amdgcn_mbcnt_lo((uint32_t)w.mid, (uint32_t)w.base & 63u));
    return (PLANES ? r : r + 8u * (r & 64u)) * (uint32_t)sizeof(T);
}

// The 9 stored populations of the window's nodes.
template <typename T, bool PLANES>
__device__ __forceinline__ void win_load(const StepArgs &a, const Win &w, T *raw)
{
    const LBM_GLOBAL char *base = (const LBM_GLOBAL char *)a.fin + win_base<T, PLANES>(w);
    const uint32_t off = win_offset<T, PLANES>(w);
    const int64_t apart = PLANES ? a.g.plane * (int64_t)sizeof(T) : (int64_t)(64 * sizeof(T));
#pragma unroll
    for (int d = 0; d < 9; ++d, base += apart) raw[d] = *(const LBM_GLOBAL T *)(base + off);
}

// Stores o for the lanes of m, without a branch: the other lanes' offsets
// lie outside the buffer descriptor's range, so their writes are dropped.
template <typename T, bool PLANES>
__device__ __forceinline__ void win_store(const StepArgs &a, const Win &w, uint64_t m, const T *o)
{
    char *base = (char *)a.fout + win_base<T, PLANES>(w);
    const uint32_t off = __builtin_amdgcn_inverse_ballot_w64(m) ? win_offset<T, PLANES>(w) : 0x40000000u;
    auto rsrc = __builtin_amdgcn_make_buffer_rsrc(base, 0, (PLANES ? 2 : 2 * 9) * 64 * (int)sizeof(T), 0x00027000);
#pragma unroll
    for (int d = 0; d < 9; ++d) {
        if constexpr (PLANES) {
            if (d > 0) {
                base += a.g.plane * (int64_t)sizeof(T);
                rsrc = __builtin_amdgcn_make_buffer_rsrc(base, 0, 2 * 64 * (int)sizeof(T), 0x00027000);
            }
        }
        const int at = PLANES ? 0 : d * 64 * (int)sizeof(T);
        if constexpr (sizeof(T) == 8) {
            typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
            __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(u32x2, o[d]), rsrc, (int)off + (at & 4095),
                                                  at & 4096, 0);
        } else {
            __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(uint32_t, o[d]), rsrc, (int)off + at, 0, 0);
        }
    }
}

// Waits for the nine loaded values here (empty asm naming them).
template <typename T>
__device__ __forceinline__ void arrived(T *raw)
{
    asm volatile("" : "+v"(raw[0]), "+v"(raw[1]), "+v"(raw[2]), "+v"(raw[3]), "+v"(raw[4]), "+v"(raw[5]),
                 "+v"(raw[6]), "+v"(raw[7]), "+v"(raw[8]));
}

// Moments, collision of one level of a window; EDGE: with the perimeter's
// frozen slots and closures.
template <typename T, bool EDGE>
__device__ __forceinline__ bool march_collide(const StepArgs &a, T *p, const Win &w, int i0, int j, int lane, T *o)
{
    int policy = -1;
    Prescribed v{};
    if constexpr (EDGE) {
        const int i = i0 + lane;
        if (__builtin_amdgcn_inverse_ballot_w64(w.mid) && (i == 0 || i == a.g.nr - 1 || j == 0 || j == a.g.nc - 1))
            policy = close_edge(a, i, j, p, v);
    }
    if constexpr (sizeof(T) == 8) return collide_f64<false>(a, p, policy, v, 0, j, o);
    else return collide_shifted<false, false>(a, p, policy, v, 0, j, o);
}

template <typename T, int K, bool FUSED, bool EDGE, bool PLANES>
__device__ __forceinline__ void march_wave(const StepArgs &a, int32_t i0, int32_t j0, int32_t j1, int lane)
{
    constexpr uint64_t kOut = ((1ull << (64 - 2 * K)) - 1ull) << K;  // lanes whose rows this wave owns
    const int32_t nc = a.g.nc;
    const int32_t first = EDGE ? max(j0 - K, 0) : j0 - K, last = j1 - 1 + K;
    Win w[K + 2];  // w[0]: column c + 1, w[q]: column c + 1 - q
#pragma unroll
    for (int q = 0; q < K + 2; ++q) w[q] = Win{0, 0, 0, 0};
    Level<T> lv[K];
#pragma unroll
    for (int q = 0; q < K; ++q) lv[q] = Level<T>{};
    T raw[9];
    w[0] = window(load_words(a.g, first, i0), i0);
    win_load<T, PLANES>(a, w[0], raw);
    WinWords nw = load_words(a.g, EDGE ? min(first + 1, nc) : first + 1, i0);
    bool bad = false;
    // one column: c enters, column c - K leaves (all levels active)
    auto column = [&](int32_t c, auto steady) {
        constexpr bool STEADY = decltype(steady)::value;
        T o[9], p[9];
#pragma unroll
        for (int q = K + 1; q > 0; --q) w[q] = w[q - 1];
        w[0] = window(nw, i0);
        nw = load_words(a.g, EDGE ? min(c + 2, nc) : c + 2, i0);
        feed<FUSED>(lv[0], raw, w[1], w[2], p);
        win_load<T, PLANES>(a, w[0], raw);
#pragma unroll
        for (int q = 1; q <= K; ++q) {
            // level q of column c - q
            const int32_t j = c - q;
            if (!STEADY && j < (EDGE ? max(j0 - K + q, 0) : j0 - K + q)) return;
            bool nan = false;
            if (!EDGE || j < nc) nan = march_collide<T, EDGE>(a, p, w[q + 1], i0, j, lane, o);
            if (q < K) {
                feed<FUSED>(lv[q], o, w[q + 1], w[q + 2 <= K + 1 ? q + 2 : K + 1], p);
            } else {
                const uint64_t m = j < j1 ? w[K + 1].mid & kOut : 0ull;
                bad |= nan && __builtin_amdgcn_inverse_ballot_w64(m);
                win_store<T, PLANES>(a, w[K + 1], m, o);
            }
        }
    };
    int32_t c = first;
#pragma unroll 1
    for (; c < j0 + K; ++c) column(c, std::false_type{});
    if (!EDGE) {
        arrived(raw);
        if constexpr (FUSED) {
#pragma unroll 1
            for (; c < last; c += 2) {
                column(c, std::true_type{});
                column(c + 1, std::true_type{});
            }
        }
#pragma unroll 1
        for (; c <= last; ++c) column(c, std::true_type{});
    } else {
#pragma unroll 1
        for (; c <= last; ++c) column(c, std::false_type{});
    }
    if (bad) atomicOr(a.flag, 1);
}

// K steps.  FUSED: for lattices that keep the SIMDs full, two columns per
// turn of the loop and the moves of feed() in fewer instructions.  Where a
// wave waits on its own chain instead, the fused moves' waits cost more than
// the instructions they save.  us a step, plain -> fused: porous 4096^2 FP64
// 116.5 -> 112.0, FP32 69.3 -> 67.5; open 3001 x 5003 FP64 111.7 -> 106.9;
// porous 8192^2 FP32 261.5 -> 253.8; an ensemble of 60 lattices of up to 256^2
// FP64 31.2 -> 28.7, of 8 of them FP32 6.6 -> 7.0.
//
// The XCDs take the waves in chunks of 8 work-groups: 32 stripes of one chunk
// of columns.  us a step with about one chunk of columns per XCD -> 8 (three
// rounds in turn, spread 0.4 %): TRT cavity 4096^2 FP32 78.4 -> 76.6; open
// 4096^2 FP32 76.7 -> 75.2; channel 1400 x 4000 FP32 26.2 -> 25.8, 512 x 2048
// FP32 7.9 -> 7.8; porous media and FP64 the same.  4, 6, 10 and 12 lie
// between.
constexpr uint32_t kMarchXcdChunk = 8;

template <typename T, int K, bool FUSED, bool PLANES>
__global__ __launch_bounds__(kBlockRows) void march_kernel(StepArgs a, MarchPlan m)
{
    constexpr int32_t kRows = 64 - 2 * K;
    const uint32_t b = xcd_remap(blockIdx.x, (uint32_t)a.nblocks, kMarchXcdChunk);
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int lane = threadIdx.x & 63;
    int32_t t = (int32_t)b * (kBlockRows / 64) + wave;
    const int32_t nc = a.g.nc;
    const int32_t inner = m.stripes - m.top - m.bottom;
    if (t < m.edge_waves) {
        int32_t stripe, j0, j1;
        if (t < m.edge_row_waves) {
            const int32_t q = t / m.edge_chunks;  // which edge stripe
            stripe = q < m.top ? q : m.stripes - m.bottom + (q - m.top);
            j0 = (t - q * m.edge_chunks) * m.edge_cols;
            j1 = min(j0 + m.edge_cols, nc);
        } else {
            t -= m.edge_row_waves;
            if (t >= 2 * inner) return;
            const bool right = t >= inner;
            stripe = m.top + (right ? t - inner : t);
            j0 = right ? nc - (K + 1) : 0;
            j1 = right ? nc : K + 1;
        }
        march_wave<T, K, FUSED, true, PLANES>(a, stripe * kRows - K, j0, j1, lane);
        return;
    }
    t -= m.edge_waves;
    const int32_t chunk = t / inner;
    const int32_t j0 = K + 1 + chunk * m.cols;
    const int32_t end = nc - (K + 1);
    if (j0 >= end) return;
    march_wave<T, K, FUSED, false, PLANES>(a, (m.top + t - chunk * inner) * kRows - K, j0, min(j0 + m.cols, end), lane);
}

