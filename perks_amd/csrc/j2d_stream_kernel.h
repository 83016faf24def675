// j2d_stream_kernel.h -- the 2D Jacobi kernel that streams rows through
// registers (tile variant 2; instantiated per storage type in
// j2d_stream_{f64,f32,f16,bf16}.hip).
//
// A work item is a strip of 64 columns (one per lane; two per lane: 128) and
// a segment of rows of one grid; each wave runs its own items, so there is no
// LDS and no workgroup barrier.  The wave marches down the segment one row per
// iteration: level 0 is the field row read from HBM (requested D rows ahead
// and kept as loaded until it enters the window, where it is widened, so
// nothing waits on a load before its first use), and level l (1..L) computes
// row i - R*l from the 2R+1 rows of level
// l-1 it keeps in a register ring.  East/west neighbours come from the
// adjacent lanes by DPP whole-wave shifts; box shapes shift every row of
// their window once when it is produced, star shapes shift only the centre
// row.  Each level's valid region shrinks by R columns per side, absorbed by
// a ghost rim of R*L columns, and the segment's rows are extended by R*L ghost
// rows at each end.  Only level L is stored.
//
// Boundaries: at every level, the cells just outside the grid hold what the
// boundary rule reads there -- 0 (zero) or the nearest edge cell (clamp) --
// so the update itself never tests for a face.  Level 0 gets them from its
// loads; higher levels copy the edge row into the rows beyond the top and
// bottom faces when the edge row is produced, and the edge column into the
// lanes beyond the side faces (readlane).  Items that touch no face run a form
// without any of it.  This is the per-step kernel's rule applied level by
// level, so a pass equals L stored steps bit for bit: arithmetic is the shape
// table in order without FMA contraction (eval_shape) and every level is
// rounded to the storage format.
#pragma once

#include <type_traits>

#include "j2d_kernel.h"
#include "perks_device.h"

namespace perks {
namespace j2ds {

using fmt::Fmt;
using j2dk::eval_shape;
using j2dk::shape_desc;

constexpr int kWaves = 4;  // waves per workgroup (each runs its own items)

// Wave-uniform conditions that few rows meet: what they guard opens with
// keep_branch(), which the compiler may not execute speculatively, so it stays
// behind a branch instead of becoming a select per held value, level and row.
__device__ __forceinline__ bool rarely(bool c) { return __builtin_expect_with_probability(c, 0, 0.9999); }
__device__ __forceinline__ void keep_branch() { asm volatile(""); }

// sh[R + dx] = the row value at column x + dx, for dx in [-R, R]: lane i
// receives lane i-1 (west) or lane i+1 (east), repeatedly.
template <int R, typename C>
__device__ __forceinline__ void shifts(C c, C (&sh)[2 * R + 1])
{
    sh[R] = c;
#pragma unroll
    for (int k = 1; k <= R; ++k) {
        sh[R - k] = dpp_shift0<kDppWaveShr1>(sh[R - k + 1]);
        sh[R + k] = dpp_shift0<kDppWaveShl1>(sh[R + k - 1]);
    }
}

__device__ __forceinline__ float read_lane(float v, int l)
{
    return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), l));
}
__device__ __forceinline__ double read_lane(double v, int l)
{
    const uint64_t u = __double_as_longlong(v);
    const uint32_t lo = __builtin_amdgcn_readlane((uint32_t)u, l);
    const uint32_t hi = __builtin_amdgcn_readlane((uint32_t)(u >> 32), l);
    return __longlong_as_double((long long)(((uint64_t)hi << 32) | lo));
}

// v moved by s lanes (lane i receives lane i + s), s static after unrolling.
template <int R, typename C>
__device__ __forceinline__ C lane_shift(C v, int s)
{
    C w = v;
#pragma unroll
    for (int k = 0; k < R; ++k) {
        if (s < 0 && k < -s) w = dpp_shift0<kDppWaveShr1>(w);
        if (s > 0 && k < s) w = dpp_shift0<kDppWaveShl1>(w);
    }
    return w;
}

// The pair (columns x0 + dx, x1 + dx) for dx in [-R, R] from the pair (a, b)
// of columns (x0, x1): column x0 + m is lane floor(m/2), half m mod 2.
template <int R, typename C>
__device__ __forceinline__ void pair_shifts(C a, C b, C (&sa)[2 * R + 1], C (&sb)[2 * R + 1])
{
#pragma unroll
    for (int dx = -R; dx <= R; ++dx) {
        const int m0 = dx, m1 = dx + 1;
        const int s0 = m0 >= 0 ? m0 / 2 : -((1 - m0) / 2);
        const int s1 = m1 >= 0 ? m1 / 2 : -((1 - m1) / 2);
        sa[R + dx] = lane_shift<R, C>((m0 - 2 * s0) ? b : a, s0);
        sb[R + dx] = lane_shift<R, C>((m1 - 2 * s1) ? b : a, s1);
    }
}

// ---- row access ---------------------------------------------------------------
// Through a buffer descriptor that starts at the strip's first column inside
// the grid and ends with the row: an offset past the end reads 0 and drops a
// store, so lanes outside the grid (zero boundary) and lanes or rows that store
// nothing need no select and no branch.  Raw is the register form of a loaded
// word, unpacked when it is first used.
template <typename S, bool PAIR>
struct RowBuf;
template <typename S>
struct RowBuf<S, false> {
    using C = typename Fmt<S>::C;
    using Raw = typename Fmt<S>::Raw;
    __device__ static Raw ld(rsrc_t r, uint32_t off)
    {
        if constexpr (sizeof(S) == 2) return (uint32_t)__builtin_amdgcn_raw_buffer_load_b16(r, (int)off, 0, 0);
        else return buf_load(r, off, Raw{});
    }
    __device__ static void unpack(Raw w, C (&v)[1]) { v[0] = Fmt<S>::widen(w); }
    __device__ static void st(rsrc_t r, uint32_t off, const C (&v)[1])
    {
        if constexpr (sizeof(S) == 2) {
            S o;
            Fmt<S>::st(&o, 0, v[0]);
            __builtin_amdgcn_raw_buffer_store_b16(o.v, r, (int)off, 0, 0);
        } else {
            buf_store(r, off, v[0]);
        }
    }
    __device__ static void round(C (&v)[1], bool sr, uint32_t idx, uint32_t key)
    {
        if (sr) v[0] = Fmt<S>::qsr(v[0], idx, key);
        else v[0] = Fmt<S>::q(v[0]);
    }
};
// Columns x (even) and x + 1 in one load or store.
template <>
struct RowBuf<float, true> {
    using C = float;
    using Raw = float2;
    __device__ static Raw ld(rsrc_t r, uint32_t off)
    {
        return __builtin_bit_cast(Raw, __builtin_amdgcn_raw_buffer_load_b64(r, (int)off, 0, 0));
    }
    __device__ static void unpack(Raw w, C (&v)[2])
    {
        v[0] = w.x;
        v[1] = w.y;
    }
    __device__ static void st(rsrc_t r, uint32_t off, const C (&v)[2])
    {
        using v2i = int __attribute__((ext_vector_type(2)));
        __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(v2i, make_float2(v[0], v[1])), r, (int)off, 0, 0);
    }
    __device__ static void round(C (&)[2], bool, uint32_t, uint32_t) {}
};
template <typename S16, int FMT>
struct RowBuf16 {
    using C = float;
    using Raw = uint32_t;
    __device__ static Raw ld(rsrc_t r, uint32_t off)
    {
        return __builtin_amdgcn_raw_buffer_load_b32(r, (int)off, 0, 0);
    }
    __device__ static void unpack(Raw w, C (&v)[2])
    {
        v[0] = widen_lo<FMT>(w);
        v[1] = widen_hi<FMT>(w);
    }
    // v holds storage values already: the conversion is exact.
    __device__ static void st(rsrc_t r, uint32_t off, const C (&v)[2])
    {
        __builtin_amdgcn_raw_buffer_store_b32(Store16<FMT>::narrow2(v[0], v[1]), r, (int)off, 0, 0);
    }
    __device__ static void round(C (&v)[2], bool sr, uint32_t idx, uint32_t key)
    {
        if (sr) {
            v[0] = Fmt<S16>::qsr(v[0], idx, key);
            v[1] = Fmt<S16>::qsr(v[1], idx + 1u, key);
        } else {
            const uint32_t w = Store16<FMT>::narrow2(v[0], v[1]);
            v[0] = widen_lo<FMT>(w);
            v[1] = widen_hi<FMT>(w);
        }
    }
};
template <>
struct RowBuf<fmt::f16s, true> : RowBuf16<fmt::f16s, PERKS_F16> {};
template <>
struct RowBuf<fmt::bf16s, true> : RowBuf16<fmt::bf16s, PERKS_BF16> {};

// One work item.  PAIR: each lane holds two neighbouring columns (the strip is
// 128 columns wide and starts on an even column; the grid width must be even),
// so one load, store and set of lane shifts serves two cells.  EDGE: the strip
// reaches past a side face, or the segment's rows (its ghost rows included)
// reach row 0 or past the last one.
//
// A level computes a row as soon as the row it needs last arrives, without
// asking whether it is wanted: what a segment's rows are is known by position
// only.  In the first trip of a segment level l starts at stage 2R*l, fixed at
// compile time, as its window is whole from there on (trips are longer than
// 2R*L rows).  Every stage stores, where there is nothing to store to a descriptor
// of size 0.  So away from the faces a row costs its update and some 15 scalar
// operations, whatever the depth of the pass.  The 5-point star in FP32 has 9
// vector operations per row and level; the form with range and face tests and
// 64-bit addresses per row and level had some 20 scalar ones beside them, issued at
// the same rate.
//
// At a face under the zero boundary a row's select covers side and bottom alike,
// with no branch: the levels' rows are scheduled together.  Branches per level and
// row, though hardly ever taken: 512 FP32 grids of 64 to 1024 rows and columns, 5
// points, 12.9 ms, the select 11.7; 8192^2 FP32 9 points x 500 steps 29.8 and 28.2
// ms; 6000^2 BF16 5 points 0.90 of the time.  (A second copy of the trip without
// tests, for trips away from the faces, takes registers: 9 points at two workgroups
// per CU instead of four, 31.0 ms.)
//
// A segment of one trip (per step: the small ones) runs a form of its own, which
// requests no further rows and stores none but its own: on the smallest launches a
// CU's memory instructions count, not its arithmetic.  With every trip alike, 16-bit
// fields paid the hash and the rounding for 2R*L more rows a segment and level, and
// a short segment twice its memory instructions.  us for 100 steps, every trip
// alike -> here: BF16 stochastic 9 points (radius 2) 2048^2 clamp, one step per
// launch 1535 -> 1144, 5 points 8000 x 200 807 -> 637; FP16 25 points 2048^2 zero,
// two per pass 2388 -> 1644.
//
// And the loop has one way in, one back edge and the same memory operations on
// both: the compiler's waits for the rows in flight are those of the steady
// state.  With an exit or a conditional store between the rows it waited for
// every operation in flight once per trip.
template <int SHAPE, typename S, int BC, bool HAS_DIV, int L, bool PAIR, bool EDGE>
struct Strip {
    using C = typename Fmt<S>::C;
    using Row = RowBuf<S, PAIR>;
    using Raw = typename Row::Raw;
    static constexpr const ShapeDesc& SD = shape_desc<SHAPE>();
    static constexpr int R = SD.radius;
    static constexpr bool BOX = SD.is_box != 0;
    static constexpr bool ZERO = BC == PERKS_BC_ZERO;
    static constexpr int Q = 2 * R + 1;       // rows of a level's window
    static constexpr int D = stream_trip(R);  // level-0 rows loaded ahead: a multiple of Q
    static constexpr int UF = D;              // rows per loop trip, so every ring slot is static
    static constexpr int NS = BOX ? Q : 1;    // boxes keep the x shifts of a row
    static constexpr int H = PAIR ? 2 : 1;    // columns per lane

    // A segment's first trip of several, the ones after it, and the trip of a
    // segment that has one.
    enum { FIRST, LATER, ONLY };

    const S* src;
    S* dst;
    int nx, ny;
    int ys, ye;
    C k[kMaxGroups];
    double kd[kMaxGroups];
    double kdiv;
    bool sr;
    uint32_t key[L + 1];

    int x;                // this lane's first column
    bool out;             // the lane lies outside the grid
    bool xedge;           // the strip reaches past a side face
    int lane_w, lane_e;   // lanes holding columns 0 and nx-1 (clamped into the wave)
    uint32_t loff, soff;  // byte offsets from the descriptors' first column: load, store
    uint32_t span;        // bytes from that column to the row's end
    size_t row_bytes;
    const char* lp;       // the next row to load
    char* sp;             // the next row to store
    int lrow, lend;       // index of the next row to load, and of the last that is needed

    Raw fl[D];            // level-0 rows in flight (row i in slot (i - i0) mod D)
    C win[L][Q][NS][H];   // level l's window

    static constexpr int mq(int a) { return ((a % Q) + Q) % Q; }

    // Rows above the grid: row 0 (clamp) or nothing (zero: 0); below it, the same
    // rule.  The rows requested past the last one needed are that one again, from
    // the L1 (leaving them out costs a descriptor change per row: 4-6% of a pass).
    __device__ __forceinline__ Raw next_row()
    {
        const bool in = !EDGE || !ZERO || (uint32_t)lrow < (uint32_t)ny;
        const Raw w = Row::ld(make_rsrc(lp, in ? span : 0u), loff);
        lp += (!EDGE || lrow >= 0) && lrow < lend ? row_bytes : 0;
        ++lrow;
        return w;
    }

    __device__ __forceinline__ void store(bool ok, const C (&v)[H])
    {
        Row::st(make_rsrc(sp, ok ? span : 0u), soff, v);
        sp += row_bytes;
    }

    // sh[h][R + dx]: the value at column x + h + dx.
    __device__ __forceinline__ static void shift_row(const C (&v)[H], C (&sh)[H][Q])
    {
        if constexpr (PAIR) pair_shifts<R>(v[0], v[1], sh[0], sh[1]);
        else shifts<R>(v[0], sh[0]);
    }

    __device__ __forceinline__ void keep(int lv, int slot, const C (&v)[H])
    {
        if constexpr (BOX) {
            C sh[H][Q];
            shift_row(v, sh);
#pragma unroll
            for (int t = 0; t < Q; ++t)
#pragma unroll
                for (int h = 0; h < H; ++h) win[lv][slot][t][h] = sh[h][t];
        } else {
#pragma unroll
            for (int h = 0; h < H; ++h) win[lv][slot][0][h] = v[h];
        }
    }

    // Lanes beyond a side face take the edge value of their row (clamp).
    __device__ __forceinline__ void side_faces(C (&v)[H]) const
    {
        const C vw = read_lane(v[0], lane_w);
        const C ve = read_lane(v[H - 1], lane_e);
#pragma unroll
        for (int h = 0; h < H; ++h) v[h] = out ? (x < 0 ? vw : ve) : v[h];
    }

    // Level LV1 = LV + 1 computes row q = i - R*LV1 from level LV's window.  The
    // slot it writes held row q - Q, which no level needs any more.
    template <int TRIP, int U, int LV>
    __device__ __forceinline__ void level(int i)
    {
        if constexpr (TRIP != LATER && LV < L && U < 2 * R * (LV + 1)) {
            const C none[H] = {};
            if constexpr (TRIP == FIRST) store(false, none);
            else sp += row_bytes;
        } else if constexpr (LV < L) {
            constexpr int LV1 = LV + 1;
            constexpr int REL = U - R * LV1;  // relative index of row q
            const int q = i - R * LV1;
            C sh[H][Q];
            if constexpr (!BOX) {
                C c[H];
#pragma unroll
                for (int h = 0; h < H; ++h) c[h] = win[LV][mq(REL)][0][h];
                shift_row(c, sh);
            }
            C v[H];
#pragma unroll
            for (int h = 0; h < H; ++h)
                v[h] = eval_shape<SHAPE, C, HAS_DIV>(k, kdiv, kd, [&](int dy, int dx) -> C {
                    if constexpr (BOX) return win[LV][mq(REL + dy)][R + dx][h];
                    else return dy == 0 ? sh[h][R + dx] : win[LV][mq(REL + dy)][0][h];
                });
            if constexpr (sizeof(S) == 2)
                Row::round(v, sr, (uint32_t)q * (uint32_t)nx + (uint32_t)x, key[LV1]);
            if constexpr (LV1 == L) {
                store((uint32_t)(q - ys) < (uint32_t)(ye - ys), v);
            } else {
                if constexpr (EDGE && ZERO) {
                    // Lanes beyond a side face and rows beyond the others hold 0: one select
                    // with a mask, and no branch between the levels' rows.
                    const bool outside = out | ((uint32_t)q >= (uint32_t)ny);
#pragma unroll
                    for (int h = 0; h < H; ++h) v[h] = outside ? (C)0 : v[h];
                } else if constexpr (EDGE) {
                    if (rarely(xedge)) {
                        keep_branch();
                        side_faces(v);
                    }
                    if (rarely((uint32_t)q >= (uint32_t)ny)) {
                        // Rows below the bottom face read row ny-1.
                        // (Above the top one: row 0 once it is known, below.)
                        keep_branch();
#pragma unroll
                        for (int h = 0; h < H; ++h) v[h] = win[LV1][mq(REL - 1)][BOX ? R : 0][h];
                    }
                }
                keep(LV1, mq(REL), v);
                if constexpr (EDGE && !ZERO) {
                    if (rarely(q == 0)) {
                        // Rows above the top face read row 0.
                        keep_branch();
#pragma unroll
                        for (int j = 1; j <= R; ++j)
#pragma unroll
                            for (int t = 0; t < NS; ++t)
#pragma unroll
                                for (int h = 0; h < H; ++h)
                                    win[LV1][mq(REL - j)][t][h] = win[LV1][mq(REL)][t][h];
                    }
                }
            }
            level<TRIP, U, LV + 1>(i);
        }
    }

    // Iteration i (stage U = (i - i0) mod UF): level-0 row i, loaded D
    // iterations ago, enters the window, and row i + D is requested into its
    // in-flight slot.
    template <int TRIP, int U>
    __device__ __forceinline__ void stage(int i)
    {
        const Raw w = fl[U];
        if constexpr (TRIP != ONLY) fl[U] = next_row();  // issued before row i is waited for
        C v[H];
        Row::unpack(w, v);
        if constexpr (EDGE && PAIR && !ZERO) {
            // a pair beyond a side face loaded the edge pair: both halves take the edge column
            const C a = v[0], b = v[1];
            v[0] = x > nx - 2 ? b : a;
            v[1] = x < 0 ? a : b;
        }
        keep(0, mq(U), v);
        level<TRIP, U, 0>(i);
    }

    // One trip.  Rows past the segment's last are computed and not stored
    // (segments are cut to whole trips where they can be, cut_rows in j2d.hip).
    template <int TRIP, int U = 0>
    __device__ __forceinline__ void trip(int i)
    {
        if constexpr (U < UF) {
            stage<TRIP, U>(i);
            // Rows are scheduled one by one: mixed, their values take up to
            // 50% more registers.
            __builtin_amdgcn_sched_barrier(0);
            trip<TRIP, U + 1>(i + 1);
        }
    }

    // Rows [ys, ye) of the strip whose lane 0 holds column xs0; stores columns [vx0, vx1).
    __device__ __forceinline__ void run(int lane, int xs0, int vx0, int vx1)
    {
        x = xs0 + H * lane;
        out = x < 0 || x > nx - H;
        xedge = xs0 < 0 || xs0 + 64 * H - 1 >= nx;
        lane_w = min(max(-xs0 / H, 0), 63);
        lane_e = min(max((nx - H - xs0) / H, 0), 63);
        const int xb = max(xs0, 0);  // the descriptors' first column
        const int xc = x < 0 ? 0 : (x > nx - H ? nx - H : x);
        loff = ZERO && out ? kOob : (uint32_t)(xc - xb) * (uint32_t)sizeof(S);
        soff = x >= vx0 && x < vx1 ? (uint32_t)(x - xb) * (uint32_t)sizeof(S) : kOob;
        row_bytes = (size_t)nx * sizeof(S);
        span = (uint32_t)(min(nx - xb, 64 * H) * (int)sizeof(S));
        const int i0 = ys - R * L;
        const int iend = ye - 1 + R * L;
        lrow = i0;
        lend = min(iend, ny - 1);
        lp = reinterpret_cast<const char*>(src + (size_t)max(i0, 0) * nx + xb);
        sp = reinterpret_cast<char*>(dst + xb) + (ptrdiff_t)(i0 - R * L) * (ptrdiff_t)row_bytes;
#pragma unroll
        for (int t = 0; t < D; ++t) fl[t] = next_row();
        if constexpr (L == 1) {
            if (iend < i0 + UF) {
                trip<ONLY>(i0);
                return;
            }
        }
        trip<FIRST>(i0);
        for (int i = i0 + UF; i <= iend; i += UF) trip<LATER>(i);
    }
};

template <int SHAPE, typename S, int BC, bool HAS_DIV, bool PAIR>
__global__ void __launch_bounds__(kWaves * 64) j2d_stream_kernel(J2dArgs a, KCoefs cf)
{
    using C = typename Fmt<S>::C;
    constexpr const ShapeDesc& SD = shape_desc<SHAPE>();
    constexpr int R = SD.radius;
    constexpr int LM = stream_max_levels(R);
    C k[kMaxGroups];
    double kd[kMaxGroups];
#pragma unroll
    for (int g = 0; g < kMaxGroups; ++g) {
        k[g] = (C)cf.c[g];
        kd[g] = cf.c[g];
    }
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int G = gridDim.x;
    const int me = xcd_tile_id(blockIdx.x, G) * kWaves + wave;
    const int W = G * kWaves;

    for (int pass = 0; pass < a.npass; ++pass) {
        const int gp = pass + a.step_offset;
        const int ngrids = a.active[pass];
        const int nitems = a.grids[ngrids - 1].item_end;
        // Strips use the full-pass ghost rim in every pass.
        const int VW = PAIR ? 128 - 2 * pair_ghost(R, a.levels) : 64 - 2 * R * a.levels;
        for (int item = me; item < nitems; item += W) {
            int lo = 0, hi = ngrids - 1;  // first grid whose item_end > item
            while (lo < hi) {
                const int mid = (lo + hi) >> 1;
                if (a.grids[mid].item_end > item) hi = mid;
                else lo = mid + 1;
            }
            const J2dGrid gd = a.grids[lo];
            const int L = min(a.levels, gd.steps - gp * a.levels);
            const int local = item - (gd.item_end - gd.tiles);
            const int ntx = (gd.nx + VW - 1) / VW;
            const int tx = local % ntx, sg = local / ntx;
            const int vx0 = tx * VW, vx1 = min(vx0 + VW, gd.nx);
            const S* src = (const S*)((gp & 1) ? gd.b : gd.a);
            S* dst = (S*)((gp & 1) ? gd.a : gd.b);
            const int ys = sg == 0 ? 0 : gd.seg0 + (sg - 1) * gd.seg;
            const int ye = sg == 0 ? gd.seg0 : min(ys + gd.seg, gd.ny);
            auto run = [&](auto lv, auto& s) {
                constexpr int LL = decltype(lv)::value;
                s.src = src;
                s.dst = dst;
                s.nx = gd.nx;
                s.ny = gd.ny;
                s.ys = ys;
                s.ye = ye;
#pragma unroll
                for (int g = 0; g < kMaxGroups; ++g) {
                    s.k[g] = k[g];
                    s.kd[g] = kd[g];
                }
                s.kdiv = cf.divisor;
                s.sr = a.sr != 0;
#pragma unroll
                for (int l = 1; l <= LL; ++l)
                    s.key[l] = a.sr ? sr_key((uint32_t)(gp * a.levels + l - 1), a.seed) : 0u;
                s.run(lane, vx0 - (PAIR ? pair_ghost(R, LL) : R * LL), vx0, vx1);
            };
            auto go = [&](auto lv) {
                constexpr int LL = decltype(lv)::value;
                constexpr int RL = R * LL;
                const int xs0 = vx0 - (PAIR ? pair_ghost(R, LL) : RL);
                if (xs0 < 0 || xs0 + (PAIR ? 127 : 63) >= gd.nx || ys <= RL || ye + RL > gd.ny) {
                    Strip<SHAPE, S, BC, HAS_DIV, LL, PAIR, true> s;
                    run(lv, s);
                } else {
                    Strip<SHAPE, S, BC, HAS_DIV, LL, PAIR, false> s;
                    run(lv, s);
                }
            };
            if (L <= 1 || LM < 2) {
                go(std::integral_constant<int, 1>{});
            } else if constexpr (LM >= 2) {
                if (L == 2 || LM < 3) go(std::integral_constant<int, 2>{});
                else if constexpr (LM >= 3) {
                    if (L == 3 || LM < 4) go(std::integral_constant<int, 3>{});
                    else if constexpr (LM >= 4) go(std::integral_constant<int, 4>{});
                }
            }
        }
        if (pass + 1 < a.npass && !grid_sync(a.sync, G, a.timeout, pass == 0)) return;
    }
}

template <int SHAPE, typename S, bool PAIR>
void* sptr2(int bc, bool hd)
{
    if (bc == PERKS_BC_ZERO)
        return hd ? reinterpret_cast<void*>(&j2d_stream_kernel<SHAPE, S, PERKS_BC_ZERO, true, PAIR>)
                  : reinterpret_cast<void*>(&j2d_stream_kernel<SHAPE, S, PERKS_BC_ZERO, false, PAIR>);
    return hd ? reinterpret_cast<void*>(&j2d_stream_kernel<SHAPE, S, PERKS_BC_CLAMP, true, PAIR>)
              : reinterpret_cast<void*>(&j2d_stream_kernel<SHAPE, S, PERKS_BC_CLAMP, false, PAIR>);
}

template <typename S, bool PAIR>
void* sptr_p(int shape, int bc, bool hd)
{
    switch (shape) {
    case PERKS_SHAPE_2D_STAR_R1: return sptr2<PERKS_SHAPE_2D_STAR_R1, S, PAIR>(bc, hd);
    case PERKS_SHAPE_2D_STAR_R2: return sptr2<PERKS_SHAPE_2D_STAR_R2, S, PAIR>(bc, hd);
    case PERKS_SHAPE_2D_STAR_R3: return sptr2<PERKS_SHAPE_2D_STAR_R3, S, PAIR>(bc, hd);
    case PERKS_SHAPE_2D_STAR_R4: return sptr2<PERKS_SHAPE_2D_STAR_R4, S, PAIR>(bc, hd);
    case PERKS_SHAPE_2D_STAR_R5: return sptr2<PERKS_SHAPE_2D_STAR_R5, S, PAIR>(bc, hd);
    case PERKS_SHAPE_2D_STAR_R6: return sptr2<PERKS_SHAPE_2D_STAR_R6, S, PAIR>(bc, hd);
    case PERKS_SHAPE_2D_BOX_R1: return sptr2<PERKS_SHAPE_2D_BOX_R1, S, PAIR>(bc, hd);
    case PERKS_SHAPE_2D_BOX_R2: return sptr2<PERKS_SHAPE_2D_BOX_R2, S, PAIR>(bc, hd);
    default: return nullptr;
    }
}

// pair: the two-columns-per-lane form (FP32, FP16 and BF16 storage only).
template <typename S>
void* sptr(int shape, int bc, bool hd, bool pair)
{
    if constexpr (std::is_same_v<S, double>) {
        return pair ? nullptr : sptr_p<S, false>(shape, bc, hd);
    } else {
        return pair ? sptr_p<S, true>(shape, bc, hd) : sptr_p<S, false>(shape, bc, hd);
    }
}

}  // namespace j2ds
}  // namespace perks
