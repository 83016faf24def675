// j3d_sweep_kernel.h -- one time step of the 3D shapes whose table runs plane
// by plane (the 27-point box and the 17-point type-0 stencil), instantiated
// beside the register-streaming kernel in j3d_stream_{f64,f32,f16,bf16}.hip.
//
// The table of these shapes sums the points of plane z-1 first, then those of
// z, then those of z+1.  So a plane need not stay: when plane i arrives, its
// cells close the sums of output plane i-1 (its z+1 terms), carry on those of
// plane i (z terms) and open those of plane i+1 (z-1 terms), and each cell's sum
// still runs through the table in order.  A wave keeps two running sums per cell
// instead of a window of three planes, and one set of lane shifts per plane
// instead of three.
//
// What bounds it: 27 products and 26 sums a cell in FP64 arithmetic (also for
// FP32 and 16-bit storage: the reference writes these weights as double
// literals) while the fields stay in the caches, then one read and one write of
// the field per step.  The windowed kernel takes two steps per pass to halve
// that traffic, but its 64 x 8 tile then keeps 60 x 4 cells; here a tile keeps
// all its rows and 62 of 64 columns.
//
// ms for 50 steps, clamp, windowed -> here.  27 points 256^3 persistent: FP64 4.68 ->
// 2.77 (303 Gcell/s, 16.0 T FP64 operations/s), FP32 4.54 -> 2.59, bf16 5.69 -> 2.94;
// per step 4.69 -> 2.51, 3.71 -> 2.28, 4.44 -> 2.48; 512^3 FP32 27.2 -> 17.2, per step
// 21.5 -> 15.4.  17 points 256^3 persistent: FP64 3.52 -> 2.19, FP32 3.07 -> 1.63, bf16
// 3.74 -> 1.97; per step 4.36 -> 2.20, 2.75 -> 1.35, 3.14 -> 1.49; 512^3 FP32 17.7 ->
// 16.2, per step 15.0 both.  100^3 FP64: 27 points 0.76 -> 0.60, 17 points 0.64 -> 0.51.
//
// Rows: 4 a tile.  8 read less beyond the tile (512^3 FP32 17-point plain 13.7
// against 15.5 ms) but make half the waves (64^3 FP64 27-point plain 0.43
// against 0.31 ms, 160^3 1.03 against 0.83).  Two planes are in flight; a third
// costs stages where a slab's planes do not fill a trip (64^3 0.39 ms, 200^3
// 1.60 against 1.49).  Stores are ordinary ones: past the caches (nontemporal)
// the next step reads memory (256^3 FP64 17-point 2.5 -> 3.4 ms).
//
// A work item is a tile of 62 x kSweepRows cells over a z-slab; each wave runs
// its own items.  All boundary handling is in the loads: clamped rows, columns
// and planes, or offsets and descriptors that read 0.
#pragma once

#include "j3d_general_kernel.h"
#include "perks_device.h"

namespace perks {
namespace j3z {

using fmt::Fmt;
using j3g::J3gArgs;
using j3g::shape3;

constexpr int kWaves = 4;      // waves per workgroup (each runs its own items)
constexpr int kSweepRows = 4; // rows of a tile
constexpr int kSweepCols = 62; // stored columns of a tile

constexpr int kSweepAhead = 2; // planes loaded ahead, and stages per loop trip

// Stages an item of a slab of nz planes runs (a ghost plane on either side).
inline int sweep_stages(int nz) { return (nz + 2 + kSweepAhead - 1) / kSweepAhead * kSweepAhead; }

// The table's groups run through the planes z-1, z, z+1 in that order, each group within one.
constexpr bool plane_ordered(const ShapeDesc& s)
{
    int last = -1;
    for (int g = 0; g < s.ngroups; ++g) {
        const int dz = s.g[g].off[0][0];
        for (int p = 1; p < s.g[g].npts; ++p)
            if (s.g[g].off[p][0] != dz) return false;
        if (dz < last || dz > 1 || dz < -1) return false;
        last = dz;
    }
    return s.dims == 3 && s.radius == 1 && s.g[0].off[0][0] == -1 && last == 1;
}
// Whether the kernel is built for a shape.
inline bool sweeps(int shape) { return shape == PERKS_SHAPE_3D_TYPE0_R1 || shape == PERKS_SHAPE_3D_BOX_R1; }

template <typename S>
__device__ __forceinline__ typename Fmt<S>::Raw plane_ld(rsrc_t r, uint32_t off)
{
    if constexpr (sizeof(S) == 2) return (uint32_t)__builtin_amdgcn_raw_buffer_load_b16(r, (int)off, 0, 0);
    else return buf_load(r, off, typename Fmt<S>::Raw{});
}
template <typename S>
__device__ __forceinline__ void plane_st(rsrc_t r, uint32_t off, typename Fmt<S>::C v)
{
    if constexpr (sizeof(S) == 2) {
        S o;
        Fmt<S>::st(&o, 0, v);
        __builtin_amdgcn_raw_buffer_store_b16(o.v, r, (int)off, 0, 0);
    } else {
        buf_store(r, off, v);
    }
}

template <int SHAPE, typename S, int BC, bool HAS_DIV, int NY>
struct Sweep {
    using C = typename Fmt<S>::C;
    static constexpr const ShapeDesc& SD = shape3<SHAPE>();
    static_assert(plane_ordered(SD));
    static_assert(sizeof(C) == 8 || j3g::first_f64_group3<SHAPE>() == 0, "sums are carried in double throughout");
    static constexpr bool ZERO = BC == PERKS_BC_ZERO;
    static constexpr int R = NY + 2;  // rows read of a plane
    static constexpr int D = kSweepAhead;
    using Raw = typename Fmt<S>::Raw;

    const S* src;
    S* dst;
    int nz, ny, nx;
    size_t plane;
    uint32_t plane_bytes;
    int x, y0;          // this lane's column, the tile's first stored row
    uint32_t loff[R];   // byte offsets in a plane: rows y0-1 .. y0+NY
    uint32_t soff[NY];
    int zs, ze;
    double kd[kMaxGroups];
    double kdiv;
    bool sr;
    uint32_t key;

    Raw fl[D][R];       // planes in flight
    double acc[NY];     // sums of the arriving plane's cells: their z-1 terms
    double accl[NY];    // sums of the plane before: their z-1 and z terms

    __device__ __forceinline__ void load(int q, Raw (&w)[R]) const
    {
        const int qc = q < 0 ? 0 : (q >= nz ? nz - 1 : q);
        const rsrc_t rs = make_rsrc(src + (size_t)qc * plane, !ZERO || qc == q ? plane_bytes : 0u);
#pragma unroll
        for (int r = 0; r < R; ++r) w[r] = plane_ld<S>(rs, loff[r]);
    }

    // Every stage stores, planes outside the slab to a descriptor of size 0:
    // the waits for the planes in flight then count the same operations on
    // every way through the loop.
    __device__ __forceinline__ rsrc_t store_to(int q) const
    {
        const bool ok = q >= zs && q < ze;
        return make_rsrc(dst + (size_t)(ok ? q : 0) * plane, ok ? plane_bytes : 0u);
    }

    // The terms of plane DZ added to a sum in table order (DZ = -1 opens it).
    // v[dy + 1][dx + 1]: the arriving plane's values around the cell.
    template <int DZ>
    __device__ __forceinline__ double terms(double a, const C (&v0)[3], const C (&v1)[3], const C (&v2)[3]) const
    {
        auto at = [&](int dy, int dx) -> C { return dy < 0 ? v0[dx + 1] : (dy == 0 ? v1[dx + 1] : v2[dx + 1]); };
#pragma unroll
        for (int g = 0; g < SD.ngroups; ++g) {
            if (SD.g[g].off[0][0] != DZ) continue;
            C s = at(SD.g[g].off[0][1], SD.g[g].off[0][2]);
#pragma unroll
            for (int p = 1; p < SD.g[g].npts; ++p) s = s + at(SD.g[g].off[p][1], SD.g[g].off[p][2]);
            const double prod = kd[g] * (double)s;
            a = g == 0 ? prod : a + prod;
        }
        return a;
    }

    static_assert(D == 2, "run() writes out one stage per slot");

    // Plane i is in slot U; plane i + D is requested into it when it is done.
    template <int U>
    __device__ __forceinline__ void stage(int i)
    {
        const rsrc_t rs = store_to(i - 1);
        C v[3][3];
        auto shift = [&](int r, C (&o)[3]) {
            o[1] = Fmt<S>::widen(fl[U][r]);
            o[0] = dpp_shift0<kDppWaveShr1>(o[1]);
            o[2] = dpp_shift0<kDppWaveShl1>(o[1]);
        };
        shift(0, v[0]);
        shift(1, v[1]);
#pragma unroll
        for (int r = 0; r < NY; ++r) {
            shift(r + 2, v[(r + 2) % 3]);
            const C(&a)[3] = v[r % 3];
            const C(&b)[3] = v[(r + 1) % 3];
            const C(&c)[3] = v[(r + 2) % 3];
            const double sum = terms<1>(accl[r], a, b, c);
            accl[r] = terms<0>(acc[r], a, b, c);
            acc[r] = terms<-1>(0.0, a, b, c);
            const C u = (C)(HAS_DIV ? sum / kdiv : sum);
            C out;
            if (sr) {
                const uint32_t idx = (uint32_t)(((size_t)(i - 1) * ny + (size_t)(y0 + r)) * nx + (size_t)x);
                out = Fmt<S>::qsr(u, idx, key);
            } else {
                out = Fmt<S>::q(u);
            }
            plane_st<S>(rs, soff[r], out);
        }
        load(i + D, fl[U]);
    }

    // Tile whose lane 0 is column xs0 and first row is y0, planes [zs, ze).
    __device__ __forceinline__ void run(int lane, int xs0)
    {
        x = xs0 + lane;
        const int xc = x < 0 ? 0 : (x >= nx ? nx - 1 : x);
#pragma unroll
        for (int r = 0; r < R; ++r) {
            const int y = y0 + r - 1;
            const int yc = y < 0 ? 0 : (y >= ny ? ny - 1 : y);
            const bool in = x == xc && y == yc;
            loff[r] = ZERO && !in ? kOob : (uint32_t)(yc * nx + xc) * (uint32_t)sizeof(S);
        }
#pragma unroll
        for (int r = 0; r < NY; ++r) {
            const bool mine = lane >= 1 && lane <= kSweepCols && x < nx && y0 + r < ny;
            soff[r] = mine ? (uint32_t)((y0 + r) * nx + x) * (uint32_t)sizeof(S) : kOob;
        }
#pragma unroll
        for (int r = 0; r < NY; ++r) acc[r] = accl[r] = 0.0;
#pragma unroll
        for (int t = 0; t < D; ++t) {
            const rsrc_t nowhere = store_to(-1);
#pragma unroll
            for (int r = 0; r < NY; ++r) plane_st<S>(nowhere, soff[r], (C)0);
            load(zs - 1 + t, fl[t]);
        }
        for (int i = zs - 1; i <= ze; i += D) {
            // fenced: mixed, two planes' values take more registers
            stage<0>(i);
            __builtin_amdgcn_sched_barrier(0);
            stage<1>(i + 1);
            __builtin_amdgcn_sched_barrier(0);
        }
    }
};

template <int SHAPE, typename S, int BC, bool HAS_DIV, int NY>
__global__ void __launch_bounds__(kWaves * 64) j3z_kernel(J3gArgs a, KCoefs cf)
{
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int G = gridDim.x;
    const int me = xcd_tile_id(blockIdx.x, G) * kWaves + wave;
    const int W = G * kWaves;
    const int nz = a.nz, ny = a.ny, nx = a.nx;
    const int ntx = (nx + kSweepCols - 1) / kSweepCols, nty = (ny + NY - 1) / NY;
    const int nitems = ntx * nty * a.nzs;

    for (int pass = 0; pass < a.npass; ++pass) {
        const int gp = pass + a.step_offset;
        const S* src = (const S*)((gp & 1) ? a.b : a.a);
        S* dst = (S*)((gp & 1) ? a.a : a.b);
        for (int item = me; item < nitems; item += W) {
            const int tx = item % ntx;
            const int ty = (item / ntx) % nty;
            const int zsl = item / (ntx * nty);
            Sweep<SHAPE, S, BC, HAS_DIV, NY> t;
            t.src = src;
            t.dst = dst;
            t.nz = nz;
            t.ny = ny;
            t.nx = nx;
            t.plane = (size_t)ny * nx;
            t.plane_bytes = (uint32_t)(t.plane * sizeof(S));
            t.y0 = ty * NY;
            t.zs = (int)(((long long)zsl * nz) / a.nzs);
            t.ze = (int)(((long long)(zsl + 1) * nz) / a.nzs);
#pragma unroll
            for (int g = 0; g < kMaxGroups; ++g) t.kd[g] = cf.c[g];
            t.kdiv = cf.divisor;
            t.sr = a.sr != 0;
            t.key = a.sr ? sr_key((uint32_t)gp, a.seed) : 0u;
            t.run(lane, tx * kSweepCols - 1);
        }
        if (pass + 1 < a.npass && !grid_sync(a.sync, G, a.timeout, pass == 0)) return;
    }
}

template <int SHAPE, typename S>
void* zptr_bc(int bc, bool has_div)
{
    constexpr int NY = kSweepRows;
    if (bc == PERKS_BC_ZERO)
        return has_div ? reinterpret_cast<void*>(&j3z_kernel<SHAPE, S, PERKS_BC_ZERO, true, NY>)
                       : reinterpret_cast<void*>(&j3z_kernel<SHAPE, S, PERKS_BC_ZERO, false, NY>);
    return has_div ? reinterpret_cast<void*>(&j3z_kernel<SHAPE, S, PERKS_BC_CLAMP, true, NY>)
                   : reinterpret_cast<void*>(&j3z_kernel<SHAPE, S, PERKS_BC_CLAMP, false, NY>);
}

template <typename S>
void* zptr(int shape, int bc, bool has_div)
{
    switch (shape) {
    case PERKS_SHAPE_3D_TYPE0_R1: return zptr_bc<PERKS_SHAPE_3D_TYPE0_R1, S>(bc, has_div);
    case PERKS_SHAPE_3D_BOX_R1: return zptr_bc<PERKS_SHAPE_3D_BOX_R1, S>(bc, has_div);
    default: return nullptr;
    }
}

}  // namespace j3z

// Kernel entry points per storage format (j3d_stream_<fmt>.hip).
void* j3z_kernel_f64(int shape, int bc, bool has_div);
void* j3z_kernel_f32(int shape, int bc, bool has_div);
void* j3z_kernel_f16(int shape, int bc, bool has_div);
void* j3z_kernel_bf16(int shape, int bc, bool has_div);

}  // namespace perks
