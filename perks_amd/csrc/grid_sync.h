// grid_sync.h -- the grid-wide barrier of the persistent (cooperative) kernels.
//
// State lives in one device block per launch, zeroed once when it is
// allocated.  A launch's first barrier is flat (every workgroup writes its
// L2 back and meets through kSyncGroups counters) and counts how many
// workgroups run on each XCD; the later ones meet per XCD first, and one
// workgroup of each XCD writes that XCD's L2 back and meets the other XCDs.
// Counters either return to zero within a barrier or only ever advance and
// are read relative to their value at the launch's start, so a launch needs
// no clearing kernel or memset beforehand (and a launch captured in a
// hipGraph carries none) and the next one may use any grid size.
//
// Why per XCD: the agent-scope release writes back the whole XCD's L2, and
// with every workgroup issuing one they queue up at that L2.  What a barrier
// costs on MI355X with 256 threads per workgroup and no dirty data, in us per
// barrier: 64 workgroups 4.2 flat, 2.2 with one write-back and one invalidate
// per XCD; 256: 6.3, 2.6; 512: 10.3, 3.1; 1024: 17.9, 4.0.  Counters without
// any fence take 3.9-4.6 flat and 1.9-3.7 per XCD.  Every workgroup still
// invalidates for itself (its CU's L1 has no other owner; an invalidate at
// workgroup scope leaves stale lines in it).  In the solves: 512 grids of 2D
// batch 18.6 -> 15.4 ms, CG at 64^3 13.1 -> 11.0 ms and at 256^3 819 -> 748 ms,
// 8192^2 FP32 box 34.7 -> 31.9 ms, 64^3 FP64 star 152 -> 143 us.
//
// Every wait is bounded.  A workgroup that waits longer than `timeout` ticks
// of the device wall clock sets the abort word and leaves; every other
// workgroup sees the word in its own wait (or at its next barrier) and leaves
// too, so the grid always drains.  The host checks the word after the launch
// (grid_sync_check) and reports PERKS_ERR_BARRIER_TIMEOUT.
#pragma once

#include <hip/hip_runtime.h>

namespace perks {

// Layout: the root block (the flat root counter, the root of the per-XCD
// form, the abort word, each on a line of its own), then kSyncGroups
// sub-groups, each with an arrival counter and a release word, then one block
// per XCD; blocks are 4352 bytes apart (17 x 256 B: they fall on different HBM
// channels).
//
// Flat form: workgroup w belongs to group w % kSyncGroups; the last arrival of
// a group arrives at the root; the last root arrival releases every group.  At
// most about G/32 atomics meet on one address, and each group polls its own
// word.  The last arrival of a group resets the group counter, and the
// releasing arrival resets the root, each with an atomic exchange that
// completes before the next step is issued.
constexpr int kSyncGroups = 32;
constexpr int kSyncStride = 4352 / 8;  // in 64-bit words

constexpr int kSyncXcds = 16;          // values of the XCC_ID register's field

struct GridSync {
    unsigned long long w[kSyncStride * (1 + kSyncGroups + kSyncXcds)];
};
static_assert(sizeof(GridSync) == 4352 * 49, "GridSync layout");
constexpr int kSyncAbortWord = 256;  // index of the abort word (2 KiB into the root block)
constexpr int kSyncXcdRoot = 128;    // index of the per-XCD form's root counter (1 KiB into the root block)

__device__ __forceinline__ unsigned int* gs_root(GridSync* gs) { return (unsigned int*)gs->w; }
__device__ __forceinline__ unsigned int* gs_abort(GridSync* gs) { return (unsigned int*)(gs->w + kSyncAbortWord); }
__device__ __forceinline__ unsigned int* gs_count(GridSync* gs, int g)
{
    return (unsigned int*)(gs->w + kSyncStride * (g + 1));
}

// Group layout of a grid of nblocks workgroups: ng = min(nblocks, kSyncGroups)
// groups, workgroup w in group w % ng, so group g has
// ceil((nblocks - g) / ng) members.  Host-callable so the arithmetic can be
// checked off the device.
__host__ __device__ constexpr unsigned int gs_groups(unsigned int nblocks)
{
    return nblocks < (unsigned int)kSyncGroups ? nblocks : (unsigned int)kSyncGroups;
}
__host__ __device__ constexpr unsigned int gs_members(unsigned int nblocks, unsigned int g)
{
    return (nblocks - g + gs_groups(nblocks) - 1) / gs_groups(nblocks);
}

// Waits until this thread's outstanding memory operations (here: an atomic
// exchange) have completed, and keeps the compiler from moving memory
// operations across the wait.
__device__ __forceinline__ void gs_complete()
{
    __atomic_signal_fence(__ATOMIC_SEQ_CST);
    __builtin_amdgcn_s_waitcnt(0);
    __atomic_signal_fence(__ATOMIC_SEQ_CST);
}
__device__ __forceinline__ unsigned int* gs_gen(GridSync* gs, int g)
{
    return (unsigned int*)(gs->w + kSyncStride * (g + 1) + 16);
}

// The per-XCD form.  An XCD's block: arrivals and releases (both only ever
// advance), the count of the launch's workgroups on it (zero between
// launches), and what the first barrier published for them: that count and
// the number of XCDs that hold any.
enum { kXcdCount = 0, kXcdGen = 32, kXcdCensus = 64, kXcdMembers = 96, kXcdActive = 97 };  // 32-bit words
__device__ __forceinline__ unsigned int* gs_xcd(GridSync* gs, int xcd, int word)
{
    return (unsigned int*)(gs->w + kSyncStride * (1 + kSyncGroups + xcd)) + word;
}
__device__ __forceinline__ unsigned int* gs_xcd_root(GridSync* gs) { return (unsigned int*)(gs->w + kSyncXcdRoot); }
// Whether an arrival that found `before` is the last of `members` in barrier
// `epoch` (1, 2, ...) of a launch that started with the counter at `base`.
__host__ __device__ constexpr bool gs_last(unsigned int before, unsigned int base, unsigned int epoch,
                                           unsigned int members)
{
    return before - base == epoch * members - 1;
}
// Whether a counter that started at `base` has advanced by `target` or more
// (it can be past it: others may be in a later barrier already).
__host__ __device__ constexpr bool gs_reached(unsigned int now, unsigned int base, unsigned int target)
{
    return (int)(now - base - target) >= 0;
}
// The XCD this wave runs on (a hardware register).
__device__ __forceinline__ int gs_xcc_id()
{
    int v;
    asm volatile("s_getreg_b32 %0, hwreg(HW_REG_XCC_ID, 0, 4)" : "=s"(v));
    return v & (kSyncXcds - 1);
}

// Thread 0 of a workgroup waits until done() holds.  False: the grid is
// aborting.  The abort word and the clock are looked at every 64th poll only.
template <bool SLEEP, class Done>
__device__ __forceinline__ bool gs_wait(GridSync* gs, unsigned long long timeout, const Done& done)
{
    const unsigned long long t0 = wall_clock64();
    unsigned int spins = 0;
    while (!done()) {
        if ((++spins & 63u) != 0u) {
            if (SLEEP) __builtin_amdgcn_s_sleep(1);
            continue;
        }
        if (__hip_atomic_load(gs_abort(gs), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) return false;
        if (wall_clock64() - t0 > timeout) {
            __hip_atomic_store(gs_abort(gs), 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            return false;
        }
    }
    return true;
}

// What thread 0 of a workgroup keeps from the first barrier for the later ones.
struct GridSyncState {
    int ok;
    int xcd;
    unsigned int members, active;     // workgroups on this XCD, XCDs with any
    unsigned int count0, gen0, root0; // the counters at the launch's start
    unsigned int epoch;
};

// All threads of the workgroup call this; `first` is true for the launch's
// first barrier and false for the others.  Every wave waits for its own loads
// and stores to complete and the workgroup meets; thread 0 then arrives.
// First barrier: it writes back the L2 at agent scope before it arrives (so
// the other XCDs see what the workgroup stored).  Later ones: the XCD's last
// arrival writes the L2 back for all of them -- their stores are in it, each
// arrived after its own had completed -- and meets the other XCDs.  Everyone
// invalidates L1/L2 at agent scope before the workgroup meets again and reads.
// Returns false when the grid is aborting: the caller must leave the kernel.
__device__ __forceinline__ bool grid_sync(GridSync* gs, unsigned int nblocks, unsigned long long timeout, bool first)
{
    __shared__ GridSyncState st;
    __atomic_signal_fence(__ATOMIC_SEQ_CST);
    __builtin_amdgcn_s_waitcnt(0);
    __syncthreads();
    if (nblocks == 1) return true;  // the workgroup has met
    if (threadIdx.x == 0) {
        // An offset the compiler does not know is 0: the addresses formed with
        // it stay here instead of being hoisted out of the caller's pass loop
        // into its registers.
        unsigned int here = 0;
        asm volatile("" : "+v"(here));
        gs = reinterpret_cast<GridSync*>(reinterpret_cast<char*>(gs) + here);
        bool ok = true;
        if (first) {
            const int xcd = gs_xcc_id();
            st.xcd = xcd;
            st.epoch = 0;
            // None of these moves before every workgroup has arrived here.
            st.count0 = __hip_atomic_load(gs_xcd(gs, xcd, kXcdCount), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            st.gen0 = __hip_atomic_load(gs_xcd(gs, xcd, kXcdGen), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            st.root0 = __hip_atomic_load(gs_xcd_root(gs), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            __hip_atomic_fetch_add(gs_xcd(gs, xcd, kXcdCensus), 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            const unsigned int ng = gs_groups(nblocks);
            const int g = (int)(blockIdx.x % ng);
            const unsigned int members = gs_members(nblocks, (unsigned int)g);
            unsigned int* gen = gs_gen(gs, g);
            // The release word is read before arriving (it cannot change without this
            // arrival); the release fence below also waits for this load and the count.
            const unsigned int g0 = __hip_atomic_load(gen, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "agent");
            gs_complete();
            const unsigned int before =
                __hip_atomic_fetch_add(gs_count(gs, g), 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            bool released = false;
            if (before == members - 1) {
                __hip_atomic_exchange(gs_count(gs, g), 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                gs_complete();
                const unsigned int rb =
                    __hip_atomic_fetch_add(gs_root(gs), 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                if (rb == ng - 1) {
                    __hip_atomic_exchange(gs_root(gs), 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                    unsigned int m[kSyncXcds], active = 0;
#pragma unroll
                    for (int x = 0; x < kSyncXcds; ++x)
                        m[x] = __hip_atomic_exchange(gs_xcd(gs, x, kXcdCensus), 0u, __ATOMIC_RELAXED,
                                                     __HIP_MEMORY_SCOPE_AGENT);
#pragma unroll
                    for (int x = 0; x < kSyncXcds; ++x) active += m[x] != 0 ? 1u : 0u;
#pragma unroll
                    for (int x = 0; x < kSyncXcds; ++x) {
                        if (m[x] == 0) continue;
                        __hip_atomic_store(gs_xcd(gs, x, kXcdMembers), m[x], __ATOMIC_RELAXED,
                                           __HIP_MEMORY_SCOPE_AGENT);
                        __hip_atomic_store(gs_xcd(gs, x, kXcdActive), active, __ATOMIC_RELAXED,
                                           __HIP_MEMORY_SCOPE_AGENT);
                    }
                    gs_complete();
                    for (unsigned int j = 0; j < ng; ++j)
                        __hip_atomic_fetch_add(gs_gen(gs, (int)j), 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                    released = true;
                }
            }
            if (!released)
                ok = gs_wait<true>(gs, timeout, [&] {
                    return __hip_atomic_load(gen, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != g0;
                });
            st.members =
                __hip_atomic_load(gs_xcd(gs, xcd, kXcdMembers), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            st.active = __hip_atomic_load(gs_xcd(gs, xcd, kXcdActive), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        } else {
            const int xcd = st.xcd;
            const unsigned int e = ++st.epoch;
            unsigned int* gen = gs_xcd(gs, xcd, kXcdGen);
            const unsigned int before = __hip_atomic_fetch_add(gs_xcd(gs, xcd, kXcdCount), 1u, __ATOMIC_RELAXED,
                                                               __HIP_MEMORY_SCOPE_AGENT);
            if (gs_last(before, st.count0, e, st.members)) {
                __builtin_amdgcn_fence(__ATOMIC_RELEASE, "agent");
                gs_complete();
                unsigned int* root = gs_xcd_root(gs);
                const unsigned int root0 = st.root0, target = e * st.active;
                __hip_atomic_fetch_add(root, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                // one poller per XCD: no sleep between polls
                ok = gs_wait<false>(gs, timeout, [&] {
                    return gs_reached(__hip_atomic_load(root, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT), root0,
                                      target);
                });
                if (ok) __hip_atomic_fetch_add(gen, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            } else {
                const unsigned int gen0 = st.gen0;
                ok = gs_wait<true>(gs, timeout, [&] {
                    return gs_reached(__hip_atomic_load(gen, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT), gen0, e);
                });
            }
        }
        if (ok && __hip_atomic_load(gs_abort(gs), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) ok = false;
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
        st.ok = ok ? 1 : 0;
    }
    __syncthreads();
    return st.ok != 0;
}

// Cooperative grids are sized to at most this many waves per CU.  On MI355X
// a grid of 8 four-wave workgroups per CU (every wave slot the occupancy
// query reports) did not reach its first barrier within the wait limit,
// while grids of up to 16 waves per CU meet every barrier; the persistent
// kernels' measured optimum is at or below that anyway.
constexpr int kCoopMaxWavesPerCu = 16;

// ---- host side ----------------------------------------------------------------
// Barrier blocks come from a per-device pool.  A launch leases a block of its
// own for the time from the launch until grid_sync_check has seen the launch
// complete, so launches from different host threads or streams never share
// counters or abort words.  A batch plan owns a block for its whole lifetime
// (grid_sync_alloc / grid_sync_free), so perks_release() cannot free a block
// that a captured graph still names.

// Takes a zeroed block from the current device's pool (allocating one when
// the pool is empty).
int grid_sync_acquire(GridSync** out);
// Returns a block taken with grid_sync_acquire to the pool of the device it
// came from.  The block must be idle (its launch completed and checked).
void grid_sync_return(GridSync* gs);
// A block owned by the caller (allocated and zeroed on the current device).
int grid_sync_alloc(GridSync** out);
int grid_sync_free(GridSync* gs);
// Wait limit in wall-clock ticks for one barrier (10 s of the current device).
unsigned long long grid_sync_timeout();
// After a launch has completed: PERKS_OK, or PERKS_ERR_BARRIER_TIMEOUT (the
// block is then cleared for the next launch).  Synchronises `stream`.
int grid_sync_check(GridSync* gs, hipStream_t stream);
// Frees the current device's idle pooled blocks (leased and plan-owned blocks
// stay valid).
int grid_sync_release();

// Launches a persistent grid (at most CUs x measured occupancy workgroups)
// cooperatively.  The HIP runtime refuses a cooperative launch with
// hipErrorIllegalState while another process on the device holds its
// cooperative queue; the same grid then goes out as an ordinary launch, which
// an otherwise idle device places whole, and whose barrier's bounded wait
// turns a grid that is not co-resident into PERKS_ERR_BARRIER_TIMEOUT rather
// than a hang.
hipError_t launch_persistent(const void* fn, dim3 grid, dim3 block, void** args, size_t lds, hipStream_t stream);

// Scope guard for a leased block.
struct SyncLease {
    GridSync* gs = nullptr;
    SyncLease() = default;
    SyncLease(const SyncLease&) = delete;
    SyncLease& operator=(const SyncLease&) = delete;
    int acquire() { return gs ? 0 : grid_sync_acquire(&gs); }
    ~SyncLease()
    {
        if (gs) grid_sync_return(gs);
    }
};

}  // namespace perks
