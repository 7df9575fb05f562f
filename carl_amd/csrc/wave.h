// wave.h - wave64 primitives: DPP prefix sum and a cooperative item loop.
//
// The per-car and per-ball candidate lists of one tick vary from a handful
// of triangles to several hundred, so a lane-per-object loop leaves most of
// a wavefront idle behind its longest list.  waveItemsPipelined and
// waveItemsIndexed flatten the lists of all 64 lanes and hand out (owner lane,
// item) pairs 64 at a time.
#pragma once

#include <hip/hip_runtime.h>

namespace carl {

// Inclusive scan over the 64 lanes: Hillis-Steele inside each row of 16
// lanes with row_shr 1/2/4/8, then row_bcast:15 and row_bcast:31 carry the
// row totals across the four rows.
__device__ __forceinline__ int waveInclusiveScan(int v)
{
    v += __builtin_amdgcn_update_dpp(0, v, 0x111, 0xf, 0xf, false);  // row_shr:1
    v += __builtin_amdgcn_update_dpp(0, v, 0x112, 0xf, 0xf, false);  // row_shr:2
    v += __builtin_amdgcn_update_dpp(0, v, 0x114, 0xf, 0xf, false);  // row_shr:4
    v += __builtin_amdgcn_update_dpp(0, v, 0x118, 0xf, 0xf, false);  // row_shr:8
    v += __builtin_amdgcn_update_dpp(0, v, 0x142, 0xa, 0xf, false);  // row_bcast:15 -> rows 1,3
    v += __builtin_amdgcn_update_dpp(0, v, 0x143, 0xc, 0xf, false);  // row_bcast:31 -> rows 2,3
    return v;
}

// Inclusive maximum over the 64 lanes, the same way.
__device__ __forceinline__ unsigned waveInclusiveMax(unsigned v)
{
    auto step = [&](unsigned x) { v = x > v ? x : v; };
    step((unsigned)__builtin_amdgcn_update_dpp(0, (int)v, 0x111, 0xf, 0xf, false));
    step((unsigned)__builtin_amdgcn_update_dpp(0, (int)v, 0x112, 0xf, 0xf, false));
    step((unsigned)__builtin_amdgcn_update_dpp(0, (int)v, 0x114, 0xf, 0xf, false));
    step((unsigned)__builtin_amdgcn_update_dpp(0, (int)v, 0x118, 0xf, 0xf, false));
    step((unsigned)__builtin_amdgcn_update_dpp(0, (int)v, 0x142, 0xa, 0xf, false));
    step((unsigned)__builtin_amdgcn_update_dpp(0, (int)v, 0x143, 0xc, 0xf, false));
    return v;
}

// The owner and position of the flattened items of a wave's lists, 64 items
// per call, in ascending order from 0.  Each owner whose list starts among
// the call's items leaves its lane and that place at the item's slot, and a
// maximum scan carries it to the items that follow: one LDS write, one read
// and a DPP scan, where a binary search of the starts waits for six dependent
// reads.  `slots` is 64 words of LDS private to this wave.  Every lane calls
// it.
struct ItemOwners {
    unsigned* slot;
    int excl, count;           // this lane's list: its first item and its length
    int base = 0;              // the next call's first item
    int lastOwner = 0, lastStart = 0;   // the list that the previous call ended in

    __device__ __forceinline__ ItemOwners(int* slots, int excl_, int count_)
        : slot((unsigned*)slots), excl(excl_), count(count_)
    {
        slot[threadIdx.x & 63] = 0;
    }
    // item base + lane: owner o, position q in its list (past the last item,
    // the last list's owner and a position beyond it)
    __device__ __forceinline__ void next(int& o, int& q)
    {
        const int lane = (int)(threadIdx.x & 63);
        const unsigned at = (unsigned)(excl - base);
        fence();
        if (count > 0 && at < 64u) slot[at] = (unsigned)(lane + 1) << 6 | at;
        fence();
        unsigned v = slot[lane];
        fence();
        slot[lane] = 0;
        v = waveInclusiveMax(v);
        o = v ? (int)(v >> 6) - 1 : lastOwner;
        q = v ? lane - (int)(v & 63) : base + lane - lastStart;
        const int end = __builtin_amdgcn_readlane((int)v, 63);
        if (end) {
            lastOwner = (end >> 6) - 1;
            lastStart = base + (end & 63);
        }
        base += 64;
    }
    static __device__ __forceinline__ void fence()
    {
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    }
};

// Calls process(value, owner, item, base) once for every item < count of
// every lane of the wave, with all lanes busy.  Items of one owner are visited
// in ascending order, owners in ascending lane order, 64 consecutive pairs per
// round; pair j = base + lane runs on `lane` (base is the round's first pair),
// so the items of one owner in a round sit on consecutive lanes.  A two-stage
// pipeline: fetch(owner, item, valid) issues the loads of the next round
// before process runs on the current one, so each round's memory latency
// overlaps the previous round's work.  after(last) runs on every lane of the
// wave once per round, after process.  `excl` is 64 ints of LDS private to
// this wave (ItemOwners); every lane of the wave must call it (count 0 for
// lanes without work).
template <typename Fetch, typename Process, typename After>
__device__ __forceinline__ void waveItemsPipelined(int count, int* excl, Fetch&& fetch, Process&& process,
                                                   After&& after)
{
    const int lane = (int)(threadIdx.x & 63);
    const int incl = waveInclusiveScan(count);
    const int total = __builtin_amdgcn_readlane(incl, 63);
    if (total == 0) return;
    ItemOwners owners(excl, incl - count, count);
    int o, q;
    owners.next(o, q);
    auto cur = fetch(o, q, lane < total);
    for (int base = 0; base < total; base += 64) {
        const int jn = base + 64 + lane;
        int on, qn;
        owners.next(on, qn);
        auto next = fetch(on, qn, jn < total);
        if (base + lane < total) process(cur, o, q, base);
        after(base + 64 >= total);   // every lane; true after the last round
        cur = next;
        o = on;
        q = qn;
    }
}

// waveItemsPipelined for items reached through an index: index(owner, item,
// valid) loads an item's index and fetch(index, owner, valid) its data
// through it.  The index loads run Lead + 1 rounds ahead of process(value,
// owner, base) and the data loads one round ahead, so a round waits for
// neither load's full latency (the indices are small lists, the data a small
// per-index table; both stay in the caches that per-item copies of the data
// overflow).  Same visiting order, lane placement and after() hook as
// waveItemsPipelined.
template <int Lead, typename Index, typename Fetch, typename Process, typename After>
__device__ __forceinline__ void waveItemsIndexed(int count, int* excl, Index&& index, Fetch&& fetch,
                                                 Process&& process, After&& after)
{
    const int lane = (int)(threadIdx.x & 63);
    const int incl = waveInclusiveScan(count);
    const int total = __builtin_amdgcn_readlane(incl, 63);
    if (total == 0) return;
    ItemOwners owners(excl, incl - count, count);
    // slot r of the ring holds the owner and index of round m + 1 while
    // round m (m = r mod Lead) is processed
    int ringO[Lead], ringX[Lead];
    int o0, q0;
    owners.next(o0, q0);
    const int x0 = index(o0, q0, lane < total);
#pragma unroll
    for (int r = 0; r < Lead; r++) {
        int q;
        owners.next(ringO[r], q);
        ringX[r] = index(ringO[r], q, (r + 1) * 64 + lane < total);
    }
    auto cur = fetch(x0, o0, lane < total);
    int curO = o0;
    for (int base = 0; base < total;) {
#pragma unroll
        for (int r = 0; r < Lead; r++) {
            if (base < total) {
                const int nextO = ringO[r];
                auto next = fetch(ringX[r], nextO, base + 64 + lane < total);
                const int ja = base + (Lead + 1) * 64 + lane;
                int q;
                owners.next(ringO[r], q);
                ringX[r] = index(ringO[r], q, ja < total);
                if (base + lane < total) process(cur, curO, base);
                after(base + 64 >= total);   // every lane; true after the last round
                cur = next;
                curO = nextO;
                base += 64;
            }
        }
    }
}

// Without a per-round hook.
template <typename Fetch, typename Process>
__device__ __forceinline__ void waveItemsPipelined(int count, int* excl, Fetch&& fetch, Process&& process)
{
    waveItemsPipelined(count, excl, fetch, process, [](bool) {});
}

}  // namespace carl
