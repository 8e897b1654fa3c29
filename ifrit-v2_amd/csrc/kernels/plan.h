// The tile plan: a launch of its own, or the second half of k_clip_plan.
#pragma once
#include "device_common.h"

namespace ifrit_hip {
namespace dev {

// ---------------------------------------------------------------------------
// Raster planning over the tiles of all views: each workgroup
// scans its quantities over its 256 tiles and takes its range of each with one
// atomic on the draw's totals.  The workgroups' ranges come in any order, but
// every tile's list is contiguous, the lists are disjoint, and a workgroup's
// tiles stay together.  A tile's list is cut into items of at most 1 <<
// partShift entries; items of more than kRasterPass entries are listed from
// the front of the item array and the others from its back, so that the queue
// hands out the long ones first.  Tiles with several items get a partial key
// block per item and go to the front of multiList; empty tiles go to its back.  The
// tiles of shaded views are also listed by the length of their lists (ShadeOrder).
//
// The plan is also where a draw's live counters end: it publishes the draw's
// own and leaves the tile counts and the live counters at zero, so that the
// next draw needs no clearing launch.
// ---------------------------------------------------------------------------
constexpr int kPlanQ = kTotCount + 2;  // PlanTotal, then the classes of ShadeOrder, two to a word

struct TilePlan {
    unsigned q[kPlanQ];
};

__device__ __forceinline__ TilePlan tile_plan(unsigned c, bool valid, int cls, int sh) {
    TilePlan w;
    const unsigned part = 1u << sh;
    const unsigned p = valid ? (c + part - 1u) >> sh : 0u;
    const unsigned last = c - (p ? p - 1u : 0u) * part;  // entries of the last item
    const unsigned shortItems = p && last <= (unsigned)kRasterPass ? 1u : 0u;
    w.q[kTotEntries] = valid ? c : 0u;
    w.q[kTotLong] = p - shortItems;
    w.q[kTotShort] = shortItems;
    w.q[kTotPartials] = p > 1u ? p : 0u;
    w.q[kTotMulti] = p > 1u ? 1u : 0u;
    w.q[kTotEmpty] = valid && p == 0u ? 1u : 0u;
    w.q[kTotCount] = cls < 2 ? 1u << (16 * cls) : 0u;
    w.q[kTotCount + 1] = cls == 2 || cls == 3 ? 1u << (16 * (cls - 2)) : 0u;
    return w;
}

// Exclusive scan of kPlanQ values over a 256-thread workgroup; every thread must call it.
__device__ __forceinline__ void plan_scan(unsigned* v, unsigned (*sWave)[4], unsigned* total) {
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
#pragma unroll
    for (int k = 0; k < kPlanQ; k++) {
        const unsigned x = wave_incl_scan(v[k]);
        if (lane == 63) sWave[k][w] = x;
        v[k] = x - v[k];
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < kPlanQ; k++) {
        unsigned base = 0;
#pragma unroll
        for (int i = 0; i < 4; i++) base += i < w ? sWave[k][i] : 0u;
        v[k] += base;
        total[k] = sWave[k][0] + sWave[k][1] + sWave[k][2] + sWave[k][3];
    }
}

// What other workgroups of the launch count, read past this XCD's L2.
template <class T>
__device__ __forceinline__ T shared_load(const T* p) {
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// One workgroup of the plan.
__device__ __forceinline__ void plan_block(unsigned long long* __restrict__ cnt, unsigned* __restrict__ start,
                                           unsigned* __restrict__ cursor, int n, const Views& V, const RasterQueue& q,
                                           DeviceCounters* ctr) {
    static_assert(kPlanTiles == 256, "one tile per thread");
    __shared__ unsigned sWave[kPlanQ][4];
    __shared__ unsigned sBase[kTotCount];
    __shared__ unsigned long long sOrder[2];
    const int t = threadIdx.x, tile = blockIdx.x * kPlanTiles + t;
    if (blockIdx.x == 0) {
        // publish the draw's counters and clear the live ones
        for (int v = t; v < V.count; v += kPlanTiles) {
            ViewCounters& c = V.ctr[v];
            c.fans = shared_load(&c.fanLive);
            c.clipIn = c.clipLive;
            c.fanLive = 0u;
            c.clipLive = 0u;
        }
        if (t == 0) {
            ctr->status = shared_load(&ctr->live.status);
            ctr->bigCount = ctr->live.bigCount;
            ctr->clipMax = shared_load(&ctr->live.clipMax);
            ctr->assembled = shared_load(&ctr->live.fans);
            ctr->live.status = 0u;
            ctr->live.bigCount = 0u;
            ctr->live.clipMax = 0u;
            ctr->live.fans = 0u;
            ctr->live.left = 0u;
        }
    }
    uint2 c = make_uint2(0u, 0u);  // entries with ranks, others
    if (tile < n) {
        const unsigned long long both = shared_load(&cnt[tile]);
        c = make_uint2((unsigned)both, (unsigned)(both >> 32));
        cnt[tile] = 0ull;
    }
    const unsigned total = c.x + c.y;
    // the tile's class in the shading order, 4 where it is not shaded
    int cls = 4;
    if (q.orderA && tile < n && (V.count == 1 || V.desc[V.tileView[tile]].shade != 0))
        cls = total == 0u ? 3 : !q.orderByLength || total <= (unsigned)kRasterPass ? 2 : total <= 4u * kRasterPass ? 1 : 0;
    const TilePlan w = tile_plan(total, tile < n, cls, q.partShift);
    unsigned v[kPlanQ], sum[kPlanQ];
#pragma unroll
    for (int k = 0; k < kPlanQ; k++) v[k] = w.q[k];
    plan_scan(v, sWave, sum);
    // one lane per quantity, so that the atomics' round trips overlap
#pragma unroll
    for (int k = 0; k < kPlanQ; k++)
        if (t == k && k < kTotCount) sBase[k] = sum[k] ? atomicAdd(&ctr->tot[k], sum[k]) : 0u;
#pragma unroll
    for (int k = 0; k < 2; k++) {
        const unsigned s = sum[kTotCount + k];
        if (t == kTotCount + k)
            sOrder[k] = s ? atomicAdd(reinterpret_cast<unsigned long long*>(ctr->order) + k,
                                      ((unsigned long long)(s >> 16) << 32) | (s & 0xffffu))
                          : 0ull;
    }
    __syncthreads();
    if (tile >= n) return;
#pragma unroll
    for (int k = 0; k < kTotCount; k++) v[k] += sBase[k];
    const unsigned part = 1u << q.partShift;
    const unsigned st = v[kTotEntries], p = w.q[kTotLong] + w.q[kTotShort];
    start[tile] = st;
    cursor[tile] = st + c.x;  // the entries with ranks come first
    for (unsigned k = 0; k < p; k++) {
        const uint4 item = make_uint4((unsigned)tile, st + k * part, min(part, total - k * part),
                                      p > 1u ? v[kTotPartials] + k : 0xFFFFFFFFu);
        if (k < w.q[kTotLong]) {
            if (v[kTotLong] + k < q.itemCap) q.items[v[kTotLong] + k] = item;
        } else if (v[kTotShort] < q.itemCap) {
            q.items[q.itemCap - 1u - v[kTotShort]] = item;
        }
    }
    if (p > 1u) q.multiList[v[kTotMulti]] = (unsigned)tile;
    if (p == 0u) q.multiList[(unsigned)n - 1u - v[kTotEmpty]] = (unsigned)tile;
    if (cls < 4) {
        // a and b from the front, b and a from the back
        const unsigned at = (unsigned)(sOrder[cls >> 1] >> (32 * (cls & 1))) +
                            ((v[kTotCount + (cls >> 1)] >> (16 * (cls & 1))) & 0xffffu);
        (cls == 0 || cls == 3 ? q.orderA : q.orderB)[cls < 2 ? at : (unsigned)n - 1u - at] = (unsigned)tile;
    }
    q.tilePartial[tile] = p > 1u ? (int)v[kTotPartials] : -1;
}

}  // namespace dev
}  // namespace ifrit_hip
