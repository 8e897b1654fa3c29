// Tile binning on gfx950 (the reference's executeBinner,
// projects/softgraphics/src/engine/tileraster/TileRasterWorker.cpp:314-397):
// every assembled triangle is tested against the 16x16 tiles of its tile
// rectangle; a tile whose trivial-reject corner is inside all three edges
// receives the triangle, flagged as fully covered when the trivial-accept
// corner is inside too.
//
// The geometry and clip kernels counted the entries of every tile, triangles of
// up to four tiles and others apart.  Here the tile plan turns the counts into list
// ranges and raster work, and the scatter writes the contiguous per-tile
// lists: the place of a triangle of up to four tiles is the list's start plus
// the rank its count returned (no atomic, and its record is not read), the
// others follow them through a cursor per tile.  Lanes of a wave that hit the same tile
// share one atomic (wave_inc).  Triangles spanning more than bigThreshold
// tiles go through a workgroup each, so that a few screen-sized triangles do
// not serialise one lane.
#include <hip/hip_runtime.h>

#include "device_common.h"

namespace ifrit_hip {

namespace {

using dev::Edges;
using dev::load_edges;

// ---------------------------------------------------------------------------
// Raster planning over the tiles of all views, in one launch: each workgroup
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
        const unsigned x = dev::wave_incl_scan(v[k]);
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

__global__ void __launch_bounds__(kPlanTiles) k_plan(uint2* __restrict__ cnt, unsigned* __restrict__ start,
                                                     unsigned* __restrict__ cursor, int n, Views V, RasterQueue q,
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
            c.fans = c.fanLive;
            c.clipIn = c.clipLive;
            c.fanLive = 0u;
            c.clipLive = 0u;
        }
        if (t == 0) {
            ctr->status = ctr->live.status;
            ctr->bigCount = ctr->live.bigCount;
            ctr->clipMax = ctr->live.clipMax;
            ctr->assembled = ctr->live.fans;
            ctr->live.status = 0u;
            ctr->live.bigCount = 0u;
            ctr->live.clipMax = 0u;
            ctr->live.fans = 0u;
        }
    }
    uint2 c = make_uint2(0u, 0u);
    if (tile < n) {
        c = cnt[tile];
        cnt[tile] = make_uint2(0u, 0u);
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

// One geometry wave's entries as a scatter wave holds them.
struct Region {
    bool any;                  // uniform: there is one
    unsigned r;                // geometry wave over all views
    bool single, few, multi;   // the lane's kind of entry
    uint2 e;
    uint4 f;
};

template <class F>
__device__ __forceinline__ Region next_region(const WaveInfo& W, unsigned long long& pend, F&& bcast, unsigned r0,
                                              unsigned step, int lane, const BinBufs& B) {
    Region R{pend != 0ull, 0u, false, false, false, make_uint2(0u, 0u), make_uint4(0u, 0u, 0u, 0u)};
    if (!R.any) return R;
    const int l = __ffsll(pend) - 1;
    pend &= pend - 1ull;
    R.r = r0 + step * (unsigned)l;
    R.single = (bcast(W.single, l) >> lane) & 1ull;
    R.few = (bcast(W.few, l) >> lane) & 1ull;
    R.multi = (bcast(W.multi, l) >> lane) & 1ull;
    if (R.single || R.few || R.multi) R.e = B.entry[(size_t)R.r * 64 + lane];
    if (R.few) R.f = B.entry1[(size_t)R.r * 64 + lane];
    return R;
}

// Writes the tile lists.  A wave takes the 64 triangles of one geometry wave at
// a time (one lane each), `regions` geometry waves after another: one where
// that leaves enough waves to fill the chip, more in batches of many views,
// where most geometry waves lie outside the view and are skipped by their
// WaveInfo.  They lie a grid's waves apart: neighbours are seen or culled
// together, and waves that took 42 neighbours each ran for up to 148 us of 167
// (34 views; 140 us as it is).
//
// Bound by the latency of the entries, the list starts and the scattered stores.
__global__ void __launch_bounds__(256) k_scatter(BinParams P, Views V, TriRecs recs, BinBufs B, RasterQueue q,
                                                 DeviceCounters* ctr) {
    __shared__ unsigned sMade[4];
    const int lane = dev::lane_id();
    const unsigned gw = blockIdx.x * 4u + (threadIdx.x >> 6), G = gridDim.x * 4u;
    const unsigned R = (unsigned)V.count * V.waves, C = (unsigned)P.regions;
    unsigned made = 0;
    for (unsigned r0 = gw; r0 < R; r0 += G * C) {
        WaveInfo W{0ull, 0ull, 0ull, 0ull, 0u, 0u};
        if ((unsigned)lane < C && r0 + G * (unsigned)lane < R) W = B.waves[r0 + G * (unsigned)lane];
        made += W.made;
        unsigned long long pend = __ballot((W.single | W.few | W.multi) != 0ull);
        auto bcast = [](unsigned long long x, int l) {
            return ((unsigned long long)(unsigned)__builtin_amdgcn_readlane((int)(x >> 32), l) << 32) |
                   (unsigned)__builtin_amdgcn_readlane((int)x, l);
        };
        // the entries of the next geometry wave are read while the current one's are written
        Region N = next_region(W, pend, bcast, r0, G, lane, B);
        while (N.any) {
            const Region A = N;
            N = next_region(W, pend, bcast, r0, G, lane, B);
            const unsigned v = A.r / V.waves;
            const uint2 e = A.e;
            const uint4 f = A.f;
            const unsigned slot = v * V.slotsPerView + (A.r - v * V.waves) * 64u + (unsigned)lane;
            if (A.single) {
                const unsigned at = B.start[e.x & 0x7fffffffu] + e.y;
                if (at < P.binCap) B.list[at] = slot | (e.x & 0x80000000u);
            }
            if (__ballot(A.few) != 0ull) {
                const int tilesX = V.desc[v].tilesX;
                const int cols = (int)(f.w & 3u) + 1;
                const unsigned rank[4] = {e.y, f.x, f.y, f.z};
                unsigned st[4];
#pragma unroll
                for (int k = 0; k < 4; k++) {  // the list starts in one round trip
                    st[k] = 0u;
                    if ((f.w >> (8 + 2 * k)) & 3u)
                        st[k] = B.start[e.x + (unsigned)(dev::few_row(k, cols) * tilesX + dev::few_col(k, cols))];
                }
#pragma unroll
                for (int k = 0; k < 4; k++) {
                    const unsigned c = (f.w >> (8 + 2 * k)) & 3u, at = st[k] + rank[k];
                    if (c && at < P.binCap) B.list[at] = slot | (c == 2u ? 0x80000000u : 0u);
                }
            }
            if (__ballot(A.multi) != 0ull) {
                const ViewDesc& D = V.desc[v];
                Edges E = {};
                if (A.multi) E = load_edges(recs, slot);
                const int4 b = A.multi ? dev::unpack_box(e) : make_int4(1, 0, 0, 0);
                dev::bin_lanes<true>(E, b, D.tileBase, D.tilesX, slot, B, P.binCap);
            }
        }
    }
    // clip fans, one lane each: wave k takes view k / per, as few fans per wave as that many
    // waves allow (a large fan takes the whole wave)
    const unsigned per = max(1u, G / (unsigned)V.count);
    for (unsigned k = gw; k < per * (unsigned)V.count; k += G) {
        const unsigned v = k / per;
        const unsigned n = fan_extent(V.ctr[v].clipIn, V.ctr[v].fans, P.clipCap), each = min(64u, (n + per - 1u) / per);
        for (unsigned i0 = (k % per) * each; i0 < n; i0 += per * each) {
            const ViewDesc& D = V.desc[v];
            const unsigned i = i0 + (unsigned)lane, slot = D.slotBase + (unsigned)P.ntri + i;
            int4 b = make_int4(1, 0, 0, 0);
            Edges E = {};
            if ((unsigned)lane < each && i < n) b = dev::unpack_box(B.fanBox[(size_t)v * P.clipCap + i]);
            if (b.x <= b.z) E = load_edges(recs, slot);
            dev::bin_lanes<true>(E, b, D.tileBase, D.tilesX, slot, B, P.binCap);
        }
    }
    dev::bin_big<true>(min(ctr->bigCount, P.bigCap), V, recs, B, P.binCap);
    // the workgroup's assembled triangles, for the statistics
    made = dev::wave_incl_scan(made);
    if (lane == 63) sMade[threadIdx.x >> 6] = made;
    __syncthreads();
    if (threadIdx.x == 0) {
        atomicAdd(&B.made[(blockIdx.x % kMadeSums) * kMadeStride],
                  (unsigned long long)(sMade[0] + sMade[1] + sMade[2] + sMade[3]));
        if (blockIdx.x == 0) {
            // on a bin or work-list overflow nothing is rasterised (plan_fits) and nothing shaded, as the
            // record slots are those of earlier draws; the host grows the buffers and draws again
            if (!dev::plan_fits(ctr, q))
                for (int k = 0; k < 4; k++) ctr->order[k] = 0u;
            if (ctr->tot[kTotEntries] > q.binCap) atomicOr(&ctr->status, kStatusBinOverflow);
            if (!dev::plan_items_fit(ctr, q)) atomicOr(&ctr->status, kStatusRasterOverflow);
        }
    }
}

}  // namespace

void launch_bin(const BinParams& p, const Views& views, TriRecs recs, const BinBufs& bins, const RasterQueue& q,
                DeviceCounters* ctr, hipStream_t s) {
    hipLaunchKernelGGL(k_plan, dim3((p.tiles + kPlanTiles - 1) / kPlanTiles), dim3(kPlanTiles), 0, s,
                       reinterpret_cast<uint2*>(bins.cnt), bins.start, bins.cursor, p.tiles, views, q, ctr);
    hipLaunchKernelGGL(k_scatter, dim3(p.grid), dim3(256), 0, s, p, views, recs, bins, q, ctr);
}

}  // namespace ifrit_hip
