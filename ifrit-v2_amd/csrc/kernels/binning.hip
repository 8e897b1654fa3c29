// Tile binning on gfx950 (the reference's executeBinner,
// projects/softgraphics/src/engine/tileraster/TileRasterWorker.cpp:314-397):
// every assembled triangle is tested against the 16x16 tiles of its tile
// rectangle; a tile whose trivial-reject corner is inside all three edges
// receives the triangle, flagged as fully covered when the trivial-accept
// corner is inside too.
//
// The geometry and clip kernels counted the entries of every tile, triangles of
// up to four tiles and others apart, and the tile plan turned the counts into list
// ranges and raster work.  Here the scatter writes the contiguous per-tile
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
                                                 StatPartials st, DeviceCounters* ctr) {
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
        const unsigned n = min(V.ctr[v].fans, P.clipCap), each = min(64u, (n + per - 1u) / per);
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
    dev::bin_big<true>(min(ctr->bigCount, P.bigCap), V, recs, B, P.binCap, blockIdx.x, gridDim.x);
    // the workgroup's assembled triangles, for the statistics
    made = dev::wave_incl_scan(made);
    if (lane == 63) sMade[threadIdx.x >> 6] = made;
    __syncthreads();
    if (threadIdx.x == 0) {
        atomicAdd(&B.made[(blockIdx.x % kMadeSums) * kMadeStride],
                  (unsigned long long)(sMade[0] + sMade[1] + sMade[2] + sMade[3]));
        if (blockIdx.x == 0) {
            // on a bin or work-list overflow nothing is rasterised (plan_fits); the host grows the
            // buffers and draws again
            if (ctr->tot[kTotEntries] > q.binCap) atomicOr(&ctr->status, kStatusBinOverflow);
            if (!dev::plan_items_fit(ctr, q)) atomicOr(&ctr->status, kStatusRasterOverflow);
        }
    }
}

}  // namespace

void launch_bin(const BinParams& p, const Views& views, TriRecs recs, const BinBufs& bins, const RasterQueue& q,
                StatPartials st, DeviceCounters* ctr, hipStream_t s) {
    hipLaunchKernelGGL(k_scatter, dim3(p.grid), dim3(256), 0, s, p, views, recs, bins, q, st, ctr);
}

}  // namespace ifrit_hip
