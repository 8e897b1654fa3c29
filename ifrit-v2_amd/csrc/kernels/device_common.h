// Device helpers shared by the rasterizer kernels.
#pragma once
#include <hip/hip_runtime.h>

#include "../common/x86_fp.h"
#include "pipeline.h"

namespace ifrit_hip {
namespace dev {

constexpr float kClearDepth = 3.3961514e38f;  // bit pattern 0x7f7f7f7f (TileRasterWorker.cpp:40)
constexpr float kEps = 1e-8f;                  // TileRasterWorker.h:85

inline unsigned blocks(size_t n, unsigned b) { return (unsigned)((n + b - 1) / b); }

__device__ __forceinline__ TriRec load_rec(const TriRecs& R, unsigned slot) {
    TriRec r;
    r.q0 = R.q0[slot];
    r.q1 = R.q1[slot];
    r.q2 = R.q2[slot];
    r.f1 = R.f1[slot];
    r.f2 = R.f2[slot];
    r.f3 = R.f3[slot];
    return r;
}

// Edge coefficients of a TriRec: inside when fma(ey, y, ex * x) < -ez.
struct Edges {
    float x[3], y[3], z[3];
};

__device__ __forceinline__ Edges load_edges(const TriRec& r) {
    Edges E;
    E.x[0] = r.q0.x; E.y[0] = r.q0.y; E.z[0] = r.q0.z;
    E.x[1] = r.q0.w; E.y[1] = r.q1.x; E.z[1] = r.q1.y;
    E.x[2] = r.q1.z; E.y[2] = r.q1.w; E.z[2] = r.q2.x;
    return E;
}

__device__ __forceinline__ Edges load_edges(const TriRecs& R, unsigned slot) {
    const float4 a = R.q0[slot], b = R.q1[slot];
    const float c = R.q2[slot].x;
    Edges E;
    E.x[0] = a.x; E.y[0] = a.y; E.z[0] = a.z;
    E.x[1] = a.w; E.y[1] = b.x; E.z[1] = b.y;
    E.x[2] = b.z; E.y[2] = b.w; E.z[2] = c;
    return E;
}

__device__ __forceinline__ Edges edges_of(const float e[3][3]) {
    Edges E;
#pragma unroll
    for (int k = 0; k < 3; k++) {
        E.x[k] = e[k][0];
        E.y[k] = e[k][1];
        E.z[k] = e[k][2];
    }
    return E;
}

// Tile classification of the binner (TileRasterWorker.cpp:341-395, SIMD128
// form): 0 rejected, 1 partially covered, 2 fully covered.
__device__ __forceinline__ int tile_class(const Edges& E, int tx, int ty) {
    const float x0 = (float)tx * 16.0f, y0 = (float)ty * 16.0f;
    const float x1 = x0 + 16.0f, y1 = y0 + 16.0f;
    int ntr = 0, nta = 0;
#pragma unroll
    for (int k = 0; k < 3; k++) {
        const bool right = E.x[k] < 0.0f, down = E.y[k] < 0.0f;
        const float xr = right ? x1 : x0, yr = down ? y1 : y0;
        const float xa = right ? x0 : x1, ya = down ? y0 : y1;
        ntr += fmaf(E.x[k], xr, fmaf(E.y[k], yr, E.z[k])) < 0.0f;
        nta += fmaf(E.x[k], xa, fmaf(E.y[k], ya, E.z[k])) < 0.0f;
    }
    return ntr != 3 ? 0 : (nta == 3 ? 2 : 1);
}

// 4x4 block trivial reject / accept (TileRasterWorker.cpp:887-934): block
// corners chosen from the edge normals, test fma(ey, Y, ex * X) < -ez.
__device__ __forceinline__ void block_test(const Edges& E, float bMinX, float bMinY, int& trn, int& tan) {
    const float bMaxX = bMinX + 4.0f, bMaxY = bMinY + 4.0f;
    trn = 0;
    tan = 0;
#pragma unroll
    for (int k = 0; k < 3; k++) {
        const bool right = E.x[k] < 0.0f, down = E.y[k] < 0.0f;
        const float xr = right ? bMaxX : bMinX, yr = down ? bMaxY : bMinY;
        const float xa = right ? bMinX : bMaxX, ya = down ? bMinY : bMaxY;
        const float nz = ifx::neg(E.z[k]);
        trn += fmaf(E.y[k], yr, E.x[k] * xr) < nz;
        tan += fmaf(E.y[k], ya, E.x[k] * xa) < nz;
    }
}

// Pixel / sample coverage test (TileRasterWorker.cpp:1042-1066).
__device__ __forceinline__ bool inside(const Edges& E, float x, float y) {
    int n = 0;
#pragma unroll
    for (int k = 0; k < 3; k++) n += fmaf(E.y[k], y, E.x[k] * x) < ifx::neg(E.z[k]);
    return n == 3;
}

// Rejects the whole unit square [x, x+1] x [y, y+1] when an edge excludes
// the corner that minimises it.  Rounding is monotone, so no point of the
// square can pass inside() when this returns false.
__device__ __forceinline__ bool square_may_cover(const Edges& E, float x, float y) {
    bool ok = true;
#pragma unroll
    for (int k = 0; k < 3; k++) {
        const float cx = E.x[k] < 0.0f ? x + 1.0f : x;
        const float cy = E.y[k] < 0.0f ? y + 1.0f : y;
        ok = ok && (fmaf(E.y[k], cy, E.x[k] * cx) < ifx::neg(E.z[k]));
    }
    return ok;
}

// Depth expressions of the three proposal classes.
// SIMD256 path (TileRasterWorker.cpp:2758-2769), also used for MSAA samples.
__device__ __forceinline__ float depth256(const float4& F1, const float4& F2, const float4& F3, float x, float y) {
    const float b0 = fmaf(F1.x, x, fmaf(F1.y, y, F1.z));
    const float b1 = fmaf(F2.x, x, fmaf(F2.y, y, F2.z));
    const float b2 = fmaf(F3.x, x, fmaf(F3.y, y, F3.z));
    return fmaf(b0, F1.w, fmaf(b1, F2.w, b2 * F3.w));
}
// SIMD128 path (TileRasterWorker.cpp:2423-2434).
__device__ __forceinline__ float depth128(const float4& F1, const float4& F2, const float4& F3, float x, float y) {
    const float b0 = fmaf(F1.x, x, fmaf(F1.y, y, F1.z));
    const float b1 = fmaf(F2.x, x, fmaf(F2.y, y, F2.z));
    const float b2 = fmaf(F3.x, x, fmaf(F3.y, y, F3.z));
    return fmaf(b2, F3.w, fmaf(b0, F1.w, b1 * F2.w));
}
// Scalar path with DPPS dot products (TileRasterWorker.cpp:2261-2270).
__device__ __forceinline__ float depth_scalar(const float4& F1, const float4& F2, const float4& F3, float x, float y) {
    const float b0 = (x * F1.x + y * F1.y) + (1.0f * F1.z + 0.0f * F1.w);
    const float b1 = (x * F2.x + y * F2.y) + (1.0f * F2.z + 0.0f * F2.w);
    const float b2 = (x * F3.x + y * F3.y) + (1.0f * F3.z + 0.0f * F3.w);
    return (F1.w * b0 + F2.w * b1) + (F3.w * b2 + 0.0f);
}

// Tagging mode, tile- and block-accepted fragments (pixelShadingSIMD256Grouped,
// TileRasterWorker.cpp:2672-2684): the x term enters first, then y.
__device__ __forceinline__ float depth_grouped(const float4& F1, const float4& F2, const float4& F3, float x, float y) {
    const float b0 = fmaf(F1.y, y, fmaf(F1.x, x, F1.z));
    const float b1 = fmaf(F2.y, y, fmaf(F2.x, x, F2.z));
    const float b2 = fmaf(F3.y, y, fmaf(F3.x, x, F3.z));
    return fmaf(b0, F1.w, fmaf(b1, F2.w, b2 * F3.w));
}

// Order-preserving map of FP32 depth to uint32 (-0 and +0 compare equal, as
// they do under the CPU path's float comparison).
__device__ __forceinline__ unsigned order_key(float d) {
    unsigned u = __float_as_uint(d);
    if (u == 0x80000000u) u = 0u;
    return (u & 0x80000000u) ? ~u : (u | 0x80000000u);
}
__device__ __forceinline__ float order_key_inv(unsigned k) {
    return __uint_as_float((k & 0x80000000u) ? (k & 0x7fffffffu) : ~k);
}

// Fragment key for the depth test: lexicographic (depth, prim*4 + fan).
__device__ __forceinline__ unsigned long long frag_key(float d, unsigned tie) {
    return ((unsigned long long)order_key(d) << 32) | tie;
}

// A view at a uniform index, in the constant address space: no kernel that reads the
// table writes it, which the compiler cannot see of a plain pointer beside atomics and
// stores, so that it loads the matrix into every lane.
typedef const __attribute__((address_space(4))) ViewDesc UniformView;
__device__ __forceinline__ const UniformView& uniform_view(const ViewDesc* d) { return *(UniformView*)d; }
// Words at a uniform address that no kernel reading them writes, and entry i of a map
// of views (two bytes each; a word of it lies in the map's allocation, whose size is a
// multiple of four bytes).
__device__ __forceinline__ unsigned uniform_word(const unsigned* p) {
    return *(const __attribute__((address_space(4))) unsigned*)p;
}
__device__ __forceinline__ uint4 uniform_words(const uint4* p) {
    typedef unsigned Words __attribute__((ext_vector_type(4)));
    const Words w = *(const __attribute__((address_space(4))) Words*)p;
    return make_uint4(w.x, w.y, w.z, w.w);
}
__device__ __forceinline__ unsigned uniform_view_of(const unsigned short* map, unsigned i) {
    i = (unsigned)__builtin_amdgcn_readfirstlane((int)i);
    return (uniform_word(reinterpret_cast<const unsigned*>(map) + (i >> 1)) >> (16u * (i & 1u))) & 0xffffu;
}

__device__ __forceinline__ int lane_id() { return (int)(threadIdx.x & 63u); }

// Wave-aggregated counter increment: every active lane adds one to
// ctr[key] and receives a unique position; lanes sharing a key share one
// atomic.  The lanes are grouped by key with ballots first, so all groups'
// atomics go out as one instruction and the wave waits for memory once, or,
// with several increments issued before the first value is taken, once for
// all of them.  Must be called by the whole (converged) wave.
struct WaveInc {
    unsigned base, rank;
    int leader;
};
__device__ __forceinline__ WaveInc wave_inc_issue(unsigned* ctr, int key, bool active) {
    const int lane = lane_id();
    unsigned long long pending = __ballot(active);
    int leader = lane;
    unsigned rank = 0, size = 0;
    while (pending) {
        const int l = __ffsll((unsigned long long)pending) - 1;
        const int lk = __builtin_amdgcn_readlane(key, l);  // l is uniform
        const unsigned long long grp = __ballot(active && key == lk) & pending;
        if ((grp >> lane) & 1ull) {
            leader = l;
            rank = (unsigned)__popcll(grp & ((1ull << lane) - 1ull));
        }
        if (lane == l) size = (unsigned)__popcll(grp);
        pending &= ~grp;
    }
    WaveInc r{0u, rank, leader};
    if (active && leader == lane) r.base = atomicAdd(&ctr[key], size);
    return r;
}
__device__ __forceinline__ unsigned wave_inc_value(const WaveInc& r) { return __shfl(r.base, r.leader, 64) + r.rank; }
__device__ __forceinline__ unsigned wave_inc(unsigned* ctr, int key, bool active) {
    return wave_inc_value(wave_inc_issue(ctr, key, active));
}

// A tile rectangle from its packed form (x0 | y0 << 16, x1 | y1 << 16).
__device__ __forceinline__ int4 unpack_box(const uint2& e) {
    return make_int4((int)(e.x & 0xFFFFu), (int)(e.x >> 16), (int)(e.y & 0xFFFFu), (int)(e.y >> 16));
}

// Tile k of a rectangle of `cols` columns whose tiles number at most four.
__device__ __forceinline__ int few_col(int k, int cols) { return cols == 1 ? 0 : (cols == 2 ? k & 1 : k); }
__device__ __forceinline__ int few_row(int k, int cols) { return cols == 1 ? k : (cols == 2 ? k >> 1 : 0); }

// Where a triangle goes in the tiles: SCATTER = false counts it, true writes it
// through the tile's cursor.
template <bool SCATTER>
__device__ __forceinline__ void bin_tile(const Edges& E, int tx, int ty, unsigned tileBase, int tilesX, unsigned slot,
                                         const BinBufs& B, unsigned binCap) {
    const int c = tile_class(E, tx, ty);
    if (!c) return;
    const unsigned t = tileBase + (unsigned)(ty * tilesX + tx);
    if constexpr (!SCATTER) {
        atomicAdd(&B.cnt[2 * t + 1], 1u);
    } else {
        const unsigned at = atomicAdd(&B.cursor[t], 1u);
        if (at < binCap) B.list[at] = slot | (c == 2 ? 0x80000000u : 0u);
    }
}

// Bins one triangle per lane (b.x > b.z: none): a lane walks a rectangle of up
// to eight tiles by itself, the wave shares larger ones, one round trip for 64
// tiles (a clip fan next to the eye often spans the whole frame).  The whole
// wave must call it.
template <bool SCATTER>
__device__ __forceinline__ void bin_lanes(const Edges& E, int4 b, unsigned tileBase, int tilesX, unsigned slot,
                                         const BinBufs& B, unsigned binCap) {
    const int w = b.z - b.x + 1, area = b.x <= b.z ? w * (b.w - b.y + 1) : 0;
    if (area <= 8) {
        for (int q = 0; q < area; q++) bin_tile<SCATTER>(E, b.x + q % w, b.y + q / w, tileBase, tilesX, slot, B, binCap);
    }
    for (unsigned long long m = __ballot(area > 8); m; m &= m - 1ull) {
        const int l = __ffsll(m) - 1;
        auto rl = [l](int x) { return __builtin_amdgcn_readlane(x, l); };
        Edges F;
#pragma unroll
        for (int k = 0; k < 3; k++) {
            F.x[k] = __int_as_float(rl(__float_as_int(E.x[k])));
            F.y[k] = __int_as_float(rl(__float_as_int(E.y[k])));
            F.z[k] = __int_as_float(rl(__float_as_int(E.z[k])));
        }
        const int x0 = rl(b.x), y0 = rl(b.y), fw = rl(w), fa = rl(area);
        const unsigned fs = (unsigned)rl((int)slot);
        for (int q = lane_id(); q < fa; q += 64)
            bin_tile<SCATTER>(F, x0 + q % fw, y0 + q / fw, tileBase, tilesX, fs, B, binCap);
    }
}

// Deferred triangles: units of up to 256 tiles, kBigParts units per triangle in
// turn, so that a screen-sized one spreads over as many workgroups.
constexpr unsigned kBigParts = 32;
template <bool SCATTER>
__device__ __forceinline__ void bin_big(unsigned nbig, const Views& V, const TriRecs& recs, const BinBufs& B,
                                        unsigned binCap) {
    for (unsigned u = blockIdx.x; u < nbig * kBigParts; u += gridDim.x) {
        const uint4 g = B.big[u / kBigParts];
        const int4 b = unpack_box(make_uint2(g.y, g.z));
        const int w = b.z - b.x + 1, area = w * (b.w - b.y + 1);
        const int first = (int)(u % kBigParts) * 256;
        if (first >= area) continue;
        const ViewDesc& D = V.desc[g.w];
        const Edges E = load_edges(recs, g.x);
        for (int q = first + (int)threadIdx.x; q < area; q += (int)kBigParts * 256)
            bin_tile<SCATTER>(E, b.x + q % w, b.y + q / w, D.tileBase, D.tilesX, g.x, B, binCap);
    }
}

// Whether the tile plan's raster work fits its buffers, and its lists too.
__device__ __forceinline__ bool plan_items_fit(const DeviceCounters* ctr, const RasterQueue& q) {
    return ctr->tot[kTotLong] + ctr->tot[kTotShort] <= q.itemCap && ctr->tot[kTotPartials] <= q.partialCap;
}
__device__ __forceinline__ bool plan_fits(const DeviceCounters* ctr, const RasterQueue& q) {
    return ctr->tot[kTotEntries] <= q.binCap && plan_items_fit(ctr, q);
}

// Sum over a 256-thread workgroup (all threads must call it).
__device__ __forceinline__ unsigned long long block_sum256(unsigned long long v) {
    __shared__ unsigned long long part[4];
    for (int off = 32; off > 0; off >>= 1) v += __shfl_down(v, off, 64);
    if ((threadIdx.x & 63) == 0) part[threadIdx.x >> 6] = v;
    __syncthreads();
    const unsigned long long r = part[0] + part[1] + part[2] + part[3];
    __syncthreads();
    return r;
}

// Reduces the per-workgroup statistics of one frame into the counters and writes them
// to the host (pinned memory, visible once the stream is synchronized).  NT threads.
// Latency only; a launch of its own took 5 us at the end of every draw, and 15 us with
// 34 views whose counters one thread read in turn.
template <int NT>
__device__ __forceinline__ void finalize_block(const StatPartials& st, const Views& V, const DeviceCounters* ctr,
                                               HostCounters* out) {
    __shared__ unsigned long long red[NT / 64][4];
    __shared__ unsigned most[NT / 64];
    const int t = threadIdx.x;
    if (t < 8) out->tot[t] = ctr->tot[t];
    // what the tile plan (or the point and line kernels) left
    unsigned long long asmb = t == 0 ? ctr->assembled : 0ull, frag = 0, cov = 0, clip = 0;
    unsigned mx = t == 0 ? ctr->clipMax : 0u;
    if (t == 0) {
        out->status = ctr->status;
        out->bigCount = ctr->bigCount;
    }
    for (int i = t; i < V.count; i += NT) {
        const unsigned fans = V.ctr[i].fans;
        clip += fans;
        mx = max(mx, max(fans, V.ctr[i].clipIn));
    }
    if (t < kMadeSums) asmb += st.made[t * kMadeStride];
    // independent loads: a thread's share is in flight together
#pragma unroll 4
    for (int i = t; i < st.rasterBlocks; i += NT) {
        frag += st.rasterFrags[i];
        cov += st.rasterCovs[i];
    }
    for (int off = 32; off > 0; off >>= 1) {
        asmb += __shfl_down(asmb, off, 64);
        frag += __shfl_down(frag, off, 64);
        cov += __shfl_down(cov, off, 64);
        clip += __shfl_down(clip, off, 64);
        mx = max(mx, (unsigned)__shfl_down((int)mx, off, 64));
    }
    if ((t & 63) == 0) {
        red[t >> 6][0] = asmb;
        red[t >> 6][1] = frag;
        red[t >> 6][2] = cov;
        red[t >> 6][3] = clip;
        most[t >> 6] = mx;
    }
    __syncthreads();
    if (t < 4) {
        unsigned long long r = 0;
        for (int w = 0; w < NT / 64; w++) r += red[w][t];
        if (t == 0) out->assembled = r;
        if (t == 1) out->fragments = r;
        if (t == 2) out->coveredSamples = r;
        if (t == 3) out->clipCount = (unsigned)r;
    } else if (t == 4) {
        unsigned m = 0;
        for (int w = 0; w < NT / 64; w++) m = max(m, most[w]);
        out->clipMax = m;
    }
}

// Inclusive prefix sum over the 64 lanes of a wave with DPP moves: row
// shifts by 1, 2, 4 and 8 (a lane whose source lies outside its row of 16
// adds 0), then the last lane of rows 0 and 2 added to rows 1 and 3
// (row_bcast:15) and the last lane of row 1 to rows 2 and 3 (row_bcast:31).
template <class T>
__device__ __forceinline__ T wave_incl_scan(T v) {
    static_assert(sizeof(T) == 4, "32-bit values");
    v += (T)__builtin_amdgcn_update_dpp(0, (int)v, 0x111, 0xf, 0xf, false);
    v += (T)__builtin_amdgcn_update_dpp(0, (int)v, 0x112, 0xf, 0xf, false);
    v += (T)__builtin_amdgcn_update_dpp(0, (int)v, 0x114, 0xf, 0xf, false);
    v += (T)__builtin_amdgcn_update_dpp(0, (int)v, 0x118, 0xf, 0xf, false);
    v += (T)__builtin_amdgcn_update_dpp(0, (int)v, 0x142, 0xa, 0xf, false);
    v += (T)__builtin_amdgcn_update_dpp(0, (int)v, 0x143, 0xc, 0xf, false);
    return v;
}

}  // namespace dev
}  // namespace ifrit_hip
