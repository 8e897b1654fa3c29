// Raster helpers shared by the raster and shading kernels: the view of a
// tile, per-pixel context, the class depth, and the ordered traversal of a
// tile's list (depth functions other than LESS, blending).
#pragma once
#include "device_common.h"

namespace ifrit_hip {
namespace rc {

using namespace dev;

// Depth expression codes of a 1-sample fragment, kept in the low bits of its
// key: 1 SIMD256, 2 SIMD128, 3 scalar DPPS, or in the tagging mode
// (optsetForceDeterministic(false), TileRasterWorker.cpp:1581-1675) 3 the
// grouped form.  The deterministic mode draws tile- and block-accepted and
// 4x2-group fragments with SIMD256, 2x2 quads with SIMD128 and single pixels
// with the scalar form; the tagging mode draws accepted fragments grouped,
// 4x2 groups with SIMD256, and quads and single pixels with SIMD128
// (pixelShadingSingleQuad, TileRasterWorker.cpp:2123-2165).
__device__ __forceinline__ float class_depth(unsigned c, const float4& F1, const float4& F2, const float4& F3, float x,
                                             float y, bool tagging = false) {
    if (c == 1) return depth256(F1, F2, F3, x, y);
    if (c == 2) return depth128(F1, F2, F3, x, y);
    return tagging ? depth_grouped(F1, F2, F3, x, y) : depth_scalar(F1, F2, F3, x, y);
}

// class_depth with every expression evaluated and the class's selected:
// SIMD256 and SIMD128 share their three plane values.
__device__ __forceinline__ float class_depth_all(unsigned c, const float4& F1, const float4& F2, const float4& F3,
                                                 float x, float y, bool tagging) {
    const float b0 = fmaf(F1.x, x, fmaf(F1.y, y, F1.z));
    const float b1 = fmaf(F2.x, x, fmaf(F2.y, y, F2.z));
    const float b2 = fmaf(F3.x, x, fmaf(F3.y, y, F3.z));
    const float d256 = fmaf(b0, F1.w, fmaf(b1, F2.w, b2 * F3.w));
    const float d128 = fmaf(b2, F3.w, fmaf(b0, F1.w, b1 * F2.w));
    const float d3 = tagging ? depth_grouped(F1, F2, F3, x, y) : depth_scalar(F1, F2, F3, x, y);
    return c == 1 ? d256 : (c == 2 ? d128 : d3);
}

// Expression code of a fragment from how it was covered: accepted (tile or
// 4x4 block), its 4x2 group all inside, its 2x2 quad all inside, or alone.
__device__ __forceinline__ unsigned expr_code(bool accepted, bool group, bool quad, bool tagging) {
    if (accepted) return tagging ? 3u : 1u;
    if (group) return 1u;
    return quad || tagging ? 2u : 3u;
}

// The class byte a pixel reports: the expression code, with the tagging
// mode's grouped form as 4.
__device__ __forceinline__ uint8_t class_out(unsigned c, bool tagging) {
    return (uint8_t)(tagging && c == 3u ? 4u : c);
}

// The view a tile belongs to: its size and where its outputs and slotOf
// entries start.
struct ViewGeom {
    int width, height, tilesX;
    int tile;  // view-local tile index
    size_t pixBase;
    unsigned primBase;
    unsigned slotBase;  // record slot of the view's triangle 0
    int view;
};

__device__ __forceinline__ ViewGeom view_of_tile(const Views& V, int gtile) {
    const unsigned view = uniform_view_of(V.tileView, (unsigned)gtile);
    const UniformView& D = uniform_view(V.desc + view);
    ViewGeom G;
    G.width = D.width;
    G.height = D.height;
    G.tilesX = D.tilesX;
    G.tile = gtile - (int)D.tileBase;
    G.pixBase = (size_t)D.pixBase;
    G.primBase = D.primBase;
    G.slotBase = D.slotBase;
    G.view = (int)view;
    return G;
}

// The rectangles are read from device memory at a uniform address (scalar
// loads), so that the test holds no vector registers.
__device__ __forceinline__ bool scissor_pass(const Scissor& sc, float x, float y) {
    if (sc.count == 0) return true;
    for (int i = 0; i < sc.count; i++) {
        const float4 r = sc.rects[i];
        if (x >= r.x && x <= r.x + r.z && y >= r.y && y <= r.y + r.w) return true;
    }
    return false;
}

// Every pixel of the rectangle [x0, x1] x [y0, y1] passes (one scissor holds it whole).
__device__ __forceinline__ bool scissor_all(const Scissor& sc, int x0, int y0, int x1, int y1) {
    if (sc.count == 0) return true;
    for (int i = 0; i < sc.count; i++) {
        const float4 r = sc.rects[i];
        if ((float)x0 >= r.x && (float)x1 <= r.x + r.z && (float)y0 >= r.y && (float)y1 <= r.y + r.w) return true;
    }
    return false;
}

struct PixelCtx {
    int tx, ty, px, py;
    bool inFb;
    size_t pix;
    float fpx, fpy, bMinX, bMinY;
};

__device__ __forceinline__ PixelCtx pixel_ctx(const ViewGeom& G, int lx, int ly) {
    PixelCtx C;
    C.tx = G.tile % G.tilesX;
    C.ty = G.tile / G.tilesX;
    C.px = C.tx * 16 + lx;
    C.py = C.ty * 16 + ly;
    C.inFb = C.px < G.width && C.py < G.height;
    C.pix = (size_t)C.py * G.width + C.px;
    C.fpx = (float)C.px;
    C.fpy = (float)C.py;
    C.bMinX = fmaf((float)(lx >> 2), 4.0f, (float)(C.tx * 16) * 1.0f);
    C.bMinY = fmaf((float)(ly >> 2), 4.0f, (float)(C.ty * 16) * 1.0f);
    return C;
}

// square_may_cover of the 16 unit squares of the 4x4 window at (x0, y0), bit
// 4 * row + column: the same products and fused sums per square (corners
// are small integers, so x0 + column + 1 is exact either way), with each
// edge's column products and row corners shared and no branches.
__device__ __forceinline__ unsigned block_square_mask(const Edges& E, float x0, float y0) {
    float ax[3][4], cy[3][4], nz[3];
#pragma unroll
    for (int k = 0; k < 3; k++) {
        const float ox = E.x[k] < 0.0f ? 1.0f : 0.0f, oy = E.y[k] < 0.0f ? 1.0f : 0.0f;
        nz[k] = ifx::neg(E.z[k]);
#pragma unroll
        for (int i = 0; i < 4; i++) {
            ax[k][i] = E.x[k] * ((x0 + (float)i) + ox);
            cy[k][i] = (y0 + (float)i) + oy;
        }
    }
    unsigned m = 0;
#pragma unroll
    for (int q = 15; q >= 0; q--) {  // bits shifted in from the last: no constant per bit
        const int i = q & 3, j = q >> 2;
        const unsigned c = (unsigned)(fmaf(E.y[0], cy[0][j], ax[0][i]) < nz[0]) &
                           (unsigned)(fmaf(E.y[1], cy[1][j], ax[1][i]) < nz[1]) &
                           (unsigned)(fmaf(E.y[2], cy[2][j], ax[2][i]) < nz[2]);
        m = m + m + c;
    }
    return m;
}

// The pixels of the 4x4 window at (x0, y0) that pass the pixel test at their
// corner (1 sample per pixel), bit 4 * row + column.
__device__ __forceinline__ unsigned window_inside(const Edges& E, float x0, float y0) {
    float ax[3][4], nz[3];
#pragma unroll
    for (int k = 0; k < 3; k++) {
        nz[k] = ifx::neg(E.z[k]);
#pragma unroll
        for (int i = 0; i < 4; i++) ax[k][i] = E.x[k] * (x0 + (float)i);
    }
    unsigned m = 0;
#pragma unroll
    for (int q = 15; q >= 0; q--) {  // as in blocks_not_rejected
        const float y = y0 + (float)(q >> 2);
        const unsigned c = (unsigned)(fmaf(E.y[0], y, ax[0][q & 3]) < nz[0]) &
                           (unsigned)(fmaf(E.y[1], y, ax[1][q & 3]) < nz[1]) &
                           (unsigned)(fmaf(E.y[2], y, ax[2][q & 3]) < nz[2]);
        m = m + m + c;
    }
    return m;
}

// 4x4 block trivial accept (block_test): the corner that maximises each edge is inside it.
__device__ __forceinline__ bool block_accepted(const Edges& E, float bMinX, float bMinY) {
    int trn, tan;
    block_test(E, bMinX, bMinY, trn, tan);
    return tan == 3;
}

// Of the covered pixels m of the 4x4 window at tile column ox and row oy, those
// whose 4x2 group (groups) and whose 2x2 quad (quads) is all covered.  A group or
// quad that reaches out of the window is not: a window off the blocks' grid
// holds every pixel its triangle can cover.
__device__ __forceinline__ void window_classes(unsigned m, int ox, int oy, unsigned& groups, unsigned& quads) {
    const unsigned rows = oy & 1 ? 0x00F0u : 0x0F0Fu;  // rows where a quad starts
    const unsigned h = m & (m >> 1);
    const unsigned q = h & (h >> 4) & rows & (ox & 1 ? 0x2222u : 0x5555u);
    quads = q | (q << 1) | (q << 4) | (q << 5);
    const unsigned r = (ox & 3) == 0 ? h & (h >> 2) & 0x1111u : 0u;  // full rows
    groups = (r & (r >> 4) & rows) * 0xFFu;
}

// Pixels of a 4x4 block inside the frame (bit 4 * row + column), given the
// frame's columns and rows left from the block's corner.
__device__ __forceinline__ unsigned block_fb_mask(int ncols, int nrows) {
    const unsigned c = ncols >= 4 ? 0xFu : (ncols <= 0 ? 0u : (1u << ncols) - 1u);
    const unsigned r = nrows >= 4 ? 0xFFFFu : (nrows <= 0 ? 0u : (1u << (4 * nrows)) - 1u);
    return (c * 0x1111u) & r;
}

// ---------------------------------------------------------------------------
// Ordered traversal.  A tile's list is sorted by (prim * 4 + fan, entry), the
// order of the reference's per-tile sort (TileRasterWorker.cpp:1225-1259);
// lists longer than the LDS buffer are taken in sorted windows of kOrderCap
// entries, each the smallest keys above the previous window.
// ---------------------------------------------------------------------------
constexpr int kOrderCap = 2048;

__device__ __forceinline__ bool depth_pass(int func, float d, float cur, bool scalarPath) {
    switch (func) {
        case 0: return false;                           // NEVER
        case 1: return !(d >= cur);                     // LESS
        case 2: return !(d != cur);                     // EQUAL
        case 3: return !(d > cur);                      // LESS_OR_EQUAL
        case 4: return scalarPath ? true : !(d <= cur); // GREATER
        case 5: return !(d == cur);                     // NOT_EQUAL
        case 6: return !(d < cur);                      // GREATER_OR_EQUAL
        default: return true;                           // ALWAYS
    }
}

// Expression code of a covered 1-sample pixel (class_depth): accepted, its
// 4x2 group all inside, its 2x2 quad all inside, or a single pixel.
template <int UNROLL = 8>
__device__ __forceinline__ unsigned pixel_class(const Edges& E, bool accepted, float fpx, float fpy, float bMinX,
                                                bool tagging) {
    if (accepted) return expr_code(true, false, false, tagging);
    const float gy = floorf(fpy * 0.5f) * 2.0f;
    bool g = true;
#pragma unroll UNROLL
    for (int l = 0; l < 8; l++) g = g && inside(E, bMinX + (float)(l & 3), gy + (float)(l >> 2));
    if (g) return 1u;
    const float qx = floorf(fpx * 0.5f) * 2.0f;
    bool q = true;
#pragma unroll UNROLL
    for (int l = 0; l < 4; l++) q = q && inside(E, qx + (float)(l & 1), gy + (float)(l >> 1));
    return expr_code(false, false, q, tagging);
}

// Ascending bitonic sort of n 64-bit keys in LDS (n a power of two).
__device__ __forceinline__ void bitonic_sort(unsigned long long* a, int n) {
    for (int k = 2; k <= n; k <<= 1)
        for (int j = k >> 1; j > 0; j >>= 1) {
            for (int i = threadIdx.x; i < n; i += 256) {
                const int l = i ^ j;
                if (l > i) {
                    const unsigned long long x = a[i], y = a[l];
                    if ((x > y) == ((i & k) == 0)) {
                        a[i] = y;
                        a[l] = x;
                    }
                }
            }
            __syncthreads();
        }
}

// Sorts a bitonic sequence of n keys ascending.
__device__ __forceinline__ void bitonic_merge(unsigned long long* a, int n) {
    for (int j = n >> 1; j > 0; j >>= 1) {
        for (int i = threadIdx.x; i < n; i += 256) {
            const int l = i ^ j;
            if (l > i) {
                const unsigned long long x = a[i], y = a[l];
                if (x > y) {
                    a[i] = y;
                    a[l] = x;
                }
            }
        }
        __syncthreads();
    }
}

// Ascending sort of n = 64 * 2^k keys (at most 256 * K) in a, with b as scratch; returns
// the one that holds the result.  Waves sort runs of 64 in registers; then pairs of
// runs are merged, every key finding its place by a search in the sibling run.  A
// thread's K keys go through each step together, as both are chains of LDS
// latencies.  With a bitonic sort in LDS, 55 barriers for 1024 keys, the blending
// draw of k_blend_ordered's figures took 71 us instead of 60.
template <int K>
__device__ __forceinline__ unsigned long long* merge_sort(unsigned long long* a, unsigned long long* b, int n) {
    const int lane = lane_id(), t = threadIdx.x;
    unsigned long long x[K];
#pragma unroll
    for (int q = 0; q < K; q++) x[q] = t + 256 * q < n ? a[t + 256 * q] : ~0ull;
#pragma unroll
    for (int k = 2; k <= 64; k <<= 1)
#pragma unroll
        for (int j = k >> 1; j > 0; j >>= 1) {
            const bool low = ((lane & j) == 0) == ((lane & k) == 0);
#pragma unroll
            for (int q = 0; q < K; q++) {
                const unsigned long long y = __shfl_xor(x[q], j, 64);
                x[q] = (y < x[q]) == low ? y : x[q];
            }
        }
    for (int run = 64;; run <<= 1) {
#pragma unroll
        for (int q = 0; q < K; q++)
            if (t + 256 * q < n) a[t + 256 * q] = x[q];
        __syncthreads();
        if (run >= n) return a;
        int lo[K];
#pragma unroll
        for (int q = 0; q < K; q++) lo[q] = 0;
        // keys of the sibling run below x; the first run's go first among equal ones (padding)
        for (int step = run; step > 0; step >>= 1)
#pragma unroll
            for (int q = 0; q < K; q++) {
                const int i = min(t + 256 * q, n - 1), at = lo[q] + step;
                const unsigned long long y = a[((i & ~(run - 1)) ^ run) + min(at, run) - 1];
                if (at <= run && (y < x[q] || ((i & run) && y == x[q]))) lo[q] = at;
            }
#pragma unroll
        for (int q = 0; q < K; q++) {
            const int i = t + 256 * q;
            if (i < n) b[(i & ~(2 * run - 1)) + (i & (run - 1)) + lo[q]] = x[q];
        }
        __syncthreads();
        unsigned long long* const c = a;
        a = b;
        b = c;
#pragma unroll
        for (int q = 0; q < K; q++) x[q] = t + 256 * q < n ? a[t + 256 * q] : ~0ull;
    }
}

// Sort key of a list entry: the record's primitive key, then the entry.  Triangle p
// that was not clipped sits in slot slotBase + p; only a fan's key is read.
__device__ __forceinline__ unsigned long long order_entry_key(const TriRecs& recs, unsigned ent, unsigned slotBase,
                                                              unsigned ntri) {
    const unsigned slot = ent & 0x7fffffffu, p = slot - slotBase;
    const unsigned key = p < ntri ? p * 4u : __float_as_uint(recs.q2[slot].y);
    return ((unsigned long long)key << 32) | ent;
}

// A workgroup's four waves take the four 8x8 quarters of its tile, so that a
// wave's pixels lie together: lane l holds pixel (l & 7, l >> 3) of quarter w.
__device__ __forceinline__ int quarter_x(int t) { return ((t >> 6) & 1) * 8 + (t & 7); }
__device__ __forceinline__ int quarter_y(int t) { return (t >> 7) * 8 + ((t >> 3) & 7); }

// Coverage of the wave's pixels by one triangle at 1 sample, and the lane's
// expression code: every lane tests its own pixel, and the ballot tells whether
// its 2x2 quad, 4x2 group and 4x4 block are all inside.  A block's accept implies
// that all its pixels are inside and its reject that none is (rounding is
// monotone), so the corner test of the accept runs only where a block is full.
__device__ __forceinline__ bool wave_covers(const Edges& E, const PixelCtx& C, bool tagging, unsigned& cls) {
    const bool in = inside(E, C.fpx, C.fpy);
    const unsigned long long b = __ballot(in);
    const int l = lane_id();
    const bool quad = ((b >> (l & 0x36)) & 0x0303ull) == 0x0303ull;
    const bool group = ((b >> (l & 0x34)) & 0x0F0Full) == 0x0F0Full;
    bool accepted = false;
    const bool block = ((b >> (l & 0x24)) & 0x0F0F0F0Full) == 0x0F0F0F0Full;
    if (__ballot(block) != 0ull) {
        int trn, tan;
        block_test(E, C.bMinX, C.bMinY, trn, tan);
        accepted = tan == 3;
    }
    cls = expr_code(accepted, group, quad, tagging);
    return in;
}

// A value all lanes hold, in scalar registers.
__device__ __forceinline__ unsigned long long uniform64(unsigned long long v) {
    return ((unsigned long long)(unsigned)__builtin_amdgcn_readfirstlane((int)(v >> 32)) << 32) |
           (unsigned)__builtin_amdgcn_readfirstlane((int)v);
}

constexpr int kOrderWords = 2, kOrderChunk = 64 * kOrderWords;  // records covered at a time

struct OrderLds {
    unsigned long long key[kOrderCap];
    // the chunk's records, and per tile pixel and record (a bit each) bits 0 and 1 of the code it is
    // covered with; sorting a list longer than kOrderCap has its second run here
    TriRec rec[kOrderChunk];
    unsigned long long code0[kOrderWords][256], code1[kOrderWords][256];
    unsigned long long full[kOrderWords];          // records that cover the tile
    unsigned long long big[2][kOrderWords];        // records of many windows, for the tile's upper and lower half
};
static_assert(offsetof(OrderLds, full) - offsetof(OrderLds, rec) >= sizeof(unsigned long long) * kOrderCap, "sort run");

// The tiles of an ordered draw, taken by the workgroups as they come free: the tile
// plan's lists of more than one part, its items from the longest class on, then
// the empty tiles.  In tile order the workgroups that met several long lists, or a
// long one late, held the draw (60 us instead of 50 for that draw).
struct OrderedTiles {
    static constexpr unsigned kEmpties = 4;  // empty tiles per claim: a few stores each
    unsigned multi, longs, items, empties, total;
    unsigned empty, emptyEnd;  // the claimed ones that are left
    unsigned stream, claimed;
    __attribute__((address_space(1))) unsigned* head;

    // as the key raster's: thread 0 claims an item ahead, through an address in vector registers
    __device__ __forceinline__ OrderedTiles(const RasterQueue& q, DeviceCounters* ctr, bool on = true)
        : empty(0), emptyEnd(0), claimed(0) {
        const bool fits = plan_fits(ctr, q);
        multi = fits ? ctr->tot[kTotMulti] : 0u;
        longs = ctr->tot[kTotLong];
        items = fits ? longs + ctr->tot[kTotShort] : 0u;
        empties = fits ? ctr->tot[kTotEmpty] : 0u;
        total = multi + items + (empties + kEmpties - 1u) / kEmpties;
        stream = blockIdx.x % kItemStreams;
        head = (__attribute__((address_space(1))) unsigned*)&ctr->itemHeads[stream][0];
        asm volatile("" : "+v"(head));
        if (on) claim();
    }
    __device__ __forceinline__ void claim() {
        if (threadIdx.x == 0) claimed = __hip_atomic_fetch_add(head, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    // The next tile and its list, or false; every thread must call it, with a word of LDS.
    __device__ __forceinline__ bool next(const RasterQueue& q, const BinBufs& B, int tiles, unsigned* sItem, int& tile,
                                         unsigned& start, unsigned& cnt) {
        start = cnt = 0u;
        for (;;) {
            if (empty < emptyEnd) {
                tile = (int)q.multiList[(unsigned)tiles - 1u - empty++];
                return true;
            }
            if (threadIdx.x == 0) *sItem = claimed;
            __syncthreads();
            unsigned k = (unsigned)__builtin_amdgcn_readfirstlane((int)*sItem) * kItemStreams + stream;
            __syncthreads();
            if (k >= total) return false;
            claim();
            if (k < multi) {
                tile = (int)q.multiList[k];
                start = B.start[tile];
                cnt = B.cursor[tile] - start;
                return true;
            }
            k -= multi;
            if (k >= items) {
                empty = (k - items) * kEmpties;
                emptyEnd = min(empty + kEmpties, empties);
                continue;
            }
            const uint4 it = q.items[k < longs ? k : q.itemCap - 1u - (k - longs)];
            if (it.w != 0xFFFFFFFFu) continue;  // a part of a list taken above
            tile = (int)it.x;
            start = it.y;
            cnt = it.z;
            return true;
        }
    }
};

// Calls visit(record, slot, code) in every thread for the entries of a tile's
// list that can cover the thread's pixel, in sorted order.  At 1 sample they do
// cover it and code is the expression code; else code is 3 for a record that
// covers the tile and 1 for one whose samples visit has to test.  256 threads,
// all must call it; thread t has pixel C = (quarter_x(t), quarter_y(t)).
//
// A chunk's records are covered by one lane each per half of the tile, which
// sets the record's bit at the pixels of its windows (as in the key raster), or by
// the waves over their quarters where a triangle has more than four windows;
// then every thread walks the bits of its own pixel.  A wave that took one record of a
// few pixels after the other was a serial chain: tiles of 800 entries held the draw
// (306 us instead of 72 for the draw of k_blend_ordered's figures).
template <int S, class F>
__device__ __forceinline__ void for_each_ordered(const TriRecs& recs, const unsigned* __restrict__ binList,
                                                 unsigned start, unsigned cnt, unsigned slotBase, unsigned ntri,
                                                 const PixelCtx& C, bool tagging, OrderLds& L, F&& visit) {
    const int t = threadIdx.x, w = t >> 6;
    const int tx0 = C.tx * 16, ty0 = C.ty * 16;
    const int pixel = quarter_y(t) * 16 + quarter_x(t);
    unsigned long long* const sA = L.key;
    unsigned long long* const sB = reinterpret_cast<unsigned long long*>(L.rec);
    unsigned long long last = 0;
    bool haveLast = false;
    while (cnt > 0u) {
        // the window: the (up to) kOrderCap smallest keys above `last`, sorted in sA
        int m;
        if (cnt <= (unsigned)kOrderCap) {
            int n2 = 64;
            while (n2 < (int)cnt) n2 <<= 1;
            for (int i = t; i < n2; i += 256)
                sA[i] = i < (int)cnt ? order_entry_key(recs, binList[start + i], slotBase, ntri) : ~0ull;
            __syncthreads();
            const unsigned long long* const sorted =
                n2 <= 256 ? merge_sort<1>(sA, sB, n2) : n2 <= 1024 ? merge_sort<4>(sA, sB, n2) : merge_sort<8>(sA, sB, n2);
            if (sorted != sA) {  // the records go over the scratch
                for (int i = t; i < n2; i += 256) sA[i] = sorted[i];
                __syncthreads();
            }
            m = (int)cnt;
        } else {
            for (int i = t; i < kOrderCap; i += 256) sA[i] = ~0ull;
            for (unsigned b0 = 0; b0 < cnt; b0 += kOrderCap) {
                for (int i = t; i < kOrderCap; i += 256) {
                    unsigned long long k = ~0ull;
                    if (b0 + i < cnt) {
                        k = order_entry_key(recs, binList[start + b0 + i], slotBase, ntri);
                        if (haveLast && k <= last) k = ~0ull;
                    }
                    sB[i] = k;
                }
                __syncthreads();
                bitonic_sort(sB, kOrderCap);
                // the lower halves of two sorted runs form a bitonic sequence
                for (int i = t; i < kOrderCap; i += 256) sA[i] = min(sA[i], sB[kOrderCap - 1 - i]);
                __syncthreads();
                bitonic_merge(sA, kOrderCap);
            }
            // entries of the window: the keys below ~0 (sorted, so a count)
            unsigned mine = 0;
            for (int i = t; i < kOrderCap; i += 256) mine += sA[i] != ~0ull;
            m = (int)block_sum256((unsigned long long)mine);
        }
        // thread t holds half of record t & 127: the next chunk's are loaded during the current one
        const int r = t & (kOrderChunk - 1), half = t >> 7;
        float4 a = make_float4(0, 0, 0, 0), b = a, c = a;
        auto load = [&](int c0) {
            if (c0 + r < m) {
                const unsigned slot = (unsigned)sA[c0 + r] & 0x7fffffffu;
                a = (half ? recs.f1 : recs.q0)[slot];
                b = (half ? recs.f2 : recs.q1)[slot];
                c = (half ? recs.f3 : recs.q2)[slot];
            }
        };
        load(0);
        for (int c0 = 0; c0 < m; c0 += kOrderChunk) {
            __syncthreads();  // the previous chunk has been visited
            if (half) {
                L.rec[r].f1 = a;
                L.rec[r].f2 = b;
                L.rec[r].f3 = c;
            } else {
                L.rec[r].q0 = a;
                L.rec[r].q1 = b;
                L.rec[r].q2 = c;
            }
#pragma unroll
            for (int k = 0; k < kOrderWords; k++) L.code0[k][t] = L.code1[k][t] = 0ull;
            __syncthreads();
            load(c0 + kOrderChunk);
            bool full = false, big = false;
            if (c0 + r < m) {
                full = ((unsigned)sA[c0 + r] >> 31) != 0u;
                const unsigned lo = __float_as_uint(L.rec[r].q2.z), hi = __float_as_uint(L.rec[r].q2.w);
                // the pixel box within the tile's half
                const int x0 = max((int)(lo & 0xFFFFu) - tx0, 0), y0 = max((int)(lo >> 16) - ty0, 8 * half);
                const int x1 = min((int)(hi & 0xFFFFu) - tx0, 15), y1 = min((int)(hi >> 16) - ty0, 8 * half + 7);
                if (!full && x0 <= x1 && y0 <= y1) {
                    // one window, on the blocks' grid or off it: off it, every block lacks a pixel
                    const bool one = x1 - x0 < 4 && y1 - y0 < 4;
                    const int gx = one ? x0 : x0 & ~3, gy = one ? y0 : y0 & ~3;
                    const int wcols = (x1 - gx + 4) >> 2, n = wcols * ((y1 - gy + 4) >> 2);
                    big = n > 4;
                    if (!big) {
                        const Edges E = load_edges(L.rec[r]);
                        const unsigned long long bit = 1ull << (r & 63);
                        for (int k = 0; k < n; k++) {
                            const int wx = gx + 4 * few_col(k, wcols), wy = gy + 4 * few_row(k, wcols);
                            const float fx = (float)(tx0 + wx), fy = (float)(ty0 + wy);
                            unsigned pm = block_fb_mask(x1 + 1 - wx, y1 + 1 - wy), groups = 0, quads = 0;
                            bool acc = false;
                            if constexpr (S == 1) {
                                if (((wx | wy) & 3) == 0) acc = block_accepted(E, fx, fy);
                                const unsigned in = window_inside(E, fx, fy);
                                window_classes(in, wx, wy, groups, quads);
                                pm &= in;
                            } else {
                                pm &= block_square_mask(E, fx, fy);
                            }
                            while (pm) {
                                const int i = __ffs(pm) - 1;
                                pm &= pm - 1u;
                                const int p = (wy + (i >> 2)) * 16 + wx + (i & 3);
                                const unsigned code =
                                    S == 1 ? expr_code(acc, (groups >> i) & 1u, (quads >> i) & 1u, tagging) : 1u;
                                if (code & 1u) atomicOr(&L.code0[r >> 6][p], bit);
                                if (code & 2u) atomicOr(&L.code1[r >> 6][p], bit);
                            }
                        }
                    }
                }
            }
            const unsigned long long fulls = __ballot(full), bigs = __ballot(big);
            if ((t & 63) == 0) {
                if (half == 0) L.full[r >> 6] = fulls;
                L.big[half][r >> 6] = bigs;
            }
            __syncthreads();
            unsigned long long code0[kOrderWords], code1[kOrderWords];
            const unsigned long long tag = tagging || S > 1 ? ~0ull : 0ull;
#pragma unroll
            for (int k = 0; k < kOrderWords; k++) {
                code0[k] = L.code0[k][pixel] | L.full[k];
                code1[k] = L.code1[k][pixel] | (L.full[k] & tag);
                for (unsigned long long mask = uniform64(L.big[w >> 1][k]); mask; mask &= mask - 1ull) {
                    const int i = __ffsll(mask) - 1;
                    const Edges E = load_edges(L.rec[64 * k + i]);
                    unsigned code = 1u;
                    const bool in = S == 1 ? wave_covers(E, C, tagging, code) : square_may_cover(E, C.fpx, C.fpy);
                    code = in ? code : 0u;
                    code0[k] |= (unsigned long long)(code & 1u) << i;
                    code1[k] |= (unsigned long long)(code >> 1) << i;
                }
            }
            // the pixel's own entries in order
            for (;;) {
                const unsigned long long first = code0[0] | code1[0];
                const bool lower = first != 0ull;
                const unsigned long long left = lower ? first : code0[1] | code1[1];
                if (!left) break;
                const int i = __ffsll(left) - 1;
                const unsigned long long bit = 1ull << i;
                const unsigned code = ((lower ? code0[0] : code0[1]) & bit ? 1u : 0u) |
                                      ((lower ? code1[0] : code1[1]) & bit ? 2u : 0u);
                const unsigned long long drop0 = lower ? bit : 0ull, drop1 = lower ? 0ull : bit;
                code0[0] &= ~drop0;
                code1[0] &= ~drop0;
                code0[1] &= ~drop1;
                code1[1] &= ~drop1;
                const int q = (lower ? 0 : 64) + i;
                visit(L.rec[q], (unsigned)sA[c0 + q] & 0x7fffffffu, code);
            }
        }
        const bool done = cnt <= (unsigned)kOrderCap || m < kOrderCap;
        if (!done) last = sA[kOrderCap - 1];
        __syncthreads();  // the keys and records are reloaded by the next window or tile
        if (done) break;
        haveLast = true;
    }
}

}  // namespace rc
}  // namespace ifrit_hip
