// Fine raster and early Z on gfx950.
//
// Coverage follows the reference's hierarchy exactly
// (projects/softgraphics/src/engine/tileraster/TileRasterWorker.cpp:787-1223,
// "TRW"): fully covered tiles from the binner, then 4x4 blocks by trivial
// reject / accept, then 4x2 groups, 2x2 quads and single pixels at 1 sample
// per pixel, each class with its own depth expression (TRW:2244-2918).  With
// MSAA every sample of a partially covered block is tested individually.
//
// Depth test.  The reference shades a tile's fragments in primitive order and
// keeps a fragment when !(depth >= stored) (TRW:2286-2290, 2482-2486,
// 2828-2832).  For finite depths the survivor is the lexicographic minimum of
// (depth, prim * 4 + fan), which is order-independent: visibility is held as
// 64-bit keys (ordered depth << 32 | prim * 4 + fan) merged with atomic min.
//
// Work expansion.  One lane per list entry lists the entry's 4x4 windows: those
// that its pixel box (the record's proven bound) covers where they are at most
// four, wherever they start, else the tile's blocks that pass trivial reject.
// One lane per (entry, window) then finds the window's pixels: at 1 sample the
// covered ones, each with its coverage class, with MSAA those whose unit square
// the triangle may cover (a monotone corner bound of the sample test, exact).
// Workgroup scans turn both into flat lists in LDS, and every lane takes one
// (entry, pixel) unit: its sample tests, depths and LDS atomic-min merges.
// Lanes stay busy whatever the mix of triangle sizes, which one-triangle-per-
// lane loops do not achieve, and a triangle of a few pixels costs one window.
//
// Block reject and, with MSAA, block accept decide nothing that the sample test
// does not: a block's corner minimises (maximises) every edge over it and
// rounding is monotone, so a rejected block has no covered sample and an
// accepted one no other.  Only the binner's whole-tile accept (another
// expression) and, at 1 sample, the class of an accepted block do.
//
// Scheduling.  A tile's list is cut into parts of at most 1 << partShift entries and
// all parts form one work queue that a persistent grid drains, so a few
// tiles holding thousands of sub-pixel triangles do not serialise on one
// compute unit.  A part goes through LDS in passes, all
// merging into the tile's keys.  Each part rasterises into LDS; a tile with one part writes
// its outputs from LDS, each part of a longer list stores its LDS keys to a
// private partial block and a second kernel takes the minimum over the parts
// and writes the outputs (it also clears tiles with an empty list).  No
// workgroup waits on another and no device-scope fence is issued (on the
// multi-XCD MI355X each one writes back an L2).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <type_traits>

#include "raster_common.h"

namespace ifrit_hip {

namespace {

using namespace dev;
using namespace rc;

// inside() with the three edge results combined by bitwise and: the same
// arithmetic, and the compiler keeps the sample loop free of branches.
__device__ __forceinline__ bool inside_and(const Edges& E, float x, float y) {
    const bool a = fmaf(E.y[0], y, E.x[0] * x) < ifx::neg(E.z[0]);
    const bool b = fmaf(E.y[1], y, E.x[1] * x) < ifx::neg(E.z[1]);
    const bool c = fmaf(E.y[2], y, E.x[2] * x) < ifx::neg(E.z[2]);
    return a & b & c;
}

// Exclusive scan over an NT-thread workgroup (64 or 256); every thread must call it.
template <int NT>
__device__ __forceinline__ unsigned scan_nt(int t, unsigned v, unsigned* sWave, unsigned& total) {
    const int lane = t & 63, w = t >> 6;
    const unsigned x = wave_incl_scan(v);
    if constexpr (NT == 64) {
        total = __shfl(x, 63, 64);
        return x - v;
    } else {
        if (lane == 63) sWave[w] = x;
        __syncthreads();
        unsigned base = 0;
#pragma unroll
        for (int i = 0; i < NT / 64; i++) base += i < w ? sWave[i] : 0u;
        total = 0;
#pragma unroll
        for (int i = 0; i < NT / 64; i++) total += sWave[i];
        return base + x - v;
    }
}

// Sum over an NT-thread workgroup (all threads must call it).
template <int NT>
__device__ __forceinline__ unsigned long long sum_nt(unsigned long long v) {
    if constexpr (NT == 64) {
        for (int off = 32; off > 0; off >>= 1) v += __shfl_down(v, off, 64);
        return v;
    } else {
        return block_sum256(v);
    }
}

// The tile's 4x4 blocks (bit 4 * row + column) that pass trivial reject: the
// corner that minimises an edge is inside it, for all three edges.
__device__ __forceinline__ unsigned blocks_not_rejected(const Edges& E, int tx0, int ty0) {
    float ax[3][4], cy[3][4], nz[3];
#pragma unroll
    for (int k = 0; k < 3; k++) {
        const float ox = E.x[k] < 0.0f ? 4.0f : 0.0f, oy = E.y[k] < 0.0f ? 4.0f : 0.0f;
        nz[k] = ifx::neg(E.z[k]);
#pragma unroll
        for (int i = 0; i < 4; i++) {
            ax[k][i] = E.x[k] * ((float)(tx0 + 4 * i) + ox);
            cy[k][i] = (float)(ty0 + 4 * i) + oy;
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

// Coverage class and depth of the winning triangle at a 1-sample pixel,
// recomputed with the same decisions as the raster phases.
__device__ __forceinline__ unsigned winner_class(const TriRec& R, int tx, int ty, float fpx, float fpy, float bMinX,
                                                 float bMinY, float& d, bool tagging) {
    const Edges E = load_edges(R);
    bool accepted = tile_class(E, tx, ty) == 2;
    if (!accepted) {
        int trn, tan;
        block_test(E, bMinX, bMinY, trn, tan);
        accepted = tan == 3;
    }
    const unsigned c = pixel_class<1>(E, accepted, fpx, fpy, bMinX, tagging);  // rare: few registers, not speed
    d = class_depth(c, R.f1, R.f2, R.f3, fpx, fpy, tagging);
    return c;
}

// Fragment keys: the order key of the depth in the high word; in the low
// word the primitive key prim * 4 + fan (S > 1), or that key times 4 plus
// the fragment's coverage class at 1 sample per pixel (a pixel never holds
// two fragments of one (prim, fan), so the class bits never decide a
// minimum; primitives stay below 2^28 there).
template <int S>
__device__ __forceinline__ unsigned key_tie(unsigned long long k) {
    return S == 1 ? (unsigned)k >> 2 : (unsigned)k;
}

// Keys of the other depth functions whose result is a minimum too, whatever the
// order of the fragments (cleared draws): LESS_OR_EQUAL keeps the nearest and
// among equal depths the last fragment, GREATER and GREATER_OR_EQUAL the
// farthest, first or last, ALWAYS the last.  The depth's order is inverted by
// keyXor and ignored by keyMask 0; `last` inverts the low word's, whose value is
// then at least 1 (S == 1: the class bits; else the primitive key + 1), so that
// no fragment meets the clear value's low word.
template <int S>
__device__ __forceinline__ unsigned long long general_key(const RasterParams& P, float d, unsigned tie) {
    const unsigned hi = (order_key(d) ^ P.keyXor) & P.keyMask;
    const unsigned lo = P.last ? ~(tie + (S > 1 ? 1u : 0u)) : tie;
    return ((unsigned long long)hi << 32) | lo;
}
__device__ __forceinline__ unsigned long long general_clear_key(const RasterParams& P) {
    return ((unsigned long long)((order_key(P.clearDepth) ^ P.keyXor) & P.keyMask) << 32) | (P.last ? ~0u : 0u);
}
// A LESS key of the same fragment, for the output stage; ALWAYS keys, which hold no
// depth, take the depth of +-0, whose value the output stage reads from the record.
template <int S>
__device__ __forceinline__ unsigned long long less_key(const RasterParams& P, unsigned long long k) {
    const unsigned hi = P.keyMask ? (unsigned)(k >> 32) ^ P.keyXor : 0x80000000u;
    const unsigned lo = P.last ? ~(unsigned)k - (S > 1 ? 1u : 0u) : (unsigned)k;
    return ((unsigned long long)hi << 32) | lo;
}

// The record slot of a key's triangle: the geometry kernel puts triangle p in
// slot base + p, and only the triangles that crossed w = 0 (a bit per triangle
// in the geometry waves' WaveInfo) have their fans from slot ptr[p] on.
struct SlotMap {
    const unsigned* ptr;
    const WaveInfo* waves;
    unsigned base;
    bool clips;  // the view has such triangles
};

// Record slots of a pixel's S final keys, all S lookups issued before the first
// is used; a key that holds no fragment (its bit of `won` is 0) looks up
// primitive 0 and its slot is not used.
template <int S>
__device__ __forceinline__ void key_slots(const SlotMap& slotOf, const unsigned long long* keys,
                                          unsigned won, unsigned* slots) {
#pragma unroll
    for (int s = 0; s < S; s++) slots[s] = slotOf.base + (key_tie<S>(keys[s]) >> 2);
    if (!slotOf.clips) return;
    unsigned long long m[S];
#pragma unroll
    for (int s = 0; s < S; s++) {
        const unsigned prim = (won >> s) & 1u ? key_tie<S>(keys[s]) >> 2 : 0u;
        m[s] = slotOf.waves[prim >> 6].clipped >> (prim & 63u);
    }
#pragma unroll
    for (int s = 0; s < S; s++) {
        const unsigned tie = key_tie<S>(keys[s]);
        if (((won >> s) & 1u) && (m[s] & 1ull)) slots[s] = slotOf.ptr[tie >> 2] + (tie & 3u);
    }
}

// Writes the outputs of one pixel of a draw without clear from its S final keys:
// depth and record slot per sample where a fragment won (the primitive ID is the
// slot's key >> 2, expanded only on readback).
template <int S>
__device__ __forceinline__ void write_pixel(const RasterParams& P, const TriRecs& recs, const SlotMap& slotOf,
                                            const PixelCtx& C, const unsigned long long* keys, float* visDepth,
                                            uint32_t* visSlot, uint8_t* visClass) {
    if (!C.inFb || !scissor_pass(P.scissor, C.fpx, C.fpy)) return;
    unsigned won = 0;
#pragma unroll
    for (int s = 0; s < S; s++) won |= (unsigned)(keys[s] != frag_key(visDepth[C.pix * S + s], 0u)) << s;
    unsigned slots[S];
    key_slots<S>(slotOf, keys, won, slots);
    unsigned cls = 0;
#pragma unroll
    for (int s = 0; s < S; s++) {
        const unsigned long long k = keys[s];
        if (!((won >> s) & 1u)) continue;
        const unsigned slot = slots[s];
        float d = order_key_inv((unsigned)(k >> 32));
        if (S == 1 && (unsigned)(k >> 32) == 0x80000000u) {
            // +0 and -0 share a key: recompute the winner's own depth bits from its record
            cls = winner_class(load_rec(recs, slot), C.tx, C.ty, C.fpx, C.fpy, C.bMinX, C.bMinY, d, P.tagging);
        } else if (S == 1) {
            cls = (unsigned)k & 3u;
        } else if (S > 1 && (unsigned)(k >> 32) == 0x80000000u) {
            // +0 and -0 share a key; recompute to return the winner's own bits
            d = depth256(recs.f1[slot], recs.f2[slot], recs.f3[slot], C.fpx + P.sx[s], C.fpy + P.sy[s]);
        }
        visDepth[C.pix * S + s] = d;
        visSlot[C.pix * S + s] = slot;
    }
    if (S == 1 && visClass && won) visClass[C.pix] = class_out(cls, P.tagging);
}

// A view's outputs: depth per sample and, where wanted, record slots, primitive IDs and
// (1 sample per pixel) coverage classes.
// The key holds the primitive, so IDs cost their stores; expanding them from the slots
// in a pass of its own took 3 us at 256x256 and 6 us at 1080p, and a draw that is not
// shaded needs no slots.
struct VisOut {
    float* depth;
    uint32_t *slot, *ids;
    uint8_t* cls;
};
template <int S>
__device__ __forceinline__ VisOut vis_out(const RasterParams& P, const ViewGeom& G, float* depth, uint32_t* slot,
                                          uint8_t* cls) {
    const size_t at = G.pixBase * S;
    return VisOut{depth + at, slot ? slot + at : nullptr, P.ids ? P.ids + at : nullptr, cls ? cls + G.pixBase : nullptr};
}
__device__ __forceinline__ void store_ids(uint32_t* to, uint4 v, bool wide) {
    if (wide) {
        *reinterpret_cast<uint4*>(to) = v;
    } else {
        to[0] = v.x;
        to[1] = v.y;
        to[2] = v.z;
        to[3] = v.w;
    }
}

// One tile's outputs staged in LDS in global order (pixel-major, sample-
// minor) so that they leave with 16-byte stores of consecutive addresses;
// per-lane stores of one pixel's S samples would touch a partial line per
// sample.
template <int S>
struct TileOut {
    float d[256 * S];
    unsigned slot[256 * S];
};

// The S final keys of a cleared draw's pixel in the form the output stage takes
// (LESS keys), and which of them hold a fragment.
template <int S, bool G>
__device__ __forceinline__ unsigned final_keys(const RasterParams& P, unsigned long long* keys) {
    unsigned won = 0;
    const unsigned long long none = G ? general_clear_key(P) : frag_key(P.clearDepth, 0u);
#pragma unroll
    for (int s = 0; s < S; s++) {
        won |= (unsigned)(keys[s] != none) << s;
        if constexpr (G) keys[s] = less_key<S>(P, keys[s]);
    }
    return won;
}

// Outputs of one pixel of a cleared draw from its S final keys: depth and
// record slot per sample (the clear values where no fragment won) and, at 1
// sample per pixel, the coverage class.
template <int S>
__device__ __forceinline__ unsigned pixel_outputs(const RasterParams& P, const TriRecs& recs, const SlotMap& slotOf,
                                                  const PixelCtx& C, const unsigned long long* keys, unsigned won,
                                                  float* d, unsigned* slot) {
    unsigned cls = 0;
    unsigned slots[S];
    key_slots<S>(slotOf, keys, won, slots);
#pragma unroll
    for (int s = 0; s < S; s++) {
        const unsigned long long k = keys[s];
        d[s] = P.clearDepth;
        slot[s] = 0xffffffffu;
        if ((won >> s) & 1u) {
            slot[s] = slots[s];
            d[s] = order_key_inv((unsigned)(k >> 32));
            if (S == 1 && (unsigned)(k >> 32) == 0x80000000u) {
                // +0 and -0 share a key: recompute the winner's own depth bits from its record
                cls = winner_class(load_rec(recs, slot[s]), C.tx, C.ty, C.fpx, C.fpy, C.bMinX, C.bMinY, d[s],
                                   P.tagging);
            } else if (S == 1) {
                cls = (unsigned)k & 3u;
            } else if (S > 1 && (unsigned)(k >> 32) == 0x80000000u) {
                // +0 and -0 share a key; recompute to return the winner's own bits
                d[s] = depth256(recs.f1[slot[s]], recs.f2[slot[s]], recs.f3[slot[s]], C.fpx + P.sx[s],
                                C.fpy + P.sy[s]);
            }
        }
    }
    return cls;
}

// Outputs of one pixel of a cleared draw into the staging buffer; the 1-spp
// class byte goes straight out.
template <int S>
__device__ __forceinline__ void stage_pixel(const RasterParams& P, const TriRecs& recs, const SlotMap& slotOf,
                                            const PixelCtx& C, int t, const unsigned long long* keys, unsigned won,
                                            TileOut<S>& O, const VisOut& vis) {
    if (!C.inFb) return;
    if (!scissor_pass(P.scissor, C.fpx, C.fpy)) {
        // outside the scissor: the tile's line stores write the pixel's current contents back
#pragma unroll
        for (int s = 0; s < S; s++) {
            O.d[t * S + s] = vis.depth[C.pix * S + s];
            if (vis.slot) O.slot[t * S + s] = vis.slot[C.pix * S + s];
        }
        return;
    }
    float d[S];
    unsigned slot[S];
    const unsigned cls = pixel_outputs<S>(P, recs, slotOf, C, keys, won, d, slot);
#pragma unroll
    for (int s = 0; s < S; s++) {
        O.d[t * S + s] = d[s];
        O.slot[t * S + s] = slot[s];
    }
    if (S == 1 && vis.cls) vis.cls[C.pix] = class_out(cls, P.tagging);
    if (S == 1 && vis.ids) vis.ids[C.pix] = won ? key_tie<S>(keys[0]) >> 2 : 0xffffffffu;
}

// Outputs of one pixel of a cleared draw straight to memory with 16-byte
// stores (S a multiple of 4: a pixel's samples fill whole 16-byte words, and
// a row of pixels whole lines).
template <int S>
__device__ __forceinline__ void emit_pixel(const RasterParams& P, const TriRecs& recs, const SlotMap& slotOf,
                                           const PixelCtx& C, const unsigned long long* keys, unsigned won,
                                           const VisOut& vis) {
    static_assert(S % 4 == 0, "whole 16-byte words per pixel");
    if (!C.inFb || !scissor_pass(P.scissor, C.fpx, C.fpy)) return;
    float d[S];
    unsigned slot[S];
    pixel_outputs<S>(P, recs, slotOf, C, keys, won, d, slot);
    float4* const dd = reinterpret_cast<float4*>(vis.depth + C.pix * S);
    uint4* const ds = reinterpret_cast<uint4*>(vis.slot + C.pix * S);
#pragma unroll
    for (int v = 0; v < S / 4; v++) {
        dd[v] = make_float4(d[4 * v], d[4 * v + 1], d[4 * v + 2], d[4 * v + 3]);
        if (vis.slot) ds[v] = make_uint4(slot[4 * v], slot[4 * v + 1], slot[4 * v + 2], slot[4 * v + 3]);
        if (vis.ids) {
            auto id = [&](int s) { return (won >> s) & 1u ? key_tie<S>(keys[s]) >> 2 : 0xffffffffu; };
            store_ids(vis.ids + C.pix * S + 4 * v, make_uint4(id(4 * v), id(4 * v + 1), id(4 * v + 2), id(4 * v + 3)),
                      P.idsWide != 0);
        }
    }
}

// Stores a staged tile with 16-byte stores; partial columns at the right
// edge fall back to scalars.  visDepth, visSlot and visClass point at the
// view's outputs; a view's first pixel starts a 16-byte line when S > 1 or its
// pixel base is a multiple of 4.
template <int S, int NT = 256>
__device__ __forceinline__ void store_tile(int t, const ViewGeom& G, int tx, int ty, const TileOut<S>* O,
                                           const VisOut& vis) {
    constexpr int perRow = 16 * S / 4;  // float4 per tile row
    const int cols = min(16, G.width - tx * 16), rows = min(16, G.height - ty * 16);
    const bool vec = cols == 16 && (S > 1 || ((G.width & 3) == 0 && (G.pixBase & 3) == 0));
    for (int i = t; i < 64 * S; i += NT) {
        const int row = i / perRow, q = i - row * perRow;
        if (row >= rows) continue;
        const size_t g = ((size_t)(ty * 16 + row) * G.width + tx * 16) * S + q * 4;
        const int l = row * 16 * S + q * 4;
        const float4 d = *reinterpret_cast<const float4*>(&O->d[l]);
        const uint4 sl = *reinterpret_cast<const uint4*>(&O->slot[l]);
        if (vec) {
            *reinterpret_cast<float4*>(&vis.depth[g]) = d;
            if (vis.slot) *reinterpret_cast<uint4*>(&vis.slot[g]) = sl;
        } else {
            const float dv[4] = {d.x, d.y, d.z, d.w};
            const unsigned sv[4] = {sl.x, sl.y, sl.z, sl.w};
#pragma unroll
            for (int e = 0; e < 4; e++) {
                if ((q * 4 + e) / S >= cols) continue;
                vis.depth[g + e] = dv[e];
                if (vis.slot) vis.slot[g + e] = sv[e];
            }
        }
    }
}

// Clear values of one tile whose list is empty (depth clearDepth, slot
// 0xffffffff and, at 1 sample per pixel, class 0) by NT threads, with 16-byte
// stores where the tile's rows are whole.
template <int S, int NT>
__device__ __forceinline__ void clear_tile(int t, const ViewGeom& G, float clearDepth, const Scissor& sc,
                                           bool idsWide, const VisOut& vis) {
    const int tx = G.tile % G.tilesX, ty = G.tile / G.tilesX;
    const int cols = min(16, G.width - tx * 16), rows = min(16, G.height - ty * 16);
    const bool whole = scissor_all(sc, tx * 16, ty * 16, tx * 16 + cols - 1, ty * 16 + rows - 1);
    const bool vec = whole && cols == 16 && (S > 1 || ((G.width & 3) == 0 && (G.pixBase & 3) == 0));
    constexpr int perRow = 16 * S / 4;  // 16-byte words per tile row
    for (int i = t; i < 64 * S; i += NT) {
        const int row = i / perRow, q = i - row * perRow;
        if (row >= rows) continue;
        const size_t g = ((size_t)(ty * 16 + row) * G.width + tx * 16) * S + q * 4;
        if (vec) {
            *reinterpret_cast<float4*>(&vis.depth[g]) = make_float4(clearDepth, clearDepth, clearDepth, clearDepth);
            if (vis.slot) *reinterpret_cast<uint4*>(&vis.slot[g]) = make_uint4(~0u, ~0u, ~0u, ~0u);
            if (vis.ids) store_ids(&vis.ids[g], make_uint4(~0u, ~0u, ~0u, ~0u), idsWide);
        } else {
#pragma unroll
            for (int e = 0; e < 4; e++) {
                const int col = (q * 4 + e) / S;
                if (col >= cols) continue;
                if (!whole && !scissor_pass(sc, (float)(tx * 16 + col), (float)(ty * 16 + row))) continue;
                vis.depth[g + e] = clearDepth;
                if (vis.slot) vis.slot[g + e] = 0xffffffffu;
                if (vis.ids) vis.ids[g + e] = 0xffffffffu;
            }
        }
    }
    if (S == 1 && vis.cls) {
        for (int i = t; i < 256; i += NT) {
            const int row = i >> 4, col = i & 15;
            if (row < rows && col < cols &&
                (whole || scissor_pass(sc, (float)(tx * 16 + col), (float)(ty * 16 + row))))
                vis.cls[(size_t)(ty * 16 + row) * G.width + tx * 16 + col] = 0;
        }
    }
}

// LDS layout of the tile's keys: sample-major, 256 pixels per sample.
// Padded layouts lowered the bank-conflict share of LDS-active cycles (one
// key after every 32: 40 % to 35 %; four after every 32: 48 % to 31 %) but
// not the kernel time (unchanged, then 3 % slower from the extra address
// arithmetic): conflicts cost about 4 % of its cycles, and the kernel is
// bound by VALU issue.
constexpr int kVisStride = 256;
__device__ __forceinline__ int vis_at(int s, int p) { return s * kVisStride + p; }

// A record in LDS, an odd number of 16-byte words apart: lanes that read the same word of
// different records meet in a bank for one record in sixteen, at 96 bytes for one in eight:
// 4.2M half-pixel triangles at 4 samples 209 -> 202 us, 1.3M at 8 79 -> 77.5 us.
struct LdsRec : TriRec {
    float4 pad;
};

// NT threads per tile: 256 (one pixel per thread) or, at 1 sample per pixel,
// 64 (one wave per tile, four pixels per lane: more tiles in flight per
// compute unit, for many small tiles).  Passes hold NT / 2 entries, WIDE ones NT.  G: the
// general keys of a cleared draw with another depth function than LESS, which
// also marks the tiles that met a NaN depth (nanTile): in those the function's
// result depends on the order after all.
//
// Bound by the latency of an item's chain (claim, item, view, list entries,
// records, then the window and unit rounds) and by VALU issue: 69 % of its
// cycles at 1920x1080, 8 samples, 1.3M triangles, 46 % at 1 sample.  Held to the
// registers of five workgroups per compute unit at 1 and 4 samples (at 8 the
// keys' LDS allows four).  Windows from pixel boxes, one lane per entry, instead of block
// tests of every entry by two: 105 -> 84 us there, and 78 us with fewer registers; 4.2M
// half-pixel triangles at 4 samples 327 -> 213 us, 34 views at 1 sample 525 -> 355 us.
// Items and views through the scalar cache and a pass's entries loaded during the one
// before: 351 -> 330 us at the 34 views, 215 -> 207 and 81 -> 79 us at the others.
// WIDE is for draws that leave the chip idle (RasterQueue::wide), where the passes of
// the longest list are what is waited for: 15 -> 11.5 us for a 256x256 target, 26 -> 22
// at 1009x767 with 4 samples; their LDS leaves three workgroups per compute unit, and
// with 1.3M triangles it costs 48 -> 56 us (1 sample) and 79 -> 90 us (8).
template <int S, int NT, bool WIDE, bool G>
__global__ void __launch_bounds__(NT) __attribute__((amdgpu_waves_per_eu(WIDE ? (S == 8 ? 2 : 3) : S == 8 ? 4 : 5, 8)))
k_raster(RasterParams P, Views V, TriRecs recs, const unsigned* __restrict__ slotOfAll,
         const WaveInfo* __restrict__ waves, const unsigned* __restrict__ binList, RasterQueue q,
         const unsigned* __restrict__ emptyEnd, float* __restrict__ visDepthAll, uint32_t* __restrict__ visSlotAll,
         uint8_t* __restrict__ visClassAll, StatPartials st, DeviceCounters* ctr, unsigned* __restrict__ nanTile) {
    constexpr int PASS = WIDE ? NT : NT / 2;  // list entries per pass through LDS
    constexpr int UNITS = NT * 8;           // units expanded into LDS per round
    constexpr int PAIRS = 16 * PASS;        // (entry, window) pairs of a pass
    using Unit = typename std::conditional<S == 1, unsigned, unsigned short>::type;
    constexpr int PPT = 256 / NT;           // tile pixels per thread
    static_assert(PASS <= 256, "pairs and units encode the entry in 8 bits");
    // key of sample s of tile pixel p at vis_at(s, p)
    __shared__ unsigned long long sVis[S * kVisStride];
    static_assert(sizeof(TileOut<S>) <= sizeof(sVis), "output staging reuses sVis");
    __shared__ LdsRec sRec[PASS];            // q2.z: bit 31 when the tile is accepted, else the pixel box
    __shared__ Unit sUnit[UNITS];            // entry << 8 | tile pixel, and << 2 | class at 1 sample
    __shared__ unsigned short sPair[PAIRS];  // entry << 8 | window row << 4 | column
    __shared__ unsigned sWave[4];
    __shared__ unsigned sItem;

    const bool fits = plan_fits(ctr, q);
    const unsigned numLong = ctr->tot[kTotLong], numItems = fits ? numLong + ctr->tot[kTotShort] : 0u;
    // tiles with an empty list follow the items: their clear values, KE tiles
    // per claim at 1 sample per pixel (a small write each)
    constexpr unsigned KE = S == 1 ? 8u : 1u;
    const unsigned numEmpty = P.clear && fits ? ctr->tot[kTotEmpty] : 0u;
    const unsigned numEmptyItems = (numEmpty + KE - 1u) / KE;
    unsigned long long frags = 0, covs = 0;

    // thread 0 claims the next item of the workgroup's stream before the
    // output stage of the current one, so that the claim's latency overlaps
    // the output stage.  The counter's address is moved to vector registers:
    // a uniform address would turn the claim into a wave-aggregated atomic
    // whose result is awaited at once.
    const unsigned stream = blockIdx.x % kItemStreams;
    __attribute__((address_space(1))) unsigned* head =
        (__attribute__((address_space(1))) unsigned*)&ctr->itemHeads[stream][0];
    asm volatile("" : "+v"(head));
    unsigned claimed = 0;
    if (threadIdx.x == 0) claimed = __hip_atomic_fetch_add(head, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    for (;;) {
        // opaque to the compiler, which would otherwise keep every thread's share of the
        // output and clear stages' index arithmetic in registers across the whole loop
        int t = threadIdx.x;
        asm volatile("" : "+v"(t));
        if (t == 0) sItem = claimed;
        __syncthreads();
        const unsigned item = (unsigned)__builtin_amdgcn_readfirstlane((int)sItem) * kItemStreams + stream;
        if (item >= numItems) {
            const unsigned e = item - numItems;
            if (e >= numEmptyItems) break;
            if (t == 0) claimed = __hip_atomic_fetch_add(head, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            for (unsigned k = e * KE; k < min(e * KE + KE, numEmpty); k++) {
                const ViewGeom E = view_of_tile(V, (int)uniform_word(emptyEnd - k));
                clear_tile<S, NT>(t, E, P.clearDepth, P.scissor, P.idsWide != 0,
                                  vis_out<S>(P, E, visDepthAll, visSlotAll, visClassAll));
            }
            __syncthreads();  // every lane has read sItem
            continue;
        }
        // long items from the front of the array, then short ones from its back
        const uint4 it = uniform_words(q.items + (item < numLong ? item : q.itemCap - 1u - (item - numLong)));
        const int tile = (int)it.x, cnt = (int)it.z;
        const unsigned first = it.y, pslot = it.w;
        // a pass's entries are loaded during the one before, the first pass's before the view is known
        unsigned ent = t < cnt && t < PASS ? binList[first + t] : 0u;
        const ViewGeom G_ = view_of_tile(V, tile);
        const VisOut vis = vis_out<S>(P, G_, visDepthAll, visSlotAll, visClassAll);
        const SlotMap slotOf{slotOfAll + G_.primBase, waves + (size_t)G_.view * V.waves, G_.slotBase,
                             uniform_word(&V.ctr[G_.view].clipIn) != 0u};
        const int ttx = G_.tile % G_.tilesX, tty = G_.tile / G_.tilesX;
        const int tx0 = ttx * 16, ty0 = tty * 16;

#pragma unroll
        for (int k = 0; k < PPT; k++) {
            const int p = t + k * NT;
            const PixelCtx C = pixel_ctx(G_, p & 15, p >> 4);
#pragma unroll
            for (int s = 0; s < S; s++)
                sVis[vis_at(s, p)] =
                    G ? general_clear_key(P)
                      : frag_key(P.clear || !C.inFb ? P.clearDepth : vis.depth[C.pix * S + s], 0u);
        }

        const int cols = min(16, G_.width - tx0), rows = min(16, G_.height - ty0);
        // blocks with a pixel inside the frame
        const unsigned blkFb = ((1u << ((cols + 3) >> 2)) - 1u) * 0x1111u & ((1u << (4 * ((rows + 3) >> 2))) - 1u);

        auto merge = [&](unsigned long long* cell, bool on, float d, unsigned tie) {
            if constexpr (G) {
                if (on & ((d == d) | (P.keyMask == 0u))) atomicMin(cell, general_key<S>(P, d, tie));
                if (on & (d != d) & (P.keyMask != 0u)) nanTile[2 * tile] = 1u;
            } else {
                if (on & (d == d)) atomicMin(cell, frag_key(d, tie));
            }
        };

        // merges units sUnit[0, nu) into sVis
        auto merge_units = [&](int nu) {
            for (int i = t; i < nu; i += NT) {
                unsigned u = sUnit[i];
                if constexpr (S == 1) {
                    const unsigned cls = u & 3u;
                    u >>= 2;
                    const int e = (int)(u >> 8), c = (int)(u & 255u);
                    const float4 F1 = sRec[e].f1, F2 = sRec[e].f2, F3 = sRec[e].f3;
                    const unsigned tie = __float_as_uint(sRec[e].q2.y);
                    // every class's depth is computed and one selected: a wave's lanes hold all of them
                    const float d = class_depth_all(cls, F1, F2, F3, (float)(tx0 + (c & 15)), (float)(ty0 + (c >> 4)),
                                                    P.tagging);
                    merge(&sVis[vis_at(0, c)], true, d, (tie << 2) | cls);
                    frags++;
                } else {
                    const int e = (int)(u >> 8), c = (int)(u & 255u);
                    const TriRec R = sRec[e];
                    const Edges E = load_edges(R);
                    const unsigned tie = __float_as_uint(R.q2.y);
                    const bool accept = (__float_as_uint(R.q2.z) >> 31) != 0u;
                    const float fx = (float)(tx0 + (c & 15)), fy = (float)(ty0 + (c >> 4));
                    // every sample's coverage and depth are computed (the lanes of a
                    // wave cover different pixels, so branches would run both ways);
                    // only the merge is conditional
                    unsigned ncov = 0;
#pragma unroll
                    for (int s = 0; s < S; s++) {
                        const float sx = fx + P.sx[s], sy = fy + P.sy[s];
                        const bool cov = accept | inside_and(E, sx, sy);
                        const float d = depth256(R.f1, R.f2, R.f3, sx, sy);
                        ncov += cov;
                        merge(&sVis[vis_at(s, c)], cov, d, tie);
                    }
                    covs += ncov;
                    frags += ncov != 0u;
                }
            }
        };

        // passes of PASS entries through LDS, all merging into sVis
        for (int pb = 0; pb < cnt; pb += PASS) {
            const int pc = min(PASS, cnt - pb);
            // one lane per entry: its windows
            unsigned n = 0, blocks = 0;
            int bx0 = 0, by0 = 0, wcols = 0;
            if (t < pc) {
                const TriRec R = load_rec(recs, ent & 0x7fffffffu);
                static_cast<TriRec&>(sRec[t]) = R;
                const Edges E = load_edges(R);
                const bool full = (ent >> 31) != 0u;
                const unsigned lo = __float_as_uint(R.q2.z), hi = __float_as_uint(R.q2.w);
                // the pixel box within the tile
                const int x0 = max((int)(lo & 0xFFFFu) - tx0, 0), y0 = max((int)(lo >> 16) - ty0, 0);
                const int x1 = min((int)(hi & 0xFFFFu) - tx0, 15), y1 = min((int)(hi >> 16) - ty0, 15);
                if (full) {
                    blocks = blkFb;
                    n = (unsigned)__popc(blocks);
                } else if (x0 <= x1 && y0 <= y1) {
                    // at 1 sample a window off the blocks' grid must hold the whole box (window_classes)
                    constexpr int kFew = S == 1 ? 4 : 8;
                    if (x1 - x0 < kFew && y1 - y0 < kFew) {
                        wcols = (x1 - x0 + 4) >> 2;
                        n = (unsigned)(wcols * ((y1 - y0 + 4) >> 2));
                        bx0 = x0;
                        by0 = y0;
                    } else {
                        blocks = blocks_not_rejected(E, tx0, ty0) & blkFb;
                        n = (unsigned)__popc(blocks);
                    }
                }
                // the box within the tile, for the window lanes; an accepted tile has none
                sRec[t].q2.z = __uint_as_float(full ? 0x80000000u
                                                    : (unsigned)(x0 | (y0 << 4) | (max(x1, 0) << 8) | (max(y1, 0) << 12)));
            }
            if (t < PASS && pb + PASS + t < cnt) ent = binList[first + pb + PASS + t];
            unsigned TP;
            int pp = (int)scan_nt<NT>(t, n, sWave, TP);
            if (blocks) {
                while (blocks) {
                    const int q = __ffs(blocks) - 1;
                    blocks &= blocks - 1u;
                    sPair[pp++] = (unsigned short)((t << 8) | ((q >> 2) << 6) | ((q & 3) << 2));
                }
            } else {
                for (int k = 0; k < (int)n; k++) {
                    const int wx = bx0 + 4 * few_col(k, wcols), wy = by0 + 4 * few_row(k, wcols);
                    sPair[pp++] = (unsigned short)((t << 8) | (wy << 4) | wx);
                }
            }
            __syncthreads();
            for (unsigned p0 = 0; p0 < TP; p0 += NT) {
                // one lane per window: its pixels
                unsigned pm = 0, groups = 0, quads = 0;
                int pe = 0, wx = 0, wy = 0;
                bool acc = false;
                if (p0 + t < TP) {
                    const unsigned pr = sPair[p0 + t];
                    pe = (int)(pr >> 8);
                    wx = (int)(pr & 15u);
                    wy = (int)((pr >> 4) & 15u);
                    const unsigned bits = __float_as_uint(sRec[pe].q2.z);
                    acc = (bits >> 31) != 0u;  // the tile, or below the block, is accepted
                    // up to the frame's and the box's last column and row
                    const int lx = acc ? cols : min(cols, (int)((bits >> 8) & 15u) + 1);
                    const int ly = acc ? rows : min(rows, (int)((bits >> 12) & 15u) + 1);
                    pm = block_fb_mask(lx - wx, ly - wy);
                    if (!acc) {
                        const Edges E = load_edges(sRec[pe]);
                        const float fx = (float)(tx0 + wx), fy = (float)(ty0 + wy);
                        if constexpr (S == 1) {
                            if (((wx | wy) & 3) == 0) acc = block_accepted(E, fx, fy);
                            const unsigned in = window_inside(E, fx, fy);
                            window_classes(in, wx, wy, groups, quads);
                            pm &= in;
                        } else {
                            pm &= block_square_mask(E, fx, fy);
                        }
                    }
                }
                const int np = __popc(pm);
                unsigned T;
                const unsigned off = scan_nt<NT>(t, (unsigned)np, sWave, T);
                for (unsigned w0 = 0; w0 < T; w0 += UNITS) {
                    // write this lane's units that fall in [w0, w0 + UNITS): window pixel b is tile
                    // pixel (wy + (b >> 2)) * 16 + wx + (b & 3)
                    int pos = (int)off - (int)w0;
                    if (np && pos < UNITS && pos + np > 0) {
                        const int cb = (pe << 8) | (wy * 16 + wx);
                        auto unit = [&](int b) {
                            const unsigned u = (unsigned)(cb + ((b >> 2) << 4) + (b & 3));
                            if constexpr (S == 1)
                                return (Unit)((u << 2) | expr_code(acc, (groups >> b) & 1u, (quads >> b) & 1u, P.tagging));
                            else
                                return (Unit)u;
                        };
                        unsigned bits = pm;
                        if (pos >= 0 && pos + np <= UNITS) {
                            // the lane's units all fall in this window
                            while (bits) {
                                const int b = __ffs(bits) - 1;
                                bits &= bits - 1u;
                                sUnit[pos++] = unit(b);
                            }
                        } else {
                            while (bits) {
                                const int b = __ffs(bits) - 1;
                                bits &= bits - 1u;
                                if (pos >= 0 && pos < UNITS) sUnit[pos] = unit(b);
                                pos++;
                            }
                        }
                    }
                    __syncthreads();
                    merge_units((int)min((unsigned)UNITS, T - w0));
                    __syncthreads();
                }
                if (T == 0) __syncthreads();  // sWave is read by the next round's scan
            }
            __syncthreads();  // sRec and sWave are reused by the next pass
        }

        if (t == 0) claimed = __hip_atomic_fetch_add(head, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        if (pslot != 0xFFFFFFFFu) {
            // one item of a longer list: its keys, sample-major like sVis
            unsigned long long* g = q.partials + (size_t)pslot * 256 * S;
#pragma unroll
            for (int k = 0; k < PPT; k++)
#pragma unroll
                for (int s = 0; s < S; s++) g[s * 256 + t + k * NT] = sVis[vis_at(s, t + k * NT)];
        } else {
            unsigned long long keys[PPT][S];
#pragma unroll
            for (int k = 0; k < PPT; k++)
#pragma unroll
                for (int s = 0; s < S; s++) keys[k][s] = sVis[vis_at(s, t + k * NT)];
            if (G || P.clear) {
                if constexpr (S > 1) {
                    // a pixel's samples are whole 16-byte words: straight out
#pragma unroll
                    for (int k = 0; k < PPT; k++) {
                        const int p = t + k * NT;
                        const unsigned won = final_keys<S, G>(P, keys[k]);
                        emit_pixel<S>(P, recs, slotOf, pixel_ctx(G_, p & 15, p >> 4), keys[k], won, vis);
                    }
                } else {
                    // every key is in registers: stage the outputs over sVis
                    TileOut<S>* O = reinterpret_cast<TileOut<S>*>(sVis);
                    __syncthreads();
#pragma unroll
                    for (int k = 0; k < PPT; k++) {
                        const int p = t + k * NT;
                        const unsigned won = final_keys<S, G>(P, keys[k]);
                        stage_pixel<S>(P, recs, slotOf, pixel_ctx(G_, p & 15, p >> 4), p, keys[k], won, *O, vis);
                    }
                    __syncthreads();
                    store_tile<S, NT>(t, G_, ttx, tty, O, vis);
                }
            } else {
#pragma unroll
                for (int k = 0; k < PPT; k++) {
                    const int p = t + k * NT;
                    write_pixel<S>(P, recs, slotOf, pixel_ctx(G_, p & 15, p >> 4), keys[k], vis.depth, vis.slot,
                                   vis.cls);
                }
            }
        }
        __syncthreads();  // every lane has read sItem and the LDS of this item
    }
    const unsigned long long tf = sum_nt<NT>(frags);
    const unsigned long long tc = S == 1 ? tf : sum_nt<NT>(covs);  // at 1 sample a fragment is a covered sample
    if (threadIdx.x == 0) {
        st.rasterFrags[blockIdx.x] = tf;
        st.rasterCovs[blockIdx.x] = tc;
    }
}

// Minimum over the parts of every tile whose list was cut, then the outputs
// (the empty tiles' clear values come from k_raster).  The last workgroup reduces the
// draw's statistics meanwhile.
template <int S>
__global__ void __launch_bounds__(256) k_raster_merge(RasterParams P, Views V, TriRecs recs,
                                                      const unsigned* __restrict__ slotOfAll,
                                                      const WaveInfo* __restrict__ waves,
                                                      const unsigned* __restrict__ binStart,
                                                      const unsigned* __restrict__ binEnd, RasterQueue q,
                                                      float* __restrict__ visDepthAll, uint32_t* __restrict__ visSlotAll,
                                                      uint8_t* __restrict__ visClassAll, DeviceCounters* ctr, StatPartials st,
                                                      HostCounters* out) {
    if (blockIdx.x == gridDim.x - 1u) {
        finalize_block<256>(st, V, ctr, out);
        return;
    }
    const unsigned numMulti = plan_fits(ctr, q) ? ctr->tot[kTotMulti] : 0u;
    const int t = threadIdx.x;
    // tiles whose list was cut into several items: the minimum over their partial blocks
    for (unsigned m = blockIdx.x; m < numMulti; m += gridDim.x - 1u) {
        const int tile = (int)q.multiList[m];
        const ViewGeom G = view_of_tile(V, tile);
        const VisOut vis = vis_out<S>(P, G, visDepthAll, visSlotAll, visClassAll);
        const SlotMap slotOf{slotOfAll + G.primBase, waves + (size_t)G.view * V.waves, G.slotBase,
                             uniform_word(&V.ctr[G.view].clipIn) != 0u};
        const PixelCtx C = pixel_ctx(G, t & 15, t >> 4);
        const unsigned total = binEnd[tile] - binStart[tile];
        const unsigned nparts = (total + (1u << q.partShift) - 1u) >> q.partShift;
        const unsigned long long* g = q.partials + (size_t)q.tilePartial[tile] * 256 * S + t;
        unsigned long long keys[S];
#pragma unroll
        for (int s = 0; s < S; s++) keys[s] = g[s * 256];
        for (unsigned p = 1; p < nparts; p++) {
            g += 256 * S;
#pragma unroll
            for (int s = 0; s < S; s++) keys[s] = min(keys[s], g[s * 256]);
        }
        if (P.clear) {
            const unsigned won = P.general ? final_keys<S, true>(P, keys) : final_keys<S, false>(P, keys);
            if constexpr (S > 1) {
                emit_pixel<S>(P, recs, slotOf, C, keys, won, vis);
            } else {
                __shared__ TileOut<S> O;  // output staging at 1 sample per pixel
                __syncthreads();          // the previous tile's staging has been stored
                stage_pixel<S>(P, recs, slotOf, C, t, keys, won, O, vis);
                __syncthreads();
                store_tile<S>(t, G, C.tx, C.ty, &O, vis);
            }
        } else {
            write_pixel<S>(P, recs, slotOf, C, keys, vis.depth, vis.slot, vis.cls);
        }
    }
}

// ---------------------------------------------------------------------------
// Ordered raster: what the keys cannot express -- EQUAL, NOT_EQUAL and NEVER,
// GREATER at one sample (its scalar path), every function but LESS without
// clear, depth-writing programs, and tiles with NaN depths.  The result
// depends on the order of the fragments, so each tile's list is taken in the order of the reference's per-tile sort
// (TileRasterWorker.cpp:1225-1259) and every thread folds the fragments of
// its own pixel in that order (TileRasterWorker.cpp:2272-2311 and the SIMD
// forms); the scalar path's GREATER tests nothing
// (TileRasterWorker.cpp:2278-2280).
// ---------------------------------------------------------------------------
// One workgroup per tile (persistent over the tiles of all views, in the order
// of OrderedTiles), one thread per pixel holding its S samples' depth and winning
// slot; bound as k_blend_ordered is.  With nanTile
// only the tiles it marks are drawn, over the key raster's result, and their
// marks cleared.
template <int S>
__global__ void __launch_bounds__(256) k_raster_ordered(RasterParams P, Views V, TriRecs recs,
                                                        BinBufs B, RasterQueue q, int tiles, unsigned ntri,
                                                        float* __restrict__ visDepthAll,
                                                        uint32_t* __restrict__ visSlotAll,
                                                        uint8_t* __restrict__ visClassAll, StatPartials st,
                                                        unsigned* __restrict__ nanTile, DeviceCounters* ctr) {
    __shared__ OrderLds L;
    __shared__ unsigned sItem;
    const int t = threadIdx.x;
    unsigned long long frags = 0, covs = 0;
    OrderedTiles T(q, ctr, nanTile == nullptr);
    // with nanTile: the marks of up to 64 of the workgroup's tiles at a time (a bit each)
    unsigned long long marked = 0;
    int tile = 0, round = 0, left = 0;
    for (;;) {
        unsigned start, cnt;
        if (nanTile) {
            while (!marked) {
                if (left >= tiles) return;
                const int mine = (int)blockIdx.x + (64 * round + (t & 63)) * (int)gridDim.x;
                marked = __ballot(mine < tiles && nanTile[2 * mine] != 0u);
                __syncthreads();  // every wave has read the marks before the first is cleared
                left = (int)blockIdx.x + 64 * ++round * (int)gridDim.x;
            }
            tile = (int)blockIdx.x + (64 * (round - 1) + __ffsll(marked) - 1) * (int)gridDim.x;
            marked &= marked - 1ull;
            start = B.start[tile];
            cnt = start >= P.binCap ? 0u : min(B.cursor[tile] - start, P.binCap - start);
        } else if (!T.next(q, B, tiles, &sItem, tile, start, cnt)) {
            break;
        }
        const ViewGeom G = view_of_tile(V, tile);
        const PixelCtx C = pixel_ctx(G, quarter_x(t), quarter_y(t));
        const VisOut vis = vis_out<S>(P, G, visDepthAll, visSlotAll, visClassAll);
        float dep[S];
        unsigned slot[S];
        unsigned cls = 0;
#pragma unroll
        for (int s = 0; s < S; s++) {
            dep[s] = P.clear || !C.inFb ? P.clearDepth : vis.depth[C.pix * S + s];
            slot[s] = P.clear || !C.inFb ? 0xffffffffu : vis.slot[C.pix * S + s];
        }
        if (!P.clear && S == 1 && vis.cls && C.inFb) cls = vis.cls[C.pix];
        for_each_ordered<S>(
            recs, B.list, start, cnt, G.slotBase, ntri, C, P.tagging, L,
            [&](const TriRec& R, unsigned sl, unsigned c) {
                if (!C.inFb) return;
                if constexpr (S == 1) {
                    const float d = class_depth(c, R.f1, R.f2, R.f3, C.fpx, C.fpy, P.tagging);
                    frags++;
                    covs++;
                    // the scalar path's GREATER quirk belongs to the deterministic mode's single pixels
                    if (!depth_pass(P.depthFunc, d, dep[0], c == 3u && !P.tagging)) return;
                    dep[0] = P.depthWrite ? d * P.depthScale + P.depthBias : d;
                    slot[0] = sl;
                    cls = class_out(c, P.tagging);
                } else {
                    const Edges E = load_edges(R);
                    bool any = false;
#pragma unroll
                    for (int s = 0; s < S; s++) {
                        const float sx = C.fpx + P.sx[s], sy = C.fpy + P.sy[s];
                        if (!(c == 3u || inside(E, sx, sy))) continue;
                        any = true;
                        covs++;
                        const float d = depth256(R.f1, R.f2, R.f3, sx, sy);
                        if (!depth_pass(P.depthFunc, d, dep[s], false)) continue;
                        dep[s] = P.depthWrite ? d * P.depthScale + P.depthBias : d;
                        slot[s] = sl;
                    }
                    frags += any;
                }
            });
        if (C.inFb && scissor_pass(P.scissor, C.fpx, C.fpy)) {
#pragma unroll
            for (int s = 0; s < S; s++) {
                vis.depth[C.pix * S + s] = dep[s];
                if (vis.slot) vis.slot[C.pix * S + s] = slot[s];
                if (vis.ids)
                    vis.ids[C.pix * S + s] = slot[s] == 0xffffffffu ? slot[s] : __float_as_uint(recs.q2[slot[s]].y) >> 2;
            }
            if (S == 1 && vis.cls) vis.cls[C.pix] = (uint8_t)cls;
        }
        if (nanTile && t == 0) nanTile[2 * tile] = 0u;
    }
    if (nanTile) return;  // the key raster has counted
    const unsigned long long tf = block_sum256(frags);
    const unsigned long long tc = block_sum256(covs);
    if (t == 0) {
        st.rasterFrags[blockIdx.x] = tf;
        st.rasterCovs[blockIdx.x] = tc;
    }
}

// Primitive ID per sample from the record slot (readback only).
__global__ void __launch_bounds__(256) k_slot_to_prim(const uint32_t* __restrict__ visSlot, const float4* __restrict__ q2,
                                                      size_t n, uint32_t* __restrict__ visId, int polygon) {
    for (size_t i = (size_t)blockIdx.x * 256 + threadIdx.x; i < n; i += (size_t)gridDim.x * 256) {
        const unsigned slot = visSlot[i];
        const unsigned key = slot == 0xffffffffu ? 0u : __float_as_uint(q2[slot].y);
        visId[i] = slot == 0xffffffffu ? 0xffffffffu : (polygon ? (key >> 2) * 3u + (key & 3u) : key >> 2);
    }
}

// Order-independent digest: the sum over i of SplitMix64(i << 32 ^ data[i])
// (the finaliser of Steele, Lea and Flood, 2014), reduced per workgroup and
// added into *out.
__device__ __forceinline__ unsigned long long splitmix64(unsigned long long z) {
    z += 0x9E3779B97F4A7C15ull;
    z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
    z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
    return z ^ (z >> 31);
}

__global__ void __launch_bounds__(256) k_digest(const uint32_t* __restrict__ data, size_t n,
                                                unsigned long long* out) {
    unsigned long long acc = 0;
    for (size_t i = (size_t)blockIdx.x * 256 + threadIdx.x; i < n; i += (size_t)gridDim.x * 256)
        acc += splitmix64(((unsigned long long)i << 32) ^ data[i]);
    acc = block_sum256(acc);
    if (threadIdx.x == 0) atomicAdd(out, acc);
}

}  // namespace

void launch_digest(const uint32_t* data, size_t n, unsigned long long* out, hipStream_t s) {
    if (n == 0) return;
    hipLaunchKernelGGL(k_digest, dim3((unsigned)std::min<size_t>(2048, (n + 255) / 256)), dim3(256), 0, s, data, n,
                       out);
}

void launch_slot_to_prim(const uint32_t* visSlot, TriRecs recs, size_t n, uint32_t* visId, hipStream_t s,
                         bool polygon) {
    hipLaunchKernelGGL(k_slot_to_prim, dim3(2048), dim3(256), 0, s, visSlot, recs.q2, n, visId, polygon ? 1 : 0);
}

// The raster and merge launches are separate so that the host can time them.
void launch_raster(const RasterParams& p, const Views& views, int samples, TriRecs recs, const unsigned* slotOf,
                   const BinBufs& bins, const RasterQueue& q, int tiles, float* visDepth, uint32_t* visSlot,
                   uint8_t* visClass, StatPartials st, DeviceCounters* ctr, hipStream_t s) {
#define IFRIT_RASTER_LAUNCH_G(SN, NT, WIDE, G)                                                                     \
    hipLaunchKernelGGL((k_raster<SN, NT, WIDE, G>), dim3(q.grid), dim3(NT), 0, s, p, views, recs, slotOf,          \
                       bins.waves, bins.list, q, q.multiList + tiles - 1, visDepth, visSlot, visClass, st, ctr,   \
                       bins.cnt)
#define IFRIT_RASTER_LAUNCH(SN, NT, WIDE)                                                                          \
    do {                                                                                                           \
        if (p.general)                                                                                             \
            IFRIT_RASTER_LAUNCH_G(SN, NT, WIDE, true);                                                             \
        else                                                                                                       \
            IFRIT_RASTER_LAUNCH_G(SN, NT, WIDE, false);                                                            \
    } while (0)
    if (samples == 1 && q.tileThreads == 64) {
        IFRIT_RASTER_LAUNCH(1, 64, false);
        return;
    }
    switch (samples) {
        case 1:
            if (q.wide)
                IFRIT_RASTER_LAUNCH(1, 256, true);
            else
                IFRIT_RASTER_LAUNCH(1, 256, false);
            break;
        case 4:
            if (q.wide)
                IFRIT_RASTER_LAUNCH(4, 256, true);
            else
                IFRIT_RASTER_LAUNCH(4, 256, false);
            break;
        default:
            if (q.wide)
                IFRIT_RASTER_LAUNCH(8, 256, true);
            else
                IFRIT_RASTER_LAUNCH(8, 256, false);
            break;
    }
#undef IFRIT_RASTER_LAUNCH_G
#undef IFRIT_RASTER_LAUNCH
}

void launch_raster_ordered(const RasterParams& p, const Views& views, int samples, TriRecs recs,
                           const BinBufs& bins, const RasterQueue& q, int tiles, float* visDepth, uint32_t* visSlot,
                           uint8_t* visClass, StatPartials st, bool nanTilesOnly, DeviceCounters* ctr,
                           hipStream_t s) {
#define IFRIT_ORDERED_LAUNCH(SN)                                                                                  \
    hipLaunchKernelGGL(k_raster_ordered<SN>, dim3(nanTilesOnly ? (q.grid + 1) / 2 : q.grid), dim3(256), 0, s, p, views, recs, bins, q, tiles, p.ntri,  \
                       visDepth, visSlot, visClass, st, nanTilesOnly ? bins.cnt : nullptr, ctr)
    switch (samples) {
        case 1: IFRIT_ORDERED_LAUNCH(1); break;
        case 4: IFRIT_ORDERED_LAUNCH(4); break;
        default: IFRIT_ORDERED_LAUNCH(8); break;
    }
#undef IFRIT_ORDERED_LAUNCH
}

void launch_raster_merge(const RasterParams& p, const Views& views, int samples, TriRecs recs, const unsigned* slotOf,
                         const BinBufs& bins, const RasterQueue& q, float* visDepth, uint32_t* visSlot,
                         uint8_t* visClass, int tiles, DeviceCounters* ctr, StatPartials st, HostCounters* out,
                         hipStream_t s) {
    // a workgroup per tile at most, and one for the statistics
    const int grid = std::max(1, std::min(2 * q.mergeGrid, tiles)) + 1;
#define IFRIT_MERGE_LAUNCH(SN)                                                                                     \
    hipLaunchKernelGGL(k_raster_merge<SN>, dim3(grid), dim3(256), 0, s, p, views, recs, slotOf, bins.waves,       \
                       bins.start, bins.cursor, q, visDepth, visSlot, visClass, ctr, st, out)
    switch (samples) {
        case 1: IFRIT_MERGE_LAUNCH(1); break;
        case 4: IFRIT_MERGE_LAUNCH(4); break;
        default: IFRIT_MERGE_LAUNCH(8); break;
    }
#undef IFRIT_MERGE_LAUNCH
}

}  // namespace ifrit_hip
