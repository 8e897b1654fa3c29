// Device-side data layout and launch interface of the MI355X tile rasterizer.
//
// A draw renders a batch of views (one or more) of the same vertex and index
// data; every stage is one launch over all views.  HBM layout per draw
// (V vertices, T input triangles, N views, SV = T + clipCap record slots per
// view, S samples):
//   views       ViewDesc[N]               per-view camera, size and bases
//   tileView    ushort[tiles]             view of each 16x16 tile (tiles of all views)
//   order       uint[2][tiles]            the shaded views' tiles, longest lists first (ShadeOrder)
//   clip        float4[N][V]              vertex stage output (point and line modes; triangle draws
//                                         transform in the geometry kernel)
//   recs        TriRecs, N * SV slots     assembled triangles; in view v, slot v*SV + prim
//                                         for unclipped triangles, v*SV + T + k for clip fans
//   bary        float4[2 * slots]         vertex-weight bases bx, by of the slots whose record says that it
//                                         has its own (kOwnWeights): clip fans, points and lines (shading only)
//   waves       WaveInfo[N][waves]        per 64 triangles, what the geometry kernel made of them
//   entry       uint2, uint4[N][64 waves] per triangle, its bin entries or tile rectangle (WaveInfo)
//   fanBox      uint2[N][clipCap]         tile rectangle of each clip fan
//   slotOf      uint[N][T]                first fan slot of each clipped primitive (its fans follow)
//   binCnt      uint2[tiles]              entries counted: triangles of up to four tiles, others (zero
//                                         after the plan, then marks of tiles with NaN depths)
//   binStart/binCursor  uint[tiles]       a tile's list; after binning the cursor is its end
//   binList     uint[binCap]              slot | 0x80000000 when the tile is fully covered
//   visId/visDepth/visSlot  [pixels * S]  per-sample winner; views one after another, pixels
//                                         row-major within a view, samples innermost
//   rgba8       uchar4[pixels]            resolved colour
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "neural.h"

namespace ifrit_hip {

// One assembled triangle for coverage and depth (6 x 16 bytes):
//   q0 = e1.xyz, e2.x   q1 = e2.yz, e3.xy
//   q2 = e3.z, key, pixel box lo, hi (common/pixel_box.h: no sample outside it is covered)
//   f1, f2, f3 = interpolation bases (x, y, z) and vz = (z/w) * w.
// key = prim * 4 + fan orders fragments the way the reference's per-tile
// sort by originalPrimitive does (TileRasterWorker.cpp:1244-1258).
struct __align__(16) TriRec {
    float4 q0, q1, q2;
    float4 f1, f2, f3;
};

// The pixel box's high end of a record with vertex weights of its own (clip fans, which no box
// bounds, points and lines): beyond every target, and no box of an unclipped triangle ends there.
constexpr unsigned kOwnWeights = 0xfffeffffu;

// Records are stored as six float4 streams (structure of arrays) so that a
// wave's stores and the tile loader's gathers are 16-byte accesses.
struct TriRecs {
    float4 *q0, *q1, *q2, *f1, *f2, *f3;
};

// One view of a draw.  View v owns tiles [tileBase, tileBase + tilesX *
// tilesY), record slots [slotBase, slotBase + SV), slotOf entries
// [primBase, primBase + T), the geometry waves [v * waves, (v + 1) * waves) and pixels [pixBase, pixBase + width * height).
struct ViewDesc {
    float mvp[16];
    float camera[3];
    int shade;                   // 1: the fragment program runs for this view
    int width, height, tilesX, tilesY;
    float invW, invH;            // 1 / width, 1 / height (TileRasterRenderer.cpp:59-60)
    unsigned tileBase;           // first 16x16 tile
    unsigned slotBase;           // first record slot (v * SV)
    unsigned primBase;           // first slotOf entry (v * T)
    unsigned long long pixBase;  // first pixel of the view's outputs
};

// Per-view counters, one 128-byte line each so that the views' atomics do not
// share a line.  The first two are counted by the geometry and clip kernels;
// the tile plan moves them to the last two, which later kernels read, and
// leaves zeros for the next draw.
struct ViewCounters {
    unsigned fanLive;   // clip fans so far
    unsigned clipLive;  // triangles found to cross w = 0 so far
    unsigned fans;      // clip fans of the draw
    unsigned clipIn;    // triangles of the draw crossing w = 0
    unsigned pad[28];
};

// What the geometry kernel made of the 64 triangles of one wave (triangles
// 64 w .. 64 w + 63 of a view).  A triangle in `single` lies in one tile: its
// entry is (tile | full << 31, rank in the tile's list); one in `few` spans two
// to four, (first tile, rank there) and in entry1 the ranks in the others and
// its FewTiles; one in `multi` spans more: (x0 | y0 << 16, x1 | y1 << 16),
// view-local tiles.  `clipped` triangles crossed w = 0 (slotOf names their
// first fan).
struct __align__(8) WaveInfo {
    unsigned long long single, few, multi, clipped;
    unsigned made;  // triangles assembled (clip fans not counted)
    unsigned pad;
};

// A rectangle of up to four tiles in entry1.w: columns - 1 in bits 0-1, tiles
// in bits 2-4, and from bit 8 on two bits per tile, row by row: its
// classification (dev::tile_class).
__host__ __device__ inline unsigned few_tiles(int cols, int area) { return (unsigned)(cols - 1) | ((unsigned)area << 2); }

// Waves of the geometry kernel per view: whole workgroups of four.
constexpr int kGeomBlock = 256;
__host__ __device__ inline unsigned geom_waves(int ntri) {
    const unsigned b = (unsigned)((ntri + kGeomBlock - 1) / kGeomBlock);
    return (b ? b : 1u) * (kGeomBlock / 64);
}

struct Views {
    const ViewDesc* desc;
    const unsigned short* tileView;   // view of each 16x16 tile
    ViewCounters* ctr;
    int count;
    unsigned slotsPerView;            // SV = T + clipCap
    unsigned waves;                   // geometry waves per view
};

// Scissor rectangles (SetScissors / setScissorTestEnable of the CUDA renderer,
// TileRasterRendererCuda.h:101-102): a pixel (x, y) of a view passes when
// count is 0 or it lies in one rectangle, r.x <= x <= r.x + r.z and
// r.y <= y <= r.y + r.w (TileRasterCoreInvocationCuda.cu:1699-1711).  A
// draw leaves pixels that fail untouched: visibility, depth and colour
// (its clear included, as the CUDA clear kernels are scissored,
// TileRasterCoreInvocationCuda.cu:3336-3424).
constexpr int kMaxScissors = 8;
struct Scissor {
    int count;            // 0: every pixel passes
    const float4* rects;  // device memory: (x, y, width, height) per rectangle
};

// IfritCullMode (include/ifrit/softgraphics/engine/base/Constants.h:29-35).
enum CullMode { kCullNone = 0, kCullFront = 1, kCullBack = 2, kCullFrontAndBack = 3 };

// Per-view fields (width, height, tiles, invW, invH) are filled in by the
// kernels from the view's ViewDesc.
struct SetupParams {
    int width, height;
    int tilesX, tilesY;
    int ntri, nverts;
    int cullMode;       // IfritCullMode: 0 none, 1 front, 2 back (the CPU path), 3 front and back
    unsigned char* swapped;  // per record slot, cull modes none and front: 1 when the triangle was set
                             // up with its first and third vertex exchanged (null for back)
    int msaa;           // 1 disables the small-triangle cull
    unsigned clipCap;   // capacity for clip fan triangles and for triangles to clip
    unsigned weightBase;  // the slot whose vertex weights `bary` starts with
    float invW, invH;   // 1 / width, 1 / height (TileRasterRenderer.cpp:59-60)
    float invTileWidth; // ApproxReciprocal(16.0f) (TileRasterWorker.cpp:499)
    int rcpModel;       // ifx::RcpModel: whose RCPPS the reciprocals of w and of the area reproduce
    // object-space bounds of each group of kGroupTris triangles (null: no group culling)
    const float4* groupBounds;
    int groups;
    unsigned bigCap;
    int bigThreshold;   // triangles spanning more tiles are binned by whole workgroups
};

// Vertex input of the geometry kernel: clipAt < 0 transforms a record's first
// three floats by each view's matrix, otherwise the record holds the clip
// position at float clipAt.
struct VertexInput {
    const float* vtx;
    int stride, clipAt;
};

// Binning buffers (see the layout above).
struct BinBufs {
    uint2* entry;
    uint4* entry1;
    WaveInfo* waves;
    uint2* fanBox;
    uint4* big;  // deferred triangles: slot, tile rectangle (as in entry), view
    unsigned long long* made;  // triangles assembled: kMadeSums sums of the scatter workgroups
    unsigned* cnt;
    unsigned *start, *cursor, *list;
};
// The scatter's workgroups add to as many sums as spread their atomics, a 128-byte line each.
constexpr int kMadeSums = 64, kMadeStride = 16;

// Slots of the clip fans.  Where a view has few triangles to clip, each takes as many slots as it can
// have fans, in the order of the triangles, so that the same triangles leave their fans in the same
// slots: a pixel that a later draw without clear leaves alone keeps its slot.  Ranking one
// against all others costs n^2 / 64 comparisons a view; above kClipRanked, or where the capacity is
// short, the fans take slots as they come.
constexpr unsigned kFanSlots = 3;  // at most three vertices kept and two made, for edges that change sign
constexpr unsigned kClipRanked = 4096;
__host__ __device__ inline bool clips_ranked(unsigned clips, unsigned clipCap) {
    return clips <= kClipRanked && kFanSlots * clips <= clipCap;
}
// Clip slots of a view that may hold a fan.
__host__ __device__ inline unsigned fan_extent(unsigned clips, unsigned fans, unsigned clipCap) {
    return clips_ranked(clips, clipCap) ? kFanSlots * clips : fans < clipCap ? fans : clipCap;
}

// Triangles per culling group (one workgroup of the geometry kernel).
constexpr int kGroupTris = kGeomBlock;

struct BinParams {
    int tiles;          // tiles of all views
    int grid;           // workgroups of the scatter launch
    int regions;        // geometry waves a scatter wave takes at a time (1 .. 64)
    int ntri;
    unsigned clipCap;
    unsigned binCap;
    unsigned bigCap;
};

struct RasterParams {
    int depthFunc;
    int clear;
    float clearDepth;    // depth a cleared sample starts from (0x7f7f7f7f in the CPU path)
    int tagging;         // 1 spp: the tagging mode's depth expressions (class_depth)
    int depthWrite;      // the fragment program stores depth * depthScale + depthBias after the test
    float depthScale, depthBias;
    Scissor scissor;
    unsigned binCap, ntri;
    // cleared draws with a depth function other than LESS that is a minimum of keys (raster.hip
    // general_key)
    int general, last;
    unsigned keyXor, keyMask;
    // primitive ID per sample of a cleared draw, written with the depth (null: the caller expands slots
    // itself); idsWide: the array starts on a 16-byte line
    uint32_t* ids;
    int idsWide;
    float sx[8], sy[8];  // sample offsets from the pixel corner
};

struct TexDesc {
    unsigned long long base;  // byte offset of level 0 in the texture pool
    int width, height, levels, layers;
    // levels follow level 0 packed, each max(1, width >> l) x max(1, height >> l) texels per
    // layer, the layers of a level one after another (a cube map has six, +x -x +y -y +z -z);
    // the sampler computes the offsets from width, height and layers
};

// Sampler state of a program (IfritSamplerT, include/ifrit/softgraphics/engine/base/Structures.h:52-61)
// beyond the level-of-detail choice: addressing per axis, the filter within a level and the border.
enum AddressMode { kAddrRepeat = 0, kAddrMirroredRepeat = 1, kAddrClampToEdge = 2, kAddrClampToBorder = 3,
                   kAddrMirrorClampToEdge = 4 };
struct SamplerMode {
    int addrU, addrV;  // AddressMode
    int nearest;       // 1: nearest texel within a level (IF_FILTER_NEAREST), 0: bilinear
    unsigned border;   // RGBA8 border colour: 0xff000000 opaque black, 0xffffffff opaque white
};

struct ShadeParams {
    int samples;
    int program;
    int stride, offWorld, offNormal, offUv, offTangent;
    int trisPerMaterial;
    int sampler, maxAniso;
    int numTextures;
    float ambient, kd, ks, shininess;
    int numLights;
    float lightPos[4][4];
    float lightColor[4][4];
    int writeFloat;          // also write RGBA32F
    int ntri;                // view-local slots >= ntri are clip fans with their own bx, by
    unsigned weightBase;     // the slot whose weights `bary` starts with
    unsigned lastTri, lastVertex;  // the last ones that the index and vertex buffers have room for
    int shadeTile;           // side of a square of as many pixels as one wave shades (8, 16 or 32),
                             // its 8x8 sub-tiles in turn
    int cleared;             // the draw cleared its targets
    NeuralShadeParams neural;  // programs 4 (neural material) and 5 (training features)
    const unsigned char* swapped;  // per record slot: vertices 0 and 2 exchanged by setup (null: none)
    float clearColor[4];     // colour of samples no triangle covers (the resolve weighs them)
    float clearDepth;        // depth a cleared pixel starts from (blending draws)
    int depthWrite;          // blending draws: the program stores depth * depthScale + depthBias
    float depthScale, depthBias;
    Scissor scissor;
    SamplerMode samp;        // addressing and filter of the program's lookups
    int sampGeneric;         // 1: samp differs from repeat + bilinear (the sampled-kernel variant runs)
    float lod;               // cube-map program: the level of detail of its lookups
};

// Blend factors, each encoded (c0, c1, c2, c3) as the reference does
// (TileRasterRenderer.cpp:212-333): colour source, colour destination, alpha
// source, alpha destination.
struct BlendCoefs {
    float sc[4], dc[4], sa[4], da[4];
};

// Status word bits raised by the kernels; checked by the host after a frame.
enum StatusBits : unsigned {
    kStatusClipOverflow = 1u,
    kStatusBinOverflow = 2u,
    kStatusBigOverflow = 4u,
    kStatusBadIndex = 8u,
    kStatusRasterOverflow = 16u,
};

// Per-workgroup statistics (no same-address atomics in the hot kernels);
// k_finalize reduces them into DeviceCounters.
struct StatPartials {
    unsigned long long* made;            // BinBufs::made
    unsigned long long* rasterFrags;     // one per raster workgroup
    unsigned long long* rasterCovs;      // one per raster workgroup
    int rasterBlocks;
};

// Raster work items are drained through this many counters, one per XCD:
// stream k holds items k, k + kItemStreams, ... and is taken by the
// workgroups with blockIdx.x % kItemStreams == k (one XCD's), so the claims
// of the persistent raster spread over separate lines instead of one.
constexpr int kItemStreams = 8;

// Totals of the tile plan (DeviceCounters::tot).
enum PlanTotal { kTotEntries = 0, kTotLong, kTotShort, kTotPartials, kTotMulti, kTotEmpty, kTotCount = 6 };

// Counters written by the kernels (device memory).  `live` is counted by the
// geometry and clip kernels; the tile plan moves it to the fields above and
// leaves zeros for the next draw, so that a draw needs no clearing launch.
// The totals and item heads are cleared by the geometry kernel.
struct DeviceCounters {
    unsigned status;
    unsigned bigCount;
    unsigned clipMax;    // largest per-view fan or clip count so far (sizes clipCap on overflow)
    unsigned long long assembled;
    alignas(16) unsigned order[4];  // tiles in ShadeOrder's classes
    unsigned tot[8];     // PlanTotal: list entries, items of more than kRasterPass entries (front of the
                         // item array), other items, partial blocks, tiles cut into parts, empty tiles
    struct alignas(128) Live {
        unsigned status, bigCount, clipMax, fans;  // fans: fan triangles assembled
    } live;
    alignas(128) unsigned itemHeads[kItemStreams][32];  // next item of each stream, one 128-byte line each
};

// A finished draw's counters as the host reads them (pinned memory written by
// finalize_block: a copy of DeviceCounters after the stream's end cost a second round trip).
struct HostCounters {
    unsigned long long fragments, coveredSamples, assembled;
    unsigned status, clipCount, bigCount, clipMax;
    unsigned tot[8];  // PlanTotal
};

// Raster work: a work item covers at most 1 << partShift list entries of
// one tile (256 to 1024), taken in passes of kRasterPass entries (the LDS
// capacity).
constexpr int kRasterPass = 128;
// Tiles per workgroup of the tile-plan kernel (one per thread).
constexpr int kPlanTiles = 256;
constexpr int kRasterPartShift = 9;

// Raster work: items {tile, first list entry, entries, partial block or
// ~0u} drained through DeviceCounters::itemHeads; per tile the first partial
// block of a tile cut into several items (-1 otherwise); the list of such
// tiles from the front and of the empty tiles from the back (index `tiles` - 1
// down); partial key blocks of 256 * samples keys each.
struct RasterQueue {
    uint4* items;
    int* tilePartial;
    unsigned* multiList;
    unsigned long long* partials;
    unsigned itemCap, partialCap, binCap;
    int grid;         // raster workgroups
    int mergeGrid;    // half the merge workgroups
    unsigned *orderA, *orderB;  // ShadeOrder's arrays, null where nothing is shaded
    int orderByLength;          // classes 0 and 1 are used
    int partShift;
    int tileThreads;  // threads per tile at 1 sample per pixel: 64 or 256
    int wide;         // the raster takes passes of 2 kRasterPass entries: no more triangles than one
                      // pass of kRasterPass per workgroup
};

// The order in which tiles are shaded: those whose lists are empty (class 3) last and,
// at 8 samples, those of more than 4 kRasterPass entries (0) and of more than
// kRasterPass (1) before the others (2), so that none of them is started last.  Class 0
// fills `a` from the front and class 3 from its back, classes 1 and 2 `b`; count[] tells
// how many each holds.  a is null where the tiles are taken as they are numbered
// (point and line modes).
//
// List lengths order the work only where a pixel can hold many triangles; at one
// sample it holds one and its cost is its texture taps, and the neighbours that no
// longer follow each other cost the caches.  By length or not, in us, for 1.3M
// triangles at 1920x1080, the same at 640x480, 4.2M half-pixel ones, and 82k at 1280x720:
// 8 samples 107 or 114, 59 or 64, 36 or 40, 41 or 42; 4 samples 81 or 84, 41 or 42, 27 or
// 28, 29 or 29; 1 sample 55 or 54, 24 or 24, 25 or 25, 18 or 18, and 34 views 109 or 103.
// The gain follows the length of the lists; at 4 samples the line leaves some of it.
struct ShadeOrder {
    const unsigned *a, *b;
    const uint4* count;
    int tiles;   // tiles of all views: entries of a and of b
    int shaded;  // tiles of shaded views
};

// Launch wrappers.  launch_vertex (point and line modes) writes every view's
// clip positions and clears the counters; launch_reset only clears them.
void launch_vertex(const VertexInput& in, int nverts, const Views& views, float4* clip, DeviceCounters* ctr,
                   hipStream_t s);
void launch_group_bounds(const float* vtx, int stride, int nverts, const int* idx, int ntri, float4* bounds,
                         hipStream_t s);
void launch_reset(const Views& views, DeviceCounters* ctr, hipStream_t s);
// Vertex transform, triangle setup and the bin counts, then the triangles that
// cross w = 0 and those deferred by the bin count.
void launch_geometry(const SetupParams& p, const Views& views, const VertexInput& in, const int* idx, TriRecs recs,
                     float4* bary, const BinBufs& bins, unsigned* slotOf, unsigned* clipList, DeviceCounters* ctr,
                     hipStream_t s);
void launch_finalize(StatPartials st, const Views& views, DeviceCounters* ctr, HostCounters* out, hipStream_t s);
// The tile plan and the scatter into the tile lists.
void launch_bin(const BinParams& p, const Views& views, TriRecs recs, const BinBufs& bins, const RasterQueue& q,
                DeviceCounters* ctr, hipStream_t s);
void launch_raster(const RasterParams& p, const Views& views, int samples, TriRecs recs, const unsigned* slotOf,
                   const BinBufs& bins, const RasterQueue& q, int tiles, float* visDepth, uint32_t* visSlot,
                   uint8_t* visClass, StatPartials st, DeviceCounters* ctr, hipStream_t s);
void launch_raster_merge(const RasterParams& p, const Views& views, int samples, TriRecs recs, const unsigned* slotOf,
                         const BinBufs& bins, const RasterQueue& q, float* visDepth, uint32_t* visSlot,
                         uint8_t* visClass, int tiles, DeviceCounters* ctr, StatPartials st, HostCounters* out,
                         hipStream_t s);
// Depth functions that are no minimum: each tile's list in primitive order, folded
// per pixel (replaces launch_raster and launch_raster_merge); with nanTilesOnly the tiles in which
// they met a NaN depth (after launch_raster_merge of a general draw).
void launch_raster_ordered(const RasterParams& p, const Views& views, int samples, TriRecs recs,
                           const BinBufs& bins, const RasterQueue& q, int tiles, float* visDepth, uint32_t* visSlot,
                           uint8_t* visClass, StatPartials st, bool nanTilesOnly, DeviceCounters* ctr,
                           hipStream_t s);
// IDs from record slots: the primitive key >> 2, or for point and line records (polygon) the key's
// triangle * 3 + its point or edge.
void launch_slot_to_prim(const uint32_t* visSlot, TriRecs recs, size_t n, uint32_t* visId, hipStream_t s,
                         bool polygon = false);
void launch_shade(const ShadeParams& p, const Views& views, const ShadeOrder& order, TriRecs recs, const float4* bary, const uint32_t* visSlot,
                  const float* vtx, const int* idx, const TexDesc* tex, const uint8_t* texPool, uchar4* rgba8,
                  float4* rgba32f, hipStream_t s);

// Blending, 1 sample per pixel: the ordered traversal with the depth test, each
// passing fragment shaded and blended in primitive order (replaces the raster,
// merge and shade launches).
void launch_blend_ordered(const ShadeParams& p, const BlendCoefs& b, int depthFunc, int clear,
                          const Views& views, TriRecs recs, const float4* bary, const float* vtx, const int* idx,
                          const TexDesc* tex, const uint8_t* texPool, const BinBufs& bins,
                          const RasterQueue& q, int tiles, float* visDepth, uint32_t* visSlot, uint8_t* visClass,
                          uchar4* rgba8, float4* rgba32f, StatPartials st, DeviceCounters* ctr, hipStream_t s);

// Point (mode 2) and line (mode 1) polygon modes, one sample per pixel (polygon.hip):
// candidates per pixel meet in keys (order_key(depth) << 32 | primitive id),
// then the resolve writes depth and record slot where the nearest one is below
// the stored depth.  Record slots: the index position of a point, 3 * triangle
// + edge of a line.
struct PolyParams {
    int mode;
    int width, height;
    int nidx, nverts;
    int clear;
    float clearDepth;
    unsigned long long* keys;  // width * height
};
void launch_polygons(const PolyParams& p, const float4* clip, const int* idx, TriRecs recs, float4* bary,
                     float* visDepth, uint32_t* visSlot, uint8_t* visClass, StatPartials st, DeviceCounters* ctr,
                     int grid, hipStream_t s);

// The built-in meshlet program of DrawMeshTasks (mesh.hip): work groups first .. first + groups - 1,
// meshlet m owning vertices vo[m] .. vo[m + 1] - 1 and indices io[m] .. io[m + 1] - 1 (local to the
// meshlet); emitted vertices are (clip xyzw, record) at vo[m] - vertexBase, indices at
// io[m] - indexBase.
struct MeshParams {
    float mvp[16];
    int recordFloats;
    int first, groups;
    int vertexBase, indexBase;
};
void launch_mesh_expand(const MeshParams& p, const float* records, const int* indices, const int* vo, const int* io,
                        float* outVtx, int* outIdx, DeviceCounters* ctr, hipStream_t s);
// The built-in geometry program: triangle t's vertices, transformed (or passed through) and moved
// by offset, emitted as records (input record, then clip xyzw) 3t .. 3t + 2, indices 3t .. 3t + 2.
struct GeometryParams {
    float mvp[16];
    float offset[4];
    int passthrough;
    int stride;        // floats per input vertex record
    int nverts, ntri;
};
void launch_geometry_expand(const GeometryParams& p, const float* vtx, const int* idx, float* outVtx, int* outIdx,
                            DeviceCounters* ctr, hipStream_t s);

// Texture helpers (texture.hip).
// Order-independent 64-bit digest of n words (equal buffers give equal digests).
void launch_digest(const uint32_t* data, size_t n, unsigned long long* out, hipStream_t s);
void launch_fbm_texture(uint8_t* level0, int size, unsigned seed, hipStream_t s);
void launch_mip_level(const uint8_t* src, int sw, int sh, uint8_t* dst, int dw, int dh, hipStream_t s);
// blitImage (TileRasterImageOpInvocationsCuda.cu:36-131) between RGBA8 levels: destination texel
// (dx0 + x, dy0 + y) for x < dx1 - dx0, y < dy1 - dy0 reads the source at
// (x / (dx1 - dx0) (sx1 - sx0) + sx0, likewise y); linear: bilinear with the right and lower
// neighbours clamped to the source level, on the 0..255 values, rounded half up; nearest:
// the texel at the rounded coordinate, clamped.
struct BlitArgs {
    int sw, sh, dw, dh;               // level sizes
    unsigned sx0, sy0, sx1, sy1;      // source region
    unsigned dx0, dy0, dx1, dy1;      // destination region
    int linear;
};
void launch_blit(const uint8_t* src, uint8_t* dst, const BlitArgs& a, hipStream_t s);

}  // namespace ifrit_hip
