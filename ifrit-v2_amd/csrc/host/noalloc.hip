// The no-allocation draw (iftrDrawNoAlloc): the draw of the bound single
// target, from the caller's device-resident vertices and indices into the
// caller's device outputs, with every intermediate buffer carved out of one
// static device array.  It calls no hipMalloc or hipFree, so callers that
// cannot allocate (serving loops, harnesses that forbid it) can draw.
//
// The array `scratch` below is a device symbol: in host code its name is not
// a device address.  Its address on each device is looked up once with
// hipGetSymbolAddress (at iftrInit, with that device current) and only that
// address is used: as kernel arguments, for copies and for clears.  Every
// renderer on a GPU shares the GPU's array, and calls keep the last call's
// contents; the kernels clear what must start at zero, and calls that overlap
// on one GPU race.
#include <algorithm>
#include <cstring>
#include <mutex>

#include "../common/x86_fp.h"
#include "renderer.hpp"

namespace ifrit_hip {

static __device__ __align__(256) unsigned char scratch[IFHIP_NOALLOC_SCRATCH_BYTES];

namespace {

constexpr int kMaxDevices = 64;
std::mutex g_scratchMutex;
void* g_scratchAddr[kMaxDevices] = {};

constexpr int kTile = 16;

// Bump allocation of 256-byte aligned ranges inside the scratch array.
struct Arena {
    uint8_t* base;
    size_t cap;
    size_t used = 0;
    void* take(size_t n) {
        used = (used + 255) & ~(size_t)255;
        void* p = base + used;
        used += std::max<size_t>(n, 1);
        return p;
    }
    bool fits() const { return used <= cap; }
};

}  // namespace

// Looks up the scratch array's address on the current device (once per device).
bool noalloc_register_device(std::string* err) {
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= kMaxDevices) {
        *err = "no-allocation scratch: no current HIP device below index 64";
        return false;
    }
    std::lock_guard<std::mutex> lock(g_scratchMutex);
    if (g_scratchAddr[dev]) return true;
    void* p = nullptr;
    const hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    if (e != hipSuccess || !p) {
        *err = std::string("no-allocation scratch: hipGetSymbolAddress failed: ") + hipGetErrorString(e);
        return false;
    }
    g_scratchAddr[dev] = p;
    return true;
}

static void* noalloc_scratch_address(std::string* err) {
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= kMaxDevices) {
        *err = "no-allocation scratch: no current HIP device below index 64";
        return nullptr;
    }
    {
        std::lock_guard<std::mutex> lock(g_scratchMutex);
        if (g_scratchAddr[dev]) return g_scratchAddr[dev];
    }
    // a device other than the one current at iftrInit: look it up now
    if (!noalloc_register_device(err)) return nullptr;
    std::lock_guard<std::mutex> lock(g_scratchMutex);
    return g_scratchAddr[dev];
}

// The draw's tables, passed as kernel arguments, and its zeroed memory in one launch.
// Bound by the launch; two blocking copies and a memset in its place, with the copy of
// the counters after the draw, cost 40 us: a 256x256 ID draw 113 -> 69 us.
constexpr int kTableTextures = 96;
struct TableArgs {
    ViewDesc view;
    int first, textures;
    TexDesc tex[kTableTextures];
};
static_assert(sizeof(TableArgs) < 3072, "kernel arguments end at 4 KB");

static __global__ void __launch_bounds__(256) k_tables(TableArgs a, ViewDesc* view, TexDesc* tex, uint4* zero,
                                                       size_t words) {
    const size_t i = (size_t)blockIdx.x * 256 + threadIdx.x;
    if (i < words) zero[i] = make_uint4(0u, 0u, 0u, 0u);
    if (i < (size_t)a.textures) tex[a.first + i] = a.tex[i];
    if (i == 0 && a.first == 0) *view = a.view;
}

void TileRasterRenderer::drawNoAlloc(const IfritNoAllocDraw& d) {
    if (!initialized_) return setError("iftrDrawNoAlloc: call iftrInit first");
    if (!d.vertices || !d.indices || !d.depth) return setError("iftrDrawNoAlloc: vertices, indices and depth are required");
    if (!batch_.empty()) return setError("iftrDrawNoAlloc draws the single bound target: clear the view batch first");
    if (width_ <= 0 || height_ <= 0) return setError("iftrDrawNoAlloc: no render target set");
    if (width_ > 16384 || height_ > 16384) return setError("iftrDrawNoAlloc: render target larger than 16384 x 16384");
    if (hostVs_ || !vsBound_) return setError("iftrDrawNoAlloc needs a GPU vertex program");
    if (blend_.blendEnable) return setError("iftrDrawNoAlloc does not blend");
    if (polygonMode_ != 0) return setError("iftrDrawNoAlloc draws filled triangles only");
    if (gsBound_) return setError("iftrDrawNoAlloc does not run geometry programs");
    if (depthFunc_ < IF_COMPARE_OP_NEVER || depthFunc_ > IF_COMPARE_OP_ALWAYS)
        return setError("unknown depth function");
    if (d.numIndices < 0 || d.numVertices <= 0 || d.strideFloats <= 0)
        return setError("iftrDrawNoAlloc: bad vertex or index count");
    if (vs_.desc.kind == IFHIP_VS_CLIP_PASSTHROUGH ? d.strideFloats < 4 : d.strideFloats < 3)
        return setError("iftrDrawNoAlloc: vertex records too short for the vertex program");
    const bool shade = d.rgba8 && fsBound_ && fs_.desc.kind != IFHIP_FS_DEPTH_ONLY;
    if (shade) {
        const int k = fs_.desc.kind;
        if (k == IFHIP_FS_NEURAL && (!nnReady_ || textures_.size() < 3))
            return setError("the neural material has not been trained or its textures are not bound");
        if ((k == IFHIP_FS_GGX_LAYERED || k == IFHIP_FS_NEURAL) &&
            (textures_.size() < 3 || d.strideFloats < 11 || fs_.desc.offTangent + 3 > d.strideFloats))
            return setError("the layered-GGX and neural programs need three textures and a tangent");
    }
    const int ntri = d.numIndices / 3;
    if (samples_ == 1 && ntri >= (1 << 28)) return setError("too many triangles at 1 sample per pixel");
    std::string err;
    uint8_t* base = static_cast<uint8_t*>(noalloc_scratch_address(&err));
    if (!base) return setError(err);

    // everything the draw reads from the renderer's own buffers and sizes, restored on every exit
    DevBuf* const bufs[] = {&vtx_, &idx_, &recs_[0], &recs_[1], &recs_[2], &recs_[3], &recs_[4], &recs_[5],
                            &bary_, &binFront_, &slotOf_, &binCount_, &binStart_, &binCursor_, &binList_,
                            &ctr_, &groupBounds_, &clipList_, &statPart_, &items_, &tilePartial_,
                            &multiList_, &partials_, &visDepth_, &visSlot_, &visClass_, &rgba8_, &rgba32f_,
                            &texDesc_, &viewDev_, &tileView_, &order_, &viewCtr_, &swapped_};
    constexpr size_t kBufs = sizeof(bufs) / sizeof(bufs[0]);
    struct Restore {
        TileRasterRenderer& r;
        DevBuf* const* bufs;
        DevBuf saved[kBufs];
        unsigned caps[5];
        int ints[5];
        unsigned tiles, shadeTiles;
        size_t pixels;
        std::vector<ViewDesc> views;
        FrameBuffer* fb;
        bool floatOut;
        uint8_t* pool;
        // the counters of the draw before, which may not have been asked for yet, once it has ended
        bool ended = false, pending = false;
        HostCounters counters;
        Restore(TileRasterRenderer& rr, DevBuf* const* b) : r(rr), bufs(b) {
            for (size_t i = 0; i < kBufs; i++) saved[i] = *bufs[i];
            const unsigned c[5] = {r.clipCap_, r.binCap_, r.bigCap_, r.itemCap_, r.partialCap_};
            std::memcpy(caps, c, sizeof(caps));
            const int n[5] = {r.curTris_, r.nverts_, r.stride_, r.nidx_, r.boundsTris_};
            std::memcpy(ints, n, sizeof(ints));
            tiles = r.totalTiles_;
            shadeTiles = r.shadeTiles_;
            pixels = r.totalPixels_;
            views = r.viewDesc_;
            fb = r.fb_;
            floatOut = r.floatOut_;
            pool = r.texPool_;
        }
        ~Restore() {
            for (size_t i = 0; i < kBufs; i++) *bufs[i] = saved[i];
            r.clipCap_ = caps[0];
            r.binCap_ = caps[1];
            r.bigCap_ = caps[2];
            r.itemCap_ = caps[3];
            r.partialCap_ = caps[4];
            r.curTris_ = ints[0];
            r.nverts_ = ints[1];
            r.stride_ = ints[2];
            r.nidx_ = ints[3];
            r.boundsTris_ = ints[4];
            r.totalTiles_ = tiles;
            r.shadeTiles_ = shadeTiles;
            r.totalPixels_ = pixels;
            r.viewDesc_ = views;
            r.fb_ = fb;
            r.floatOut_ = floatOut;
            r.texPool_ = pool;
            r.ids_ = nullptr;
            r.keepSlots_ = true;
            r.weightBase_ = 0;
            if (ended) {
                *r.hostCtr_ = counters;
                r.reducePending_ = pending;
            }
        }
    } restore(*this, bufs);

    // sizes, as prepare() and layoutViews() set them for one view
    curTris_ = ntri;
    nverts_ = d.numVertices;
    stride_ = d.strideFloats;
    nidx_ = d.numIndices;
    boundsTris_ = 0;  // bounding the groups anew (3 to 5 us) costs what testing their triangles does
    fb_ = nullptr;
    floatOut_ = false;
    clipCap_ = std::max(4096u, (unsigned)(ntri / 8));
    const unsigned part = 1u << partShift_;
    binCap_ = std::max(1u << 20, (unsigned)std::min<size_t>(0xFFFFFFF0ull, (size_t)ntri * 6));
    bigCap_ = std::max(1024u, (unsigned)(ntri / 16));
    const int tilesX = (width_ + kTile - 1) / kTile, tilesY = (height_ + kTile - 1) / kTile;
    totalTiles_ = (unsigned)(tilesX * tilesY);
    shadeTiles_ = shade ? totalTiles_ : 0u;
    totalPixels_ = ((size_t)width_ * height_ + 63) & ~(size_t)63;
    itemCap_ = totalTiles_ + binCap_ / part + 1u;
    partialCap_ = std::max(256u, binCap_ / (8u * part));
    ViewDesc vd;
    std::memset(&vd, 0, sizeof(vd));
    std::memcpy(vd.mvp, vs_.desc.mvp, sizeof(vd.mvp));
    for (int k = 0; k < 3; k++) vd.camera[k] = fs_.desc.camera[k];
    vd.shade = shade ? 1 : 0;
    vd.width = width_;
    vd.height = height_;
    vd.tilesX = tilesX;
    vd.tilesY = tilesY;
    vd.invW = 1.0f / (float)width_;  // TileRasterRenderer.cpp:59-60
    vd.invH = 1.0f / (float)height_;
    viewDesc_.assign(1, vd);

    // the scratch layout: every buffer of the draw except the caller's inputs and outputs
    const size_t slots = (size_t)ntri + clipCap_, tiles = totalTiles_, px = (size_t)width_ * height_;
    const size_t groups = vs_.desc.kind == IFHIP_VS_TRANSFORM ? (size_t)(ntri + kGroupTris - 1) / kGroupTris : 0;
    Arena A{base, (size_t)IFHIP_NOALLOC_SCRATCH_BYTES};
    auto put = [&](DevBuf& b, size_t n) {
        b.ptr = A.take(n);
        b.bytes = n;
    };
    // first what starts at zero: counters, the tile maps (all view 0), the tile counts
    put(ctr_, sizeof(DeviceCounters));
    put(viewCtr_, sizeof(ViewCounters));
    put(tileView_, std::max<size_t>(1, tiles) * 2);
    put(binCount_, tiles * 8);
    const size_t zeroed = A.used;
    put(viewDev_, sizeof(ViewDesc));
    put(texDesc_, std::max<size_t>(1, textures_.size()) * sizeof(TexDesc));
    put(groupBounds_, std::max<size_t>(1, groups) * 32);
    for (int k = 0; k < 6; k++) put(recs_[k], slots * 16);
    // 16 bytes a vertex and 48 a record slot are set aside for the fans' vertex weights and the
    // geometry kernel's outputs, which never need more: what a draw may hold does not depend on how
    // they are laid out
    const size_t weights = ((size_t)clipCap_ * 32 + 255) & ~(size_t)255;
    put(bary_, weights);
    weightBase_ = (unsigned)ntri;  // no pixel is shaded that keeps an earlier draw's slot
    put(binFront_, std::max(frontBytes(), (size_t)nverts_ * 16 + slots * 48 + std::max<size_t>(1, groups) - weights));
    put(slotOf_, (size_t)std::max(1, ntri) * 4);
    if (needSwapFlags()) put(swapped_, slots);
    put(clipList_, (size_t)clipCap_ * 4);
    put(statPart_, (2 * (size_t)rasterGrid() + 2) * 8);
    put(items_, (size_t)itemCap_ * 16);
    put(tilePartial_, tiles * 4);
    put(multiList_, tiles * 4);
    put(partials_, (size_t)partialCap_ * 256 * samples_ * 8);
    put(binStart_, tiles * 4);
    put(binCursor_, tiles * 4);
    put(binList_, (size_t)binCap_ * 4);
    put(visSlot_, px * samples_ * 4);
    // the order takes what the coverage classes, which such a draw does not keep, and a map of
    // shading tiles took
    const size_t shadeMap = shade ? (size_t)((width_ + shadeTile_ - 1) / shadeTile_) * ((height_ + shadeTile_ - 1) / shadeTile_) : 1;
    put(order_, std::max(tiles * 8, px + 2 * shadeMap));
    if (!A.fits())
        return setError("iftrDrawNoAlloc: the draw needs " + std::to_string(A.used) + " bytes of scratch; the "
                        "no-allocation entry point holds " + std::to_string((size_t)IFHIP_NOALLOC_SCRATCH_BYTES));
    // the caller's inputs and outputs
    vtx_.ptr = const_cast<float*>(d.vertices);
    vtx_.bytes = (size_t)d.numVertices * d.strideFloats * 4;
    idx_.ptr = const_cast<int32_t*>(d.indices);
    idx_.bytes = (size_t)d.numIndices * 4;
    visDepth_.ptr = d.depth;
    visDepth_.bytes = px * samples_ * 4;
    rgba8_.ptr = d.rgba8;
    rgba8_.bytes = d.rgba8 ? px * 4 : 0;
    rgba32f_ = DevBuf{};

    // tables: the view, its tile maps (all view 0), the texture descriptors
    if (!ok(hipStreamSynchronize(stream_), "iftrDrawNoAlloc")) return;
    restore.counters = *hostCtr_;
    restore.pending = reducePending_;
    restore.ended = true;
    std::vector<TexDesc> td(std::max<size_t>(1, textures_.size()));
    texPool_ = nullptr;
    for (const TextureSlot& t : textures_)
        if (!texPool_ || t.dev < texPool_) texPool_ = t.dev;
    for (size_t i = 0; i < textures_.size(); i++) {
        const TextureSlot& t = textures_[i];
        td[i] = TexDesc{};
        td[i].base = (unsigned long long)(t.dev - texPool_);
        td[i].width = t.width;
        td[i].height = t.height;
        td[i].levels = t.levels;
        td[i].layers = t.layers;
    }
    for (size_t i = 0; i < td.size(); i += kTableTextures) {
        TableArgs a;
        a.view = vd;
        a.first = (int)i;
        a.textures = (int)std::min<size_t>(kTableTextures, td.size() - i);
        std::memcpy(a.tex, td.data() + i, a.textures * sizeof(TexDesc));
        const size_t words = i == 0 ? (zeroed + 15) / 16 : 0;
        hipLaunchKernelGGL(k_tables, dim3((unsigned)std::max<size_t>(1, (words + 255) / 256)), dim3(256), 0, stream_, a,
                           viewDev_.as<ViewDesc>(), texDesc_.as<TexDesc>(), reinterpret_cast<uint4*>(base), words);
    }
    ids_ = d.primIds;
    keepSlots_ = false;
    reducePending_ = !drawsKeys(true);
    enqueue(true);
    if (!ok(hipGetLastError(), "kernel launch")) return;
    if (!finish(true, d.numIndices))
        setError("iftrDrawNoAlloc: the frame overflowed its scratch buffers (clip, bin or raster queue); the "
                 "outputs are incomplete");
}

}  // namespace ifrit_hip
