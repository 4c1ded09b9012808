// api.hip — the C ABI (include/rgrt.h) over the HIP kernels.
#include <algorithm>
#include <cstdio>
#include <cstring>
#include <memory>
#include <mutex>
#include <string>
#include <vector>

#include "rgrt_internal.h"

namespace rgrt {
uint32_t trace_spill_words_per_thread();
uint32_t trace_block_size();
uint32_t trace_resident_blocks();
void launch_trace_queue_impl(hipStream_t s, const TraceScene& sc, const WavefrontState& st, int cur, uint32_t gridBlocks,
                             int32_t* spill, uint32_t* hostSlot, bool ahead);
void launch_trace_rays_impl(hipStream_t s, const TraceScene& sc, const rgrt_ray* rays, uint32_t n, uint32_t cullMask,
                            rgrt_hit* hits, const InstanceShade* inst, int32_t* spill, uint32_t gridBlocks, uint32_t simds,
                            uint32_t* fetch);
} // namespace rgrt

using namespace rgrt;

namespace {

struct BlasRec {
    rgrt_blas_desc desc{};
    Node* nodes = nullptr;  // canonical binary tree
    Node4* wide = nullptr;  // the 4-wide tree (full-precision boxes)
    Node4q* wideq = nullptr; // its compressed form, which the traversal walks
    uint32_t* numWide = nullptr;
    Tri* tris = nullptr;
    uint32_t* leafPrim = nullptr;
    bool valid = false;
};

template<typename T>
void dev_free(T*& p)
{
    if(p) (void)hipFree((void*)p);
    p = nullptr;
}

// Frees p and allocates it anew. A buffer's recorded capacity is set to zero
// before it grows: if memory runs out, p is null, the call reports it, and the
// next call allocates again instead of handing the null to a kernel.
template<typename T>
void dev_alloc(T*& p, size_t count)
{
    dev_free(p);
    check(hipMalloc((void**)&p, std::max<size_t>(count, 1) * sizeof(T)));
}

} // namespace
struct rgrt_ctx;
namespace {

// Geometry, materials and BLASes. Contexts created with rgrt_create_shared
// share one SceneData (each keeps its own TLAS, images, wavefront state and
// stream, so their frames overlap on the GPU); a change of the scene first
// waits for every sharing context's stream.
struct SceneData {
    rgrt_vertex* vb = nullptr;
    uint64_t nv = 0;
    uint32_t* ib = nullptr;
    uint64_t ni = 0;
    rgrt_material* mats = nullptr;
    uint32_t nm = 0;
    ShadeTri* srec = nullptr; // shading record per triangle of the index buffer (ni / 3)
    std::vector<BlasRec> blas;
    DevBlas* dBlasTable = nullptr;
    float4* dBlasRoot = nullptr;
    uint32_t blasCap = 0;
    std::mutex m;
    std::vector<rgrt_ctx*> users; // the contexts sharing it

    ~SceneData()
    {
        for(auto& b: blas) {
            dev_free(b.nodes);
            dev_free(b.wide);
            dev_free(b.wideq);
            dev_free(b.numWide);
            dev_free(b.tris);
            dev_free(b.leafPrim);
        }
        dev_free(vb);
        dev_free(ib);
        dev_free(srec);
        dev_free(mats);
        dev_free(dBlasTable);
        dev_free(dBlasRoot);
    }
    void add_user(rgrt_ctx* c)
    {
        std::lock_guard<std::mutex> g(m);
        users.push_back(c);
    }
    void remove_user(rgrt_ctx* c)
    {
        std::lock_guard<std::mutex> g(m);
        users.erase(std::remove(users.begin(), users.end(), c), users.end());
    }
};

// Bound on the rays one pixel can trace one after another for one sample
// when every material reflects and refracts with rayConsumption 1:
// B(r) = (R - r) shadow-chain rays + 2 * (1 + B(r + 1)), B(R) = 0.
uint32_t max_sequential_rays(int maxRec)
{
    uint64_t b = 0;
    for(int r = maxRec - 1; r >= 0; --r) b = (uint64_t)(maxRec - r) + 2 * (1 + b);
    return (uint32_t)std::min<uint64_t>(b + 1, 1u << 20);
}

} // namespace

struct rgrt_ctx {
    int device = 0;
    uint32_t flags = 0;
    hipStream_t stream = nullptr;
    std::string err;
    uint32_t numCUs = 256;

    std::shared_ptr<SceneData> sd; // geometry, materials, BLASes (possibly shared)

    uint32_t instCap = 0;
    uint32_t numInstances = 0;
    bool haveTlas = false;
    std::vector<uint32_t> tlasBlas; // BLAS per instance position of the last build
    // Two pinned staging buffers used in turn, each free again once the
    // upload from it has run (stageDone): the host prepares frame N + 1
    // while the GPU still works on frame N.
    rgrt_instance* hInstStage[2] = {nullptr, nullptr};
    hipEvent_t stageDone[2] = {nullptr, nullptr};
    hipEvent_t sceneEv = nullptr; // orders in-place scene writes against sharing contexts
    int stageIdx = 0;
    rgrt_instance* dInstIn = nullptr;
    Node* tlasNodes = nullptr;
    Node4* tlasWide = nullptr;
    Node4q* tlasWideq = nullptr;
    uint32_t* tlasNumWide = nullptr;
    uint32_t* tlasLeaf = nullptr;
    DevInstance* dInst = nullptr;
    InstanceShade* dShade = nullptr;
    float* dW2O = nullptr;
    float4* tlasRoot = nullptr;

    LbvhBuilder builder;

    rgrt_ubo ubo{};
    bool haveUbo = false;

    uint32_t w = 0, h = 0;
    Images img;
    WavefrontState st;
    int32_t* spill = nullptr;
    size_t spillBytes = 0;
    uint32_t traceGrid = 0, shadeGrid = 0, drainGrid = 0;
    rgrt_tuning tuning{6, 5, 8, 4, 2, 1}; // measured on config 2 (1080p, 2M triangles)
    rgrt_sampling sampling{RGRT_SAMPLING_WHITTED, 0u, {0u, 0u}};
    hipEvent_t evDrainStart = nullptr, evDrainEnd = nullptr;
    bool lastDrained = false;

    // Graph frames in bands: the streams bands 1.. run on (band 0 runs on
    // `stream`), their fork and join events, and the frame's executable
    // graphs (instance upload and TLAS; each band's trace; the post passes).
    uint32_t bands = 1;
    hipStream_t bandStream[kMaxBands] = {};
    hipEvent_t bandFork = nullptr;
    hipEvent_t bandJoin[kMaxBands] = {};
    hipGraphExec_t preExec = nullptr, postExec = nullptr;
    hipGraphExec_t bandExec[kMaxBands] = {};
    uint32_t lastBands = 1;   // bands of the last traced frame (their counter blocks hold its statistics)
    uint32_t passStride = 0;  // per-band stride of the pass counts in hostCounts
    size_t spillWords = 0;    // spill words of one band

    // Grids from the tuning; the traversal spill region covers the larger of
    // the persistent traversal and drain grids (they never run at once), once
    // per band (the bands' launches run side by side).
    void apply_tuning()
    {
        // the traversal grid is persistent: blocks past what a CU holds would
        // start on their share when the others are done (4K at 4 samples with
        // six blocks per CU, five of them resident: 95.8 ms, clamped 86.0)
        tuning.traceBlocksPerCU = std::min(tuning.traceBlocksPerCU, trace_resident_blocks());
        traceGrid = numCUs * tuning.traceBlocksPerCU;
        shadeGrid = numCUs * tuning.shadeBlocksPerCU;
        drainGrid = numCUs * tuning.drainBlocksPerCU;
        bands = std::max<uint32_t>(1u, std::min(tuning.frameBands, kMaxBands));
        spillWords = std::max((size_t)traceGrid * trace_block_size() * trace_spill_words_per_thread(),
                              (size_t)drainGrid * drain_block_size() * drain_spill_words_per_thread());
        const size_t need = spillWords * bands * 4;
        if(need > spillBytes) {
            if(spill) {
                check(hipStreamSynchronize(stream));
                check(hipFree(spill));
                spill = nullptr;
                spillBytes = 0;
            }
            check(hipMalloc((void**)&spill, need));
            spillBytes = need;
        }
    }

    rgrt_ray* dRays = nullptr;
    rgrt_hit* dHits = nullptr;
    uint32_t rayCap = 0;
    uint32_t* rayFetch = nullptr; // chunk counter of the ray queries, error word of a context without images
    char* hRayIo = nullptr;       // pinned rays, hits and error word of small host queries (kPinnedRays),
    char* hRayIoDev = nullptr;    // and its device address, both from rgrt_create on
    size_t slotCap = 0;       // wavefront slots the slot arrays hold
    size_t sampleCap = 0;     // per-sample records the sample buffers hold
    uint32_t sampleGroups = 0; // most sample groups side by side (0: as many as fit)

    uint32_t* hostCounts = nullptr; // pinned, device-visible
    uint32_t* hostCountsDev = nullptr;
    uint32_t hostCountsCap = 0;
    std::vector<hipEvent_t> iterEvents;

    hipEvent_t evAsStart = nullptr, evAsEnd = nullptr, evRtStart = nullptr, evRtOnlyEnd = nullptr, evRoughEnd = nullptr,
               evPostEnd = nullptr;
    std::vector<hipEvent_t> traceEvents; // pairs per trace launch (timing mode)
    std::vector<hipEvent_t> shadeEvents;
    uint32_t lastTraceLaunches = 0;
    uint32_t lastWaves = 0;
    bool timedAs = false, timedRt = false, timedPost = false;

    // rgrt_frame in graph form: the executable graph, updated every frame
    hipGraphExec_t frameExec = nullptr;

    uint8_t* dRgba8 = nullptr; // display-format readback
    uint64_t rgba8Cap = 0;
    hipEvent_t evFrameStart = nullptr, evFrameEnd = nullptr;
    bool timedFrame = false;

    TraceScene scene() const
    {
        TraceScene sc;
        sc.tlasNodes = tlasWideq;
        sc.instances = dInst;
        sc.blas = sd->dBlasTable;
        sc.numInstances = haveTlas ? numInstances : 0;
        sc.tlasNodeCap = std::max<uint32_t>(sc.numInstances, 2u) - 1u;
        sc.numBlas = (uint32_t)sd->blas.size();
        sc.errors = error_word();
        return sc;
    }
    // Where the traversal kernels flag bad indices.
    uint32_t* error_word() const { return st.counters ? st.counters + kTraversalErrorWord : rayFetch + 1; }
};

namespace {

rgrt_status fail(rgrt_ctx* c, rgrt_status code, const std::string& msg)
{
    if(c) c->err = msg;
    return code;
}

// Before the scene data changes: the work queued on every context that
// shares it (frames in flight included) has finished.
void scene_quiesce(rgrt_ctx* c)
{
    std::lock_guard<std::mutex> g(c->sd->m);
    for(rgrt_ctx* u: c->sd->users) check(hipStreamSynchronize(u->stream));
}

// In-place writes of the scene (vertex updates, BLAS rebuilds) are ordered
// on the GPU rather than on the host: they start after the work already
// queued on every sharing context, and work queued later on those contexts
// starts after them. No allocation changes, so nothing waits on the host.
void scene_write_begin(rgrt_ctx* c)
{
    std::lock_guard<std::mutex> g(c->sd->m);
    for(rgrt_ctx* u: c->sd->users)
        if(u != c) {
            check(hipEventRecord(u->sceneEv, u->stream));
            check(hipStreamWaitEvent(c->stream, u->sceneEv, 0));
        }
}

void scene_write_end(rgrt_ctx* c)
{
    std::lock_guard<std::mutex> g(c->sd->m);
    if(c->sd->users.size() < 2) return;
    check(hipEventRecord(c->sceneEv, c->stream));
    for(rgrt_ctx* u: c->sd->users)
        if(u != c) check(hipStreamWaitEvent(u->stream, c->sceneEv, 0));
}

// Scratch of rgrt_rebuild_blas_noalloc: the LBVH builder's working arrays for
// up to kNoAllocMaxFaces triangles in a file-scope device array (48 MiB),
// one copy per GPU, held until the process ends. Host code never passes the
// array's name to a kernel or a copy: it uses the device address that
// hipGetSymbolAddress returns for the current device (noAllocScratch).
constexpr uint32_t kNoAllocMaxFaces = 1u << 18;
constexpr size_t kNoAllocScratchBytes = lbvh_scratch_bytes(kNoAllocMaxFaces);
static __device__ __align__(256) unsigned char scratch[kNoAllocScratchBytes];

std::mutex noAllocMutex;
std::vector<void*> noAllocScratch; // per device: the address of `scratch` there

// Looks the array's address up once per device, with that device current
// (rgrt_create sets it before calling this).
void noalloc_scratch_setup(int device)
{
    std::lock_guard<std::mutex> g(noAllocMutex);
    if((int)noAllocScratch.size() <= device) noAllocScratch.resize(device + 1, nullptr);
    if(noAllocScratch[device]) return;
    void* p = nullptr;
    check(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)));
    if(!p || (reinterpret_cast<uintptr_t>(p) & 255u)) throw std::runtime_error("no-alloc scratch: bad symbol address");
    noAllocScratch[device] = p;
}

void* noalloc_scratch(int device)
{
    std::lock_guard<std::mutex> g(noAllocMutex);
    return device < (int)noAllocScratch.size() ? noAllocScratch[device] : nullptr;
}

// Grows the LBVH builder's scratch for n primitives; earlier work queued on
// the context may still use the old scratch, so it finishes first.
void reserve_builder(rgrt_ctx* c, uint32_t n)
{
    if(n <= c->builder.capacity) return;
    check(hipStreamSynchronize(c->stream));
    c->builder.reserve(n);
}

// New geometry invalidates every BLAS, so every sharing context's TLAS.
// Shading records of the triangles of BLAS description d (launched on s).
void shade_records_of(rgrt_ctx* c, hipStream_t s, const rgrt_blas_desc& d)
{
    launch_shade_records(s, c->sd->vb, c->sd->ib, c->sd->nv, c->sd->ni, d.firstVertex, d.indexOffsetBytes / 4, d.numFaces,
                         c->sd->srec);
}

// After vertices [first, first + count) changed: the records of every BLAS
// whose vertex range overlaps them are gathered again (on the context's
// stream, after the vertex copy), so a record never holds an old normal or
// material index.
void refresh_shade_records(rgrt_ctx* c, uint64_t first, uint64_t count)
{
    for(const BlasRec& b: c->sd->blas) {
        if(!b.valid) continue;
        const uint64_t lo = b.desc.firstVertex, hi = lo + b.desc.maxVertex;
        if(first < hi && lo < first + count) shade_records_of(c, c->stream, b.desc);
    }
}

void scene_drop_tlases(rgrt_ctx* c)
{
    std::lock_guard<std::mutex> g(c->sd->m);
    for(rgrt_ctx* u: c->sd->users) u->haveTlas = false;
}

// The traversal kernels flag tree or table indices out of range (a corrupt
// structure) instead of reading past an allocation; report it once the
// stream is idle. The flag stays set: results after it are not trusted.
rgrt_status traversal_status(rgrt_ctx* c, uint32_t flags)
{
    if(!flags) return RGRT_OK;
    char buf[160];
    std::snprintf(buf, sizeof(buf), "traversal found indices out of range (flags 0x%x: 1 node, 2 instance, 4 BLAS, 8 triangle)",
                  flags);
    return fail(c, RGRT_ERR_HIP, buf);
}

rgrt_status traversal_errors(rgrt_ctx* c)
{
    uint32_t flags = 0;
    check(hipMemcpy(&flags, c->error_word(), 4, hipMemcpyDeviceToHost));
    return traversal_status(c, flags);
}

// Host queries of up to kPinnedRays rays: copies between pageable and device
// memory and the read of the error word cost each some 10 us, more than the
// bytes. The rays are read from, and hits and error word written to, pinned
// memory of the context instead, with one wait: one ray 57 -> 35 us, 1,024
// 97 -> 71, 4,096 123 -> 95 (hits through a device buffer and one more copy: 86
// and 115). It would go on: 16,384 rays 158 -> 124 us, 65,536 284 -> 246. The
// limit is there for the memory, 208 KB of pinned memory in every context.
constexpr uint32_t kPinnedRays = 4096;
constexpr size_t kRayIoHits = kPinnedRays * sizeof(rgrt_ray), kRayIoError = kRayIoHits + kPinnedRays * sizeof(rgrt_hit);

// With the context, so that there is none without it and a first query costs
// what later ones do.
void alloc_ray_io(rgrt_ctx* c)
{
    check(hipHostMalloc((void**)&c->hRayIo, kRayIoError + 64, hipHostMallocMapped));
    check(hipHostGetDevicePointer((void**)&c->hRayIoDev, c->hRayIo, 0));
}

template<typename F>
rgrt_status guarded(rgrt_ctx* c, F f)
{
    if(!c) return RGRT_ERR_INVALID_ARG;
    try {
        return f();
    }
    catch(const HipError& e) {
        return fail(c, e.code == hipErrorOutOfMemory ? RGRT_ERR_OUT_OF_MEMORY : RGRT_ERR_HIP, std::string("HIP: ") + e.what());
    }
    catch(const std::exception& e) {
        return fail(c, RGRT_ERR_HIP, e.what());
    }
}

void free_images(rgrt_ctx* c)
{
    Images& m = c->img;
    dev_free(m.base);
    dev_free(m.normal);
    dev_free(m.rough);
    dev_free(m.final_);
    dev_free(m.transitions);
    dev_free(m.colorsA);
    dev_free(m.colorsB);
    dev_free(m.base32);
    dev_free(m.normal32);
    dev_free(m.rough32);
    dev_free(m.primary);
    dev_free(m.features);
    WavefrontState& s = c->st;
    dev_free(s.lum2);
    dev_free(s.payload);
    dev_free(s.accum);
    dev_free(s.frames);
    dev_free(s.rays[0]);
    dev_free(s.rays[1]);
    dev_free(s.hits);
    dev_free(s.ahead);
    dev_free(s.segs);
    dev_free(s.sampleAcc);
    dev_free(s.sampleLum2);
    c->slotCap = 0;
    c->sampleCap = 0;
    dev_free(s.counters);
    s.npix = 0;
    c->w = 0;
    c->h = 0;
}

// Whether a frame's shading passes queue reflection and refraction rays ahead
// (wavefront.hip): it makes the chain of passes a third shorter, but the
// shading kernel that takes such hits needs 160 VGPRs instead of 128. Small
// frames wait on the chain; large ones, and several frames in flight, on the
// work. The line lies where frames in flight stop gaining. Without and with
// rays ahead, us per frame, one sphere (depth 1) | 32 instances (depth 4):
//   slots    one at a time           2 in flight
//    57,600   449, 357 | 1916, 1619   272, 232 |  965, 825
//   230,400   518, 434 | 2055, 1988   306, 276 | 1073, 1029
//   291,600   554, 500 | 2174, 2088   327, 333 | 1123, 1076
//   518,400   654, 643 | 2232, 2196   432, 485 | 1200, 1161
// 960x540 (518,400) over 3,000 instances takes 3.66 and 3.89 ms, 1080p over 2M
// triangles 8.75 and 9.8. The number in flight is not known to a context, so
// the rule is the slot count. Slots that run several samples one after another
// keep the plain kernels.
constexpr uint32_t kAheadSlots = 300000;
static_assert(kAheadSlots <= kAheadMaxSlots, "a queue entry names its slot");

// Words of the suspended frames and of the queue of rays ahead for up to n
// slots: a frame with fewer slots may be one with rays ahead.
size_t frame_words(size_t n)
{
    return std::max(n * kFrameStride, std::min<size_t>(n, kAheadSlots) * kFrameStrideAhead) * kMaxFrames;
}
size_t ahead_words(size_t n) { return std::min<size_t>(n, kAheadSlots) * kAheadPerSlot * kAheadWords; }

void alloc_images(rgrt_ctx* c, uint32_t w, uint32_t h)
{
    free_images(c);
    const size_t npix = (size_t)w * h;
    Images& m = c->img;
    m.w = w;
    m.h = h;
    dev_alloc(m.base, npix * 4);
    dev_alloc(m.normal, npix * 4);
    dev_alloc(m.rough, npix * 4);
    dev_alloc(m.final_, npix * 4);
    dev_alloc(m.transitions, npix);
    dev_alloc(m.colorsA, npix * 4);
    dev_alloc(m.colorsB, npix * 4);
    if(c->flags & RGRT_CFG_FP32_RADIANCE) {
        dev_alloc(m.base32, npix * 4);
        dev_alloc(m.normal32, npix * 4);
        dev_alloc(m.rough32, npix * 4);
    }
    if(c->flags & RGRT_CFG_PRIMARY_AOV) dev_alloc(m.primary, npix);
    dev_alloc(m.features, npix * 8);
    check(hipMemsetAsync(m.features, 0, npix * 16, c->stream));
    check(hipMemsetAsync(m.base, 0, npix * 8, c->stream));
    check(hipMemsetAsync(m.normal, 0, npix * 8, c->stream));
    check(hipMemsetAsync(m.rough, 0, npix * 8, c->stream));
    check(hipMemsetAsync(m.final_, 0, npix * 8, c->stream));
    WavefrontState& s = c->st;
    s.npix = (uint32_t)npix;
    s.nimg = (uint32_t)npix;
    s.groups = 1;
    s.numSamples = 1;
    dev_alloc(s.payload, npix * kPayloadWords);
    dev_alloc(s.accum, npix * kAccumWords);
    dev_alloc(s.lum2, npix);
    dev_alloc(s.frames, frame_words(npix));
    dev_alloc(s.rays[0], npix * kRayWords);
    dev_alloc(s.rays[1], npix * kRayWords);
    dev_alloc(s.hits, npix * kHitWords);
    dev_alloc(s.ahead, ahead_words(npix));
    dev_alloc(s.segs, kMaxBands * kSegmentBlock);
    dev_alloc(s.counters, 64);
    check(hipMemsetAsync(s.counters, 0, 64 * 4, c->stream));
    c->slotCap = npix;
    c->w = w;
    c->h = h;
}

void ensure_blas_cap(rgrt_ctx* c, uint32_t n)
{
    if(n <= c->sd->blasCap) return;
    const uint32_t cap = std::max<uint32_t>(n, std::max<uint32_t>(16, c->sd->blasCap * 2));
    DevBlas* t = nullptr;
    float4* r = nullptr;
    check(hipMalloc((void**)&t, cap * sizeof(DevBlas)));
    check(hipMalloc((void**)&r, cap * 2 * sizeof(float4)));
    if(c->sd->blasCap) {
        check(hipMemcpyAsync(t, c->sd->dBlasTable, c->sd->blasCap * sizeof(DevBlas), hipMemcpyDeviceToDevice, c->stream));
        check(hipMemcpyAsync(r, c->sd->dBlasRoot, c->sd->blasCap * 2 * sizeof(float4), hipMemcpyDeviceToDevice, c->stream));
        check(hipStreamSynchronize(c->stream));
    }
    dev_free(c->sd->dBlasTable);
    dev_free(c->sd->dBlasRoot);
    c->sd->dBlasTable = t;
    c->sd->dBlasRoot = r;
    c->sd->blasCap = cap;
}

void ensure_inst_cap(rgrt_ctx* c, uint32_t n)
{
    if(n <= c->instCap) return;
    check(hipStreamSynchronize(c->stream)); // queued frames still use the old buffers
    const uint32_t cap = std::max<uint32_t>(n, 64);
    c->instCap = 0;
    c->haveTlas = false; // it is freed here
    for(int k = 0; k < 2; ++k) {
        if(c->hInstStage[k]) {
            check(hipEventSynchronize(c->stageDone[k]));
            (void)hipHostFree(c->hInstStage[k]);
            c->hInstStage[k] = nullptr;
        }
        check(hipHostMalloc((void**)&c->hInstStage[k], cap * sizeof(rgrt_instance), hipHostMallocDefault));
    }
    dev_alloc(c->dInstIn, cap);
    dev_alloc(c->tlasNodes, cap);
    dev_alloc(c->tlasWide, cap);
    dev_alloc(c->tlasWideq, cap);
    if(!c->tlasNumWide) dev_alloc(c->tlasNumWide, 1);
    dev_alloc(c->tlasLeaf, cap);
    dev_alloc(c->dInst, cap);
    dev_alloc(c->dShade, cap);
    dev_alloc(c->dW2O, (size_t)cap * 12);
    if(!c->tlasRoot) dev_alloc(c->tlasRoot, 2);
    c->instCap = cap;
}

void ensure_host_counts(rgrt_ctx* c, uint32_t n)
{
    if(n <= c->hostCountsCap) return;
    if(c->hostCounts) {
        check(hipStreamSynchronize(c->stream));
        (void)hipHostFree(c->hostCounts);
        c->hostCounts = nullptr;
        c->hostCountsCap = 0;
    }
    const uint32_t cap = std::max<uint32_t>(n, 1024);
    check(hipHostMalloc((void**)&c->hostCounts, cap * 4, hipHostMallocMapped));
    check(hipHostGetDevicePointer((void**)&c->hostCountsDev, c->hostCounts, 0));
    c->hostCountsCap = cap;
}

float elapsed(hipEvent_t a, hipEvent_t b)
{
    float ms = 0.0f;
    if(hipEventElapsedTime(&ms, a, b) != hipSuccess) return -1.0f;
    return ms;
}

void make_event(hipEvent_t& e)
{
    if(!e) check(hipEventCreate(&e));
}

static_assert(sizeof(rgrt_stats) == 80, "rgrt_stats layout (Python binding: records.STATS_FIELDS)");
static_assert(sizeof(rgrt_tuning) == 24, "rgrt_tuning layout (Python binding: records.TUNING)");

// The frame in c->ubo (sample groups prepared) queues rays ahead.
bool rays_ahead(const rgrt_ctx* c)
{
    return c->st.npix <= kAheadSlots && c->st.groups >= (uint32_t)std::max(1, c->ubo.numSamples);
}

ShadeParams shade_params(const rgrt_ctx* c)
{
    ShadeParams p;
    p.vb = c->sd->vb;
    p.ib = c->sd->ib;
    p.mats = c->sd->mats;
    p.inst = c->dShade;
    p.srec = c->sd->srec;
    p.numInstances = c->numInstances;
    p.numVertices = c->sd->nv;
    p.numIndices = c->sd->ni;
    p.numMaterials = c->sd->nm;
    p.ubo = c->ubo;
    p.width = c->w;
    p.height = c->h;
    p.st = c->st;
    p.img = c->img;
    p.keepF32 = (c->flags & RGRT_CFG_FP32_RADIANCE) ? 1 : 0;
    p.keepAov = (c->flags & RGRT_CFG_PRIMARY_AOV) ? 1 : 0;
    p.sampling = c->sampling.mode;
    p.seed = c->sampling.seed;
    p.aheadOn = rays_ahead(c) ? 1 : 0;
    return p;
}

// Wavefront slots at most (≈ 0.8 KB of state each: payload, frames, queues).
constexpr uint64_t kMaxSlots = 1ull << 25;

// Sample groups for the frame constants in c->ubo: with several samples per
// pixel, up to numSamples of a pixel's samples run in separate slots side by
// side (each has its own payload, so the order within a sample is kept and
// the samples' records are summed in sample order afterwards), as many as
// kMaxSlots and the context's sampleGroups allow. The slot arrays grow here,
// before anything is enqueued or captured.
void prepare_sample_groups(rgrt_ctx* c)
{
    WavefrontState& s = c->st;
    const uint32_t n = (uint32_t)std::max(1, c->ubo.numSamples);
    uint32_t g = 1;
    if(n > 1 && c->sampleGroups != 1 && s.nimg) {
        g = (uint32_t)std::min<uint64_t>(n, std::max<uint64_t>(1, kMaxSlots / s.nimg));
        if(c->sampleGroups > 1) g = std::min(g, c->sampleGroups);
    }
    const size_t slots = (size_t)s.nimg * g;
    if(slots > c->slotCap) {
        check(hipStreamSynchronize(c->stream)); // queued frames still use the old arrays
        const size_t had = c->slotCap;
        c->slotCap = 0;
        dev_alloc(s.payload, slots * kPayloadWords);
        dev_alloc(s.frames, frame_words(slots));
        dev_alloc(s.rays[0], slots * kRayWords);
        dev_alloc(s.rays[1], slots * kRayWords);
        dev_alloc(s.hits, slots * kHitWords);
        if(ahead_words(slots) > ahead_words(had)) dev_alloc(s.ahead, ahead_words(slots));
        c->slotCap = slots;
    }
    if(g > 1 && (size_t)n * s.nimg > c->sampleCap) {
        check(hipStreamSynchronize(c->stream));
        c->sampleCap = 0;
        dev_alloc(s.sampleAcc, (size_t)n * s.nimg * kAccumWords);
        dev_alloc(s.sampleLum2, (size_t)n * s.nimg);
        c->sampleCap = (size_t)n * s.nimg;
    }
    s.npix = (uint32_t)slots;
    s.chunkFirst = 0;
    s.frameSlots = (uint32_t)slots;
    s.segments = segments_for((uint32_t)slots);
    s.groups = g;
    s.numSamples = n;
}

// Bound on the passes until every slot is done: the rays of one slot's
// samples one after another, plus raygen's pass and one to spare.
uint32_t chain_iters(const rgrt_ctx* c)
{
    const uint32_t perSlot = (c->st.numSamples + c->st.groups - 1) / c->st.groups;
    return max_sequential_rays(c->ubo.maxRecursions) * perSlot + 2;
}

void ensure_band_streams(rgrt_ctx* c);
void enqueue_band(rgrt_ctx* c, uint32_t b, uint32_t bands, hipStream_t s);

rgrt_status do_trace(rgrt_ctx* c)
{
    if(!c->haveTlas) return fail(c, RGRT_ERR_NOT_READY, "rgrt_trace: no TLAS built");
    if(!c->haveUbo) return fail(c, RGRT_ERR_NOT_READY, "rgrt_trace: no frame constants (rgrt_set_frame)");
    if(!c->w || !c->h) return fail(c, RGRT_ERR_NOT_READY, "rgrt_trace: zero-sized render target");
    hipStream_t s = c->stream;
    const bool timing = (c->flags & RGRT_CFG_TIMING) != 0;
    prepare_sample_groups(c);
    const ShadeParams p = shade_params(c);

    const uint32_t maxIters = chain_iters(c);
    ensure_host_counts(c, maxIters + 2);
    const uint32_t lag = c->tuning.hostLag;
    const int ring = (int)std::max<uint32_t>(8u, lag + 2u);
    while((int)c->iterEvents.size() < ring) {
        hipEvent_t e;
        check(hipEventCreateWithFlags(&e, hipEventDisableTiming));
        c->iterEvents.push_back(e);
    }
    if(c->bands > 1 && !timing) {
        // in bands (as the graph form): band 0 on the context stream, the
        // others on theirs after its work so far, joined back before the
        // sample records are finalized; no host waits (every pass runs)
        ensure_band_streams(c);
        c->passStride = maxIters + 2;
        ensure_host_counts(c, c->passStride * c->bands);
        check(hipEventRecord(c->bandFork, s));
        for(uint32_t b = 1; b < c->bands; ++b) {
            check(hipStreamWaitEvent(c->bandStream[b], c->bandFork, 0));
            enqueue_band(c, b, c->bands, c->bandStream[b]);
            check(hipEventRecord(c->bandJoin[b], c->bandStream[b]));
        }
        enqueue_band(c, 0, c->bands, s);
        for(uint32_t b = 1; b < c->bands; ++b) check(hipStreamWaitEvent(s, c->bandJoin[b], 0));
        launch_finalize_samples(s, p);
        const uint32_t passes = std::min<uint32_t>(c->tuning.wavefrontPasses, maxIters);
        c->lastTraceLaunches = passes;
        c->lastDrained = true;
        c->lastWaves = passes;
        c->lastBands = c->bands;
        c->timedRt = false;
        return RGRT_OK;
    }
    if(timing) {
        make_event(c->evRtStart);
        make_event(c->evRtOnlyEnd);
        check(hipEventRecord(c->evRtStart, s));
    }

    const TraceScene sc = c->scene();
    launch_raygen(s, p);
    int cur = 0;
    uint32_t it = 0;
    uint32_t traceLaunches = 0;
    bool drained = false;
    for(; it < maxIters; ++it) {
        // The count of iteration it-lag's input queue is known by now (the GPU
        // runs ahead by at most `lag` iterations); zero means every pixel is done.
        if(it >= lag) {
            check(hipEventSynchronize(c->iterEvents[(it - lag) % ring]));
            if(__atomic_load_n(&c->hostCounts[it - lag], __ATOMIC_ACQUIRE) == 0u) break;
        }
        if(it == c->tuning.wavefrontPasses) {
            // the persistent drain finishes every pixel still in flight
            if(timing) {
                make_event(c->evDrainStart);
                make_event(c->evDrainEnd);
                check(hipEventRecord(c->evDrainStart, s));
            }
            launch_drain(s, p, sc, cur, c->drainGrid, c->spill);
            if(timing) check(hipEventRecord(c->evDrainEnd, s));
            drained = true;
            break;
        }
        if(timing) {
            while(c->traceEvents.size() < 2 * (traceLaunches + 1)) {
                hipEvent_t e;
                check(hipEventCreate(&e));
                c->traceEvents.push_back(e);
            }
            while(c->shadeEvents.size() < 2 * (traceLaunches + 1)) {
                hipEvent_t e;
                check(hipEventCreate(&e));
                c->shadeEvents.push_back(e);
            }
            check(hipEventRecord(c->traceEvents[2 * traceLaunches], s));
        }
        launch_trace_queue_impl(s, sc, c->st, cur, c->traceGrid, c->spill, c->hostCountsDev + it, p.aheadOn);
        check(hipEventRecord(c->iterEvents[it % ring], s));
        if(timing) {
            check(hipEventRecord(c->traceEvents[2 * traceLaunches + 1], s));
            check(hipEventRecord(c->shadeEvents[2 * traceLaunches], s));
        }
        launch_shade(s, p, cur, c->shadeGrid, it + 1 != c->tuning.wavefrontPasses);
        if(timing) check(hipEventRecord(c->shadeEvents[2 * traceLaunches + 1], s));
        ++traceLaunches;
        cur ^= 1;
    }
    if(!drained && it == maxIters) {
        // all pixels must be done after the bound; check the last count
        check(hipStreamSynchronize(s));
        std::vector<uint32_t> counts(kSegmentBlock);
        check(hipMemcpy(counts.data(), c->st.segs, kSegmentBlock * 4, hipMemcpyDeviceToHost));
        uint32_t remaining = 0;
        for(uint32_t q = 0; q < kMaxSegments; ++q) {
            const uint32_t* n = &counts[(cur * kMaxSegments + q) * kSegmentWords];
            remaining += n[0] + n[1];
        }
        if(remaining) return fail(c, RGRT_ERR_HIP, "rgrt_trace: ray queue did not drain within the recursion bound");
    }
    launch_finalize_samples(s, p);
    if(timing) check(hipEventRecord(c->evRtOnlyEnd, s));
    c->lastTraceLaunches = traceLaunches;
    c->lastDrained = drained;
    c->lastWaves = it;
    c->lastBands = 1;
    c->timedRt = timing;
    return RGRT_OK;
}

// The trace of one frame as a fixed launch sequence (no host waits or event
// records, so it can be captured into a graph): raygen, min(wavefrontPasses,
// recursion bound) trace + shade passes, then the drain, which finishes every
// pixel still in flight (with an empty queue it returns at once).
void enqueue_trace_fixed(rgrt_ctx* c)
{
    hipStream_t s = c->stream;
    const ShadeParams p = shade_params(c); // sample groups prepared by frame_prepare
    const uint32_t maxIters = chain_iters(c);
    const uint32_t passes = std::min<uint32_t>(c->tuning.wavefrontPasses, maxIters);
    const TraceScene sc = c->scene();
    launch_raygen(s, p);
    int cur = 0;
    for(uint32_t it = 0; it < passes; ++it) {
        launch_trace_queue_impl(s, sc, c->st, cur, c->traceGrid, c->spill, c->hostCountsDev + it, p.aheadOn);
        launch_shade(s, p, cur, c->shadeGrid, it + 1 < passes);
        cur ^= 1;
    }
    launch_drain(s, p, sc, cur, c->drainGrid, c->spill);
    launch_finalize_samples(s, p);
    c->lastTraceLaunches = passes;
    c->lastDrained = true;
    c->lastWaves = passes;
    c->lastBands = 1;
}

// Band b of `bands`: a run of the frame's 64-slot chunks (whole 8x8 tiles
// in tile order, so a strip of the image). Strips rather than tiles dealt
// out in turn: the strips' work differs (sky against geometry), so they
// reach their sparse last passes at different times and overlap them with
// each other's work; dealt-out tiles give every band the same tail at the
// same time (measured: 7.6-7.7 against 8.0 ms per config-2 frame). Equal
// strips: splits weighted towards either end measured 7.8-9.5 ms.
void band_chunks(uint32_t npix, uint32_t b, uint32_t bands, uint32_t& first, uint32_t& slots, uint32_t& queueFirst)
{
    const uint32_t chunks = (npix + 63u) / 64u;
    const uint32_t lo = (uint32_t)((uint64_t)chunks * b / bands), hi = (uint32_t)((uint64_t)chunks * (b + 1) / bands);
    first = lo;
    slots = std::min(npix, hi * 64u) - std::min(npix, lo * 64u);
    queueFirst = std::min(npix, lo * 64u);
}

// Band b of `bands` with queues, hit records and a counter block of its own,
// carved from the whole frame's arrays, so the bands together use what one
// frame does; the per-slot arrays are shared, each slot belonging to one
// band.
WavefrontState band_state(const WavefrontState& st, uint32_t b, uint32_t bands)
{
    uint32_t first = 0, slots = 0, q0 = 0;
    band_chunks(st.npix, b, bands, first, slots, q0);
    WavefrontState w = st;
    w.npix = slots;
    w.chunkFirst = first;
    w.rays[0] = st.rays[0] + (size_t)kRayWords * q0;
    w.rays[1] = st.rays[1] + (size_t)kRayWords * q0;
    w.hits = st.hits + (size_t)kHitWords * q0;
    w.ahead = st.ahead + (size_t)kAheadWords * kAheadPerSlot * q0;
    w.counters = st.counters + (size_t)kCounterBlock * b;
    w.segs = st.segs + (size_t)kSegmentBlock * b;
    w.segments = segments_for(slots);
    return w;
}

// Streams and fork/join events of bands 1.. (created once, default priority).
void ensure_band_streams(rgrt_ctx* c)
{
    if(c->bands < 2) return;
    if(!c->bandFork) check(hipEventCreateWithFlags(&c->bandFork, hipEventDisableTiming));
    for(uint32_t b = 1; b < c->bands; ++b) {
        if(!c->bandStream[b]) check(hipStreamCreateWithFlags(&c->bandStream[b], hipStreamNonBlocking));
        if(!c->bandJoin[b]) check(hipEventCreateWithFlags(&c->bandJoin[b], hipEventDisableTiming));
    }
}

// The trace of band b as a fixed launch sequence on stream s (capturable):
// raygen of the band's slots, the wavefront passes and the drain over its
// own queues, with its own spill region and pass-count slots. An empty band
// (a frame of fewer than bands x 64 slots) launches empty passes.
void enqueue_band(rgrt_ctx* c, uint32_t b, uint32_t bands, hipStream_t s)
{
    ShadeParams p = shade_params(c);
    p.st = band_state(c->st, b, bands);
    const uint32_t maxIters = chain_iters(c);
    const uint32_t passes = std::min<uint32_t>(c->tuning.wavefrontPasses, maxIters);
    const TraceScene sc = c->scene();
    int32_t* spill = c->spill + c->spillWords * b;
    uint32_t* counts = c->hostCountsDev + (size_t)c->passStride * b;
    launch_raygen(s, p);
    int cur = 0;
    for(uint32_t it = 0; it < passes; ++it) {
        launch_trace_queue_impl(s, sc, p.st, cur, c->traceGrid, spill, counts + it, p.aheadOn);
        launch_shade(s, p, cur, c->shadeGrid, it + 1 < passes);
        cur ^= 1;
    }
    launch_drain(s, p, sc, cur, c->drainGrid, spill);
}

rgrt_status do_post(rgrt_ctx* c, int32_t useFxaa)
{
    if(!c->haveUbo) return fail(c, RGRT_ERR_NOT_READY, "rgrt_postprocess: no frame constants");
    if(!c->w || !c->h) return fail(c, RGRT_ERR_NOT_READY, "rgrt_postprocess: zero-sized render target");
    const bool timing = (c->flags & RGRT_CFG_TIMING) != 0;
    if(timing) {
        make_event(c->evRoughEnd);
        make_event(c->evPostEnd);
        make_event(c->evRtOnlyEnd);
        make_event(c->evRtStart);
        if(!c->timedRt) {
            check(hipEventRecord(c->evRtStart, c->stream));
            check(hipEventRecord(c->evRtOnlyEnd, c->stream));
        }
    }
    launch_post(c->stream, c->img, c->ubo, useFxaa, timing ? c->evRoughEnd : nullptr);
    if(timing) check(hipEventRecord(c->evPostEnd, c->stream));
    if(useFxaa) std::swap(c->img.base, c->img.final_); // raygun/render/raytracer.cpp:139
    c->timedPost = timing;
    return RGRT_OK;
}

// Validates the instances, starts the timing event and copies them to the
// device through the pinned staging buffer.
rgrt_status validate_instances(rgrt_ctx* c, const rgrt_instance* in, uint32_t n, bool refit, const char* who)
{
    if(n && !in) return fail(c, RGRT_ERR_INVALID_ARG, std::string(who) + ": null instances");
    for(uint32_t i = 0; i < n; ++i) {
        if(in[i].blas >= c->sd->blas.size() || !c->sd->blas[in[i].blas].valid)
            return fail(c, RGRT_ERR_INVALID_ARG, std::string(who) + ": instance references an invalid BLAS");
        if(in[i].customIndex >= n)
            return fail(c, RGRT_ERR_INVALID_ARG, std::string(who) + ": customIndex must index the offset table");
    }
    if(refit) {
        if(!c->haveTlas) return fail(c, RGRT_ERR_NOT_READY, std::string(who) + ": refit without a TLAS built");
        if(n != c->numInstances)
            return fail(c, RGRT_ERR_INVALID_ARG, std::string(who) + ": refit: instance count differs from the build");
        for(uint32_t i = 0; i < n; ++i)
            if(in[i].blas != c->tlasBlas[i])
                return fail(c, RGRT_ERR_INVALID_ARG, std::string(who) + ": refit: an instance's BLAS differs from the build");
    }
    return RGRT_OK;
}

// Copies the instances into the pinned staging buffer once the previous
// upload from it has completed.
void stage_to_host(rgrt_ctx* c, const rgrt_instance* in, uint32_t n)
{
    ensure_inst_cap(c, std::max<uint32_t>(n, 1));
    c->stageIdx ^= 1;
    check(hipEventSynchronize(c->stageDone[c->stageIdx])); // the upload two frames back has left this buffer
    if(n) std::memcpy(c->hInstStage[c->stageIdx], in, n * sizeof(rgrt_instance));
}

rgrt_status stage_instances(rgrt_ctx* c, const rgrt_instance* in, uint32_t n, bool refit, const char* who)
{
    const rgrt_status st = validate_instances(c, in, n, refit, who);
    if(st != RGRT_OK) return st;
    hipStream_t s = c->stream;
    if(c->flags & RGRT_CFG_TIMING) {
        make_event(c->evAsStart);
        make_event(c->evAsEnd);
        check(hipEventRecord(c->evAsStart, s));
    }
    stage_to_host(c, in, n);
    if(n)
        check(hipMemcpyAsync(c->dInstIn, c->hInstStage[c->stageIdx], n * sizeof(rgrt_instance), hipMemcpyHostToDevice, s));
    check(hipEventRecord(c->stageDone[c->stageIdx], s));
    return RGRT_OK;
}

// The device work of a TLAS build or refit over the instances already in
// dInstIn (one workgroup up to 1024 instances, the multi-kernel LBVH above);
// the builder's scratch must be reserved for n beforehand.
void enqueue_tlas(rgrt_ctx* c, uint32_t n, bool refit)
{
    hipStream_t s = c->stream;
    if(launch_tlas_fused(s, c->dInstIn, n, c->sd->dBlasRoot, c->dW2O, c->dShade, c->tlasNodes, c->tlasLeaf, c->tlasRoot,
                         c->tlasWide, c->tlasWideq, c->tlasNumWide, c->dInst, refit))
        return;
    launch_inst_prep(s, c->dInstIn, n, c->sd->dBlasRoot, c->builder.boxLo, c->builder.boxHi, c->dW2O, c->dShade);
    if(refit) c->builder.refit(s, n, c->tlasNodes, c->tlasLeaf, c->tlasRoot);
    else c->builder.build(s, n, c->tlasNodes, c->tlasLeaf, c->tlasRoot);
    c->builder.collapse(s, n, c->tlasNodes, c->tlasWide, c->tlasNumWide);
    c->builder.quantize(s, std::max<uint32_t>(n, 2) - 1, c->tlasWide, c->tlasNumWide, c->tlasWideq);
    launch_inst_gather(s, c->dW2O, c->dInstIn, c->tlasLeaf, n, c->dInst);
}

void finish_tlas(rgrt_ctx* c, const rgrt_instance* in, uint32_t n)
{
    const bool timing = (c->flags & RGRT_CFG_TIMING) != 0;
    if(timing) check(hipEventRecord(c->evAsEnd, c->stream));
    c->timedAs = timing;
    c->numInstances = n;
    c->tlasBlas.resize(n);
    for(uint32_t i = 0; i < n; ++i) c->tlasBlas[i] = in[i].blas;
    c->haveTlas = true;
}
} // namespace

extern "C" {

const char* rgrt_version(void) { return "rgrt 0.1 (gfx950)"; }

rgrt_status rgrt_create(rgrt_ctx** out, const rgrt_config* cfg)
{
    if(!out || !cfg) return RGRT_ERR_INVALID_ARG;
    *out = nullptr;
    int ndev = 0;
    if(hipGetDeviceCount(&ndev) != hipSuccess || ndev == 0) return RGRT_ERR_NO_DEVICE;
    if(cfg->device < 0 || cfg->device >= ndev) return RGRT_ERR_INVALID_ARG;
    auto* c = new rgrt_ctx();
    c->device = cfg->device;
    c->flags = cfg->flags;
    c->sd = std::make_shared<SceneData>();
    c->sd->add_user(c);
    rgrt_status st = guarded(c, [&]() {
        check(hipSetDevice(c->device));
        noalloc_scratch_setup(c->device);
        check(hipStreamCreateWithFlags(&c->stream, hipStreamNonBlocking));
        hipDeviceProp_t prop;
        check(hipGetDeviceProperties(&prop, c->device));
        c->numCUs = (uint32_t)std::max(1, prop.multiProcessorCount);
        c->apply_tuning();
        dev_alloc(c->rayFetch, 2);
        check(hipMemsetAsync(c->rayFetch, 0, 8, c->stream));
        alloc_ray_io(c);
        for(int k = 0; k < 2; ++k) check(hipEventCreateWithFlags(&c->stageDone[k], hipEventDisableTiming));
        check(hipEventCreateWithFlags(&c->sceneEv, hipEventDisableTiming));
        if(cfg->width && cfg->height) alloc_images(c, cfg->width, cfg->height);
        return RGRT_OK;
    });
    if(st != RGRT_OK) {
        rgrt_destroy(c);
        return st;
    }
    *out = c;
    return RGRT_OK;
}

rgrt_status rgrt_create_shared(rgrt_ctx* parent, const rgrt_config* cfg, rgrt_ctx** out)
{
    if(!out) return RGRT_ERR_INVALID_ARG;
    *out = nullptr;
    if(!parent || !cfg) return RGRT_ERR_INVALID_ARG;
    if(cfg->device != parent->device) return fail(parent, RGRT_ERR_INVALID_ARG, "create_shared: other device");
    rgrt_ctx* c = nullptr;
    const rgrt_status st = rgrt_create(&c, cfg);
    if(st != RGRT_OK) return st;
    c->sd->remove_user(c);
    c->sd = parent->sd;
    c->sd->add_user(c);
    *out = c;
    return RGRT_OK;
}

void rgrt_destroy(rgrt_ctx* c)
{
    if(!c) return;
    (void)hipSetDevice(c->device);
    if(c->stream) (void)hipStreamSynchronize(c->stream);
    free_images(c);
    c->sd->remove_user(c);
    c->sd.reset(); // the last context sharing the scene frees it
    dev_free(c->dInstIn);
    dev_free(c->tlasNodes);
    dev_free(c->tlasWide);
    dev_free(c->tlasWideq);
    dev_free(c->tlasNumWide);
    dev_free(c->tlasLeaf);
    dev_free(c->dInst);
    dev_free(c->dShade);
    dev_free(c->dW2O);
    dev_free(c->tlasRoot);
    dev_free(c->spill);
    dev_free(c->dRays);
    dev_free(c->rayFetch);
    if(c->hRayIo) (void)hipHostFree(c->hRayIo);
    dev_free(c->dRgba8);
    dev_free(c->dHits);
    c->builder.release();
    for(int k = 0; k < 2; ++k)
        if(c->hInstStage[k]) (void)hipHostFree(c->hInstStage[k]);
    if(c->hostCounts) (void)hipHostFree(c->hostCounts);
    for(hipEvent_t e: c->iterEvents) (void)hipEventDestroy(e);
    for(hipEvent_t e: c->traceEvents) (void)hipEventDestroy(e);
    for(hipEvent_t e: c->shadeEvents) (void)hipEventDestroy(e);
    if(c->frameExec) (void)hipGraphExecDestroy(c->frameExec);
    for(hipGraphExec_t g: {c->preExec, c->postExec, c->bandExec[0], c->bandExec[1], c->bandExec[2], c->bandExec[3]})
        if(g) (void)hipGraphExecDestroy(g);
    static_assert(kMaxBands == 4, "band graphs destroyed above");
    for(uint32_t b = 1; b < kMaxBands; ++b) {
        if(c->bandStream[b]) {
            (void)hipStreamSynchronize(c->bandStream[b]);
            (void)hipStreamDestroy(c->bandStream[b]);
        }
        if(c->bandJoin[b]) (void)hipEventDestroy(c->bandJoin[b]);
    }
    if(c->bandFork) (void)hipEventDestroy(c->bandFork);
    for(hipEvent_t e: {c->evAsStart, c->evAsEnd, c->evRtStart, c->evRtOnlyEnd, c->evRoughEnd, c->evPostEnd, c->stageDone[0],
                       c->stageDone[1], c->sceneEv,
                       c->evDrainStart, c->evDrainEnd, c->evFrameStart, c->evFrameEnd})
        if(e) (void)hipEventDestroy(e);
    if(c->stream) (void)hipStreamDestroy(c->stream);
    delete c;
}

const char* rgrt_last_error(const rgrt_ctx* c) { return c ? c->err.c_str() : "null context"; }

void* rgrt_stream(rgrt_ctx* c) { return c ? (void*)c->stream : nullptr; }

rgrt_status rgrt_synchronize(rgrt_ctx* c)
{
    return guarded(c, [&]() {
        check(hipStreamSynchronize(c->stream));
        return traversal_errors(c);
    });
}

rgrt_status rgrt_upload_geometry(rgrt_ctx* c, const rgrt_vertex* vertices, uint64_t nv, const uint32_t* indices, uint64_t ni)
{
    return guarded(c, [&]() {
        if((nv && !vertices) || (ni && !indices) || ni % 3) return fail(c, RGRT_ERR_INVALID_ARG, "upload_geometry: bad arrays");
        check(hipSetDevice(c->device));
        scene_quiesce(c);
        dev_alloc(c->sd->vb, nv);
        dev_alloc(c->sd->ib, ni);
        dev_alloc(c->sd->srec, ni / 3);
        if(nv) check(hipMemcpy(c->sd->vb, vertices, nv * sizeof(rgrt_vertex), hipMemcpyHostToDevice));
        if(ni) check(hipMemcpy(c->sd->ib, indices, ni * 4, hipMemcpyHostToDevice));
        // no triangle has a shading record until a BLAS over it is built;
        // complete before returning, so any context's later builds (on
        // their own non-blocking streams) write after it
        check(hipMemsetAsync(c->sd->srec, 0xff, std::max<uint64_t>(ni / 3, 1) * sizeof(ShadeTri), c->stream));
        check(hipStreamSynchronize(c->stream));
        c->sd->nv = nv;
        c->sd->ni = ni;
        for(auto& b: c->sd->blas) b.valid = false; // geometry changed: every BLAS must be rebuilt
        scene_drop_tlases(c);
        return RGRT_OK;
    });
}

rgrt_status rgrt_update_vertices(rgrt_ctx* c, uint64_t first, const rgrt_vertex* vertices, uint64_t count)
{
    return guarded(c, [&]() {
        if(first + count > c->sd->nv || (count && !vertices)) return fail(c, RGRT_ERR_INVALID_ARG, "update_vertices: range");
        scene_quiesce(c);
        if(count)
            check(hipMemcpyAsync(c->sd->vb + first, vertices, count * sizeof(rgrt_vertex), hipMemcpyHostToDevice, c->stream));
        refresh_shade_records(c, first, count);
        check(hipStreamSynchronize(c->stream));
        return RGRT_OK;
    });
}

rgrt_status rgrt_update_vertices_device(rgrt_ctx* c, uint64_t first, const rgrt_vertex* vertices, uint64_t count)
{
    return guarded(c, [&]() {
        if(first + count > c->sd->nv || (count && !vertices))
            return fail(c, RGRT_ERR_INVALID_ARG, "update_vertices_device: range");
        if(!count) return RGRT_OK;
        scene_write_begin(c);
        check(hipMemcpyAsync(c->sd->vb + first, vertices, count * sizeof(rgrt_vertex), hipMemcpyDeviceToDevice, c->stream));
        refresh_shade_records(c, first, count);
        scene_write_end(c);
        return RGRT_OK;
    });
}

rgrt_status rgrt_upload_materials(rgrt_ctx* c, const rgrt_material* materials, uint32_t n)
{
    return guarded(c, [&]() {
        if(n && !materials) return fail(c, RGRT_ERR_INVALID_ARG, "upload_materials: null");
        if(n > kMaxMaterials) return fail(c, RGRT_ERR_INVALID_ARG, "upload_materials: more than 2^28 materials");
        scene_quiesce(c);
        dev_alloc(c->sd->mats, n);
        if(n) check(hipMemcpy(c->sd->mats, materials, n * sizeof(rgrt_material), hipMemcpyHostToDevice));
        c->sd->nm = n;
        return RGRT_OK;
    });
}

rgrt_status rgrt_build_blas(rgrt_ctx* c, const rgrt_blas_desc* d, rgrt_blas* out)
{
    return guarded(c, [&]() {
        if(!d || !out) return fail(c, RGRT_ERR_INVALID_ARG, "build_blas: null");
        if(d->indexOffsetBytes % 4) return fail(c, RGRT_ERR_INVALID_ARG, "build_blas: index offset not 4-aligned");
        const uint64_t io = d->indexOffsetBytes / 4;
        if(io + 3ull * d->numFaces > c->sd->ni) return fail(c, RGRT_ERR_INVALID_ARG, "build_blas: index range outside the buffer");
        if((uint64_t)d->firstVertex + d->maxVertex > c->sd->nv)
            return fail(c, RGRT_ERR_INVALID_ARG, "build_blas: vertex range outside the buffer");
        if(d->numFaces && d->maxVertex == 0) return fail(c, RGRT_ERR_INVALID_ARG, "build_blas: maxVertex is 0");
        // every index must address a vertex of the range
        std::vector<uint32_t> idx(3ull * d->numFaces);
        if(!idx.empty()) check(hipMemcpy(idx.data(), c->sd->ib + io, idx.size() * 4, hipMemcpyDeviceToHost));
        for(uint32_t v: idx)
            if(v >= d->maxVertex) return fail(c, RGRT_ERR_INVALID_ARG, "build_blas: index >= maxVertex");

        scene_quiesce(c);
        hipStream_t s = c->stream;
        const uint32_t id = (uint32_t)c->sd->blas.size();
        ensure_blas_cap(c, id + 1);
        BlasRec b;
        b.desc = *d;
        const uint32_t n = d->numFaces;
        dev_alloc(b.nodes, std::max<uint32_t>(n, 2) - 1);
        dev_alloc(b.wide, std::max<uint32_t>(n, 2) - 1);
        dev_alloc(b.wideq, std::max<uint32_t>(n, 2) - 1);
        dev_alloc(b.numWide, 1);
        dev_alloc(b.tris, 3ull * n + 1); // three axis orders, see Tri; one more: the traversal fetches 64 bytes of a leaf
        dev_alloc(b.leafPrim, n);
        reserve_builder(c, std::max<uint32_t>(n, 1));
        launch_tri_boxes(s, c->sd->vb, c->sd->ib, d->firstVertex, (uint32_t)io, n, c->builder.boxLo, c->builder.boxHi);
        c->builder.build(s, n, b.nodes, b.leafPrim, c->sd->dBlasRoot + 2 * id);
        c->builder.collapse(s, n, b.nodes, b.wide, b.numWide);
        c->builder.quantize(s, std::max<uint32_t>(n, 2) - 1, b.wide, b.numWide, b.wideq);
        launch_tri_gather(s, c->sd->vb, c->sd->ib, d->firstVertex, (uint32_t)io, b.leafPrim, n, b.tris);
        shade_records_of(c, s, *d);
        DevBlas db{b.wideq, b.tris, n, 0};
        check(hipMemcpyAsync(c->sd->dBlasTable + id, &db, sizeof(DevBlas), hipMemcpyHostToDevice, s));
        check(hipStreamSynchronize(s)); // the reference blocks on a fence (raytracer.cpp:71-73)
        b.valid = true;
        c->sd->blas.push_back(b);
        *out = id;
        return RGRT_OK;
    });
}

rgrt_status rgrt_refit_blas(rgrt_ctx* c, rgrt_blas id)
{
    return guarded(c, [&]() {
        if(id >= c->sd->blas.size() || !c->sd->blas[id].valid) return fail(c, RGRT_ERR_INVALID_ARG, "refit_blas: bad handle");
        scene_quiesce(c);
        BlasRec& b = c->sd->blas[id];
        hipStream_t s = c->stream;
        const uint32_t n = b.desc.numFaces;
        const uint32_t io = b.desc.indexOffsetBytes / 4;
        reserve_builder(c, std::max<uint32_t>(n, 1));
        launch_tri_boxes(s, c->sd->vb, c->sd->ib, b.desc.firstVertex, io, n, c->builder.boxLo, c->builder.boxHi);
        c->builder.refit(s, n, b.nodes, b.leafPrim, c->sd->dBlasRoot + 2 * id);
        c->builder.collapse(s, n, b.nodes, b.wide, b.numWide); // wide topology follows the new areas
        c->builder.quantize(s, std::max<uint32_t>(n, 2) - 1, b.wide, b.numWide, b.wideq);
        launch_tri_gather(s, c->sd->vb, c->sd->ib, b.desc.firstVertex, io, b.leafPrim, n, b.tris);
        shade_records_of(c, s, b.desc);
        check(hipStreamSynchronize(s));
        return RGRT_OK;
    });
}

rgrt_status rgrt_rebuild_blas(rgrt_ctx* c, rgrt_blas id)
{
    return guarded(c, [&]() {
        if(id >= c->sd->blas.size() || !c->sd->blas[id].valid) return fail(c, RGRT_ERR_INVALID_ARG, "rebuild_blas: bad handle");
        BlasRec& b = c->sd->blas[id];
        hipStream_t s = c->stream;
        const uint32_t n = b.desc.numFaces;
        const uint32_t io = b.desc.indexOffsetBytes / 4;
        reserve_builder(c, std::max<uint32_t>(n, 1));
        scene_write_begin(c);
        // the same kernels as rgrt_build_blas, into the BLAS's own buffers
        launch_tri_boxes(s, c->sd->vb, c->sd->ib, b.desc.firstVertex, io, n, c->builder.boxLo, c->builder.boxHi);
        c->builder.build(s, n, b.nodes, b.leafPrim, c->sd->dBlasRoot + 2 * id);
        c->builder.collapse(s, n, b.nodes, b.wide, b.numWide);
        c->builder.quantize(s, std::max<uint32_t>(n, 2) - 1, b.wide, b.numWide, b.wideq);
        launch_tri_gather(s, c->sd->vb, c->sd->ib, b.desc.firstVertex, io, b.leafPrim, n, b.tris);
        shade_records_of(c, s, b.desc);
        scene_write_end(c);
        return RGRT_OK;
    });
}

rgrt_status rgrt_rebuild_blas_noalloc(rgrt_ctx* c, rgrt_blas id)
{
    return guarded(c, [&]() {
        if(id >= c->sd->blas.size() || !c->sd->blas[id].valid)
            return fail(c, RGRT_ERR_INVALID_ARG, "rebuild_blas_noalloc: bad handle");
        BlasRec& b = c->sd->blas[id];
        const uint32_t n = b.desc.numFaces;
        if(n > kNoAllocMaxFaces)
            return fail(c, RGRT_ERR_INVALID_ARG,
                        "rebuild_blas_noalloc: " + std::to_string(n) + " triangles; its scratch holds at most " +
                            std::to_string(kNoAllocMaxFaces) + " (use rgrt_rebuild_blas)");
        void* base = noalloc_scratch(c->device);
        if(!base) return fail(c, RGRT_ERR_NOT_READY, "rebuild_blas_noalloc: no scratch on this device");
        LbvhBuilder bld; // views into the device's scratch array; owns nothing
        bld.bind(base, kNoAllocMaxFaces);
        hipStream_t s = c->stream;
        const uint32_t io = b.desc.indexOffsetBytes / 4;
        scene_write_begin(c);
        launch_tri_boxes(s, c->sd->vb, c->sd->ib, b.desc.firstVertex, io, n, bld.boxLo, bld.boxHi);
        bld.build(s, n, b.nodes, b.leafPrim, c->sd->dBlasRoot + 2 * id);
        bld.collapse(s, n, b.nodes, b.wide, b.numWide);
        bld.quantize(s, std::max<uint32_t>(n, 2) - 1, b.wide, b.numWide, b.wideq);
        launch_tri_gather(s, c->sd->vb, c->sd->ib, b.desc.firstVertex, io, b.leafPrim, n, b.tris);
        shade_records_of(c, s, b.desc);
        scene_write_end(c);
        return RGRT_OK;
    });
}

rgrt_status rgrt_blas_info(rgrt_ctx* c, rgrt_blas id, uint32_t* numNodes, uint32_t* numLeaves, float rootLo[3], float rootHi[3])
{
    return guarded(c, [&]() {
        if(id >= c->sd->blas.size() || !c->sd->blas[id].valid) return fail(c, RGRT_ERR_INVALID_ARG, "blas_info: bad handle");
        check(hipStreamSynchronize(c->stream)); // a rebuild may still be queued
        const uint32_t n = c->sd->blas[id].desc.numFaces;
        if(numNodes) *numNodes = std::max<uint32_t>(n, 2) - 1;
        if(numLeaves) *numLeaves = n;
        float4 r[2];
        check(hipStreamSynchronize(c->stream));
        check(hipMemcpy(r, c->sd->dBlasRoot + 2 * id, sizeof(r), hipMemcpyDeviceToHost));
        if(rootLo) {
            rootLo[0] = r[0].x;
            rootLo[1] = r[0].y;
            rootLo[2] = r[0].z;
        }
        if(rootHi) {
            rootHi[0] = r[1].x;
            rootHi[1] = r[1].y;
            rootHi[2] = r[1].z;
        }
        return RGRT_OK;
    });
}

rgrt_status rgrt_export_blas(rgrt_ctx* c, rgrt_blas id, rgrt_bvh_node* nodes, uint32_t nodeCap, uint32_t* leafPrim, uint32_t leafCap)
{
    return guarded(c, [&]() {
        if(id >= c->sd->blas.size() || !c->sd->blas[id].valid) return fail(c, RGRT_ERR_INVALID_ARG, "export_blas: bad handle");
        check(hipStreamSynchronize(c->stream)); // a rebuild may still be queued
        const BlasRec& b = c->sd->blas[id];
        const uint32_t nn = std::max<uint32_t>(b.desc.numFaces, 2) - 1;
        if((nodes && nodeCap < nn) || (leafPrim && leafCap < b.desc.numFaces))
            return fail(c, RGRT_ERR_INVALID_ARG, "export_blas: capacity");
        check(hipStreamSynchronize(c->stream));
        if(nodes) check(hipMemcpy(nodes, b.nodes, nn * sizeof(Node), hipMemcpyDeviceToHost));
        if(leafPrim && b.desc.numFaces) check(hipMemcpy(leafPrim, b.leafPrim, b.desc.numFaces * 4ull, hipMemcpyDeviceToHost));
        return RGRT_OK;
    });
}

rgrt_status rgrt_export_blas_wide(rgrt_ctx* c, rgrt_blas id, int32_t compressed, void* nodes, uint32_t capacity,
                                  uint32_t* numNodes)
{
    return guarded(c, [&]() {
        if(id >= c->sd->blas.size() || !c->sd->blas[id].valid) return fail(c, RGRT_ERR_INVALID_ARG, "export_blas_wide: bad handle");
        check(hipStreamSynchronize(c->stream)); // a rebuild may still be queued
        check(hipStreamSynchronize(c->stream));
        uint32_t nw = 0;
        check(hipMemcpy(&nw, c->sd->blas[id].numWide, 4, hipMemcpyDeviceToHost));
        if(numNodes) *numNodes = nw;
        if(nodes) {
            if(capacity < nw) return fail(c, RGRT_ERR_INVALID_ARG, "export_blas_wide: capacity");
            if(compressed) check(hipMemcpy(nodes, c->sd->blas[id].wideq, nw * sizeof(Node4q), hipMemcpyDeviceToHost));
            else check(hipMemcpy(nodes, c->sd->blas[id].wide, nw * sizeof(Node4), hipMemcpyDeviceToHost));
        }
        return RGRT_OK;
    });
}

rgrt_status rgrt_export_tlas_wide(rgrt_ctx* c, int32_t compressed, void* nodes, uint32_t capacity, uint32_t* numNodes)
{
    return guarded(c, [&]() {
        if(!c->haveTlas) return fail(c, RGRT_ERR_NOT_READY, "export_tlas_wide: no TLAS");
        check(hipStreamSynchronize(c->stream));
        uint32_t nw = 0;
        check(hipMemcpy(&nw, c->tlasNumWide, 4, hipMemcpyDeviceToHost));
        if(numNodes) *numNodes = nw;
        if(nodes) {
            if(capacity < nw) return fail(c, RGRT_ERR_INVALID_ARG, "export_tlas_wide: capacity");
            if(compressed) check(hipMemcpy(nodes, c->tlasWideq, nw * sizeof(Node4q), hipMemcpyDeviceToHost));
            else check(hipMemcpy(nodes, c->tlasWide, nw * sizeof(Node4), hipMemcpyDeviceToHost));
        }
        return RGRT_OK;
    });
}

rgrt_status rgrt_build_tlas(rgrt_ctx* c, const rgrt_instance* in, uint32_t n)
{
    return guarded(c, [&]() {
        const rgrt_status st = stage_instances(c, in, n, false, "build_tlas");
        if(st != RGRT_OK) return st;
        reserve_builder(c, std::max<uint32_t>(n, 1));
        enqueue_tlas(c, n, false);
        finish_tlas(c, in, n);
        return RGRT_OK;
    });
}

rgrt_status rgrt_refit_tlas(rgrt_ctx* c, const rgrt_instance* in, uint32_t n)
{
    return guarded(c, [&]() {
        const rgrt_status st = stage_instances(c, in, n, true, "refit_tlas");
        if(st != RGRT_OK) return st;
        reserve_builder(c, std::max<uint32_t>(n, 1));
        enqueue_tlas(c, n, true);
        finish_tlas(c, in, n);
        return RGRT_OK;
    });
}

rgrt_status rgrt_export_tlas(rgrt_ctx* c, rgrt_bvh_node* nodes, uint32_t nodeCap, uint32_t* leafInstance, uint32_t leafCap,
                             uint32_t* numNodes)
{
    return guarded(c, [&]() {
        if(!c->haveTlas) return fail(c, RGRT_ERR_NOT_READY, "export_tlas: no TLAS");
        const uint32_t n = c->numInstances;
        const uint32_t nn = std::max<uint32_t>(n, 2) - 1;
        if(numNodes) *numNodes = nn;
        if((nodes && nodeCap < nn) || (leafInstance && leafCap < n)) return fail(c, RGRT_ERR_INVALID_ARG, "export_tlas: capacity");
        check(hipStreamSynchronize(c->stream));
        if(nodes) check(hipMemcpy(nodes, c->tlasNodes, nn * sizeof(Node), hipMemcpyDeviceToHost));
        if(leafInstance && n) check(hipMemcpy(leafInstance, c->tlasLeaf, n * 4ull, hipMemcpyDeviceToHost));
        return RGRT_OK;
    });
}

rgrt_status rgrt_set_frame(rgrt_ctx* c, const rgrt_ubo* ubo)
{
    return guarded(c, [&]() {
        if(!ubo) return fail(c, RGRT_ERR_INVALID_ARG, "set_frame: null");
        if(ubo->numSamples < 1 || ubo->numSamples > 32) return fail(c, RGRT_ERR_INVALID_ARG, "set_frame: numSamples outside 1..32");
        if(ubo->maxRecursions < 0 || ubo->maxRecursions > 7)
            return fail(c, RGRT_ERR_INVALID_ARG, "set_frame: maxRecursions outside 0..7 (pipeline maximum 7)");
        c->ubo = *ubo;
        c->haveUbo = true;
        return RGRT_OK;
    });
}

rgrt_status rgrt_set_sampling(rgrt_ctx* c, const rgrt_sampling* smp)
{
    return guarded(c, [&]() {
        if(!smp || smp->mode > RGRT_SAMPLING_STOCHASTIC) return fail(c, RGRT_ERR_INVALID_ARG, "set_sampling: mode");
        c->sampling = *smp;
        return RGRT_OK;
    });
}

rgrt_status rgrt_resize(rgrt_ctx* c, uint32_t w, uint32_t h)
{
    return guarded(c, [&]() {
        if(!w || !h || (uint64_t)w * h > (1ull << 26)) return fail(c, RGRT_ERR_INVALID_ARG, "resize: size");
        if(w == c->w && h == c->h) return RGRT_OK;
        check(hipStreamSynchronize(c->stream));
        alloc_images(c, w, h);
        return RGRT_OK;
    });
}

rgrt_status rgrt_trace_rays_device(rgrt_ctx* c, const rgrt_ray* rays, uint32_t n, uint32_t cullMask, rgrt_hit* hits)
{
    return guarded(c, [&]() {
        if(!c->haveTlas) return fail(c, RGRT_ERR_NOT_READY, "trace_rays: no TLAS");
        if(n && (!rays || !hits)) return fail(c, RGRT_ERR_INVALID_ARG, "trace_rays: null");
        launch_trace_rays_impl(c->stream, c->scene(), rays, n, cullMask, hits, c->dShade, c->spill, c->traceGrid, 4 * c->numCUs, c->rayFetch);
        return RGRT_OK;
    });
}

} // extern "C"

namespace {

rgrt_status trace_few_rays(rgrt_ctx* c, const rgrt_ray* rays, uint32_t n, uint32_t cullMask, rgrt_hit* hits)
{
    std::memcpy(c->hRayIo, rays, n * sizeof(rgrt_ray));
    launch_trace_rays_impl(c->stream, c->scene(), reinterpret_cast<const rgrt_ray*>(c->hRayIoDev), n, cullMask,
                           reinterpret_cast<rgrt_hit*>(c->hRayIoDev + kRayIoHits), c->dShade, c->spill, c->traceGrid, 4 * c->numCUs,
                           c->rayFetch);
    check(hipMemcpyAsync(c->hRayIo + kRayIoError, c->error_word(), 4, hipMemcpyDeviceToHost, c->stream));
    check(hipStreamSynchronize(c->stream));
    std::memcpy(hits, c->hRayIo + kRayIoHits, n * sizeof(rgrt_hit));
    uint32_t flags = 0;
    std::memcpy(&flags, c->hRayIo + kRayIoError, 4);
    return traversal_status(c, flags);
}

} // namespace

extern "C" {

rgrt_status rgrt_trace_rays(rgrt_ctx* c, const rgrt_ray* rays, uint32_t n, uint32_t cullMask, rgrt_hit* hits)
{
    return guarded(c, [&]() {
        if(!c->haveTlas) return fail(c, RGRT_ERR_NOT_READY, "trace_rays: no TLAS");
        if(n && (!rays || !hits)) return fail(c, RGRT_ERR_INVALID_ARG, "trace_rays: null");
        if(n && n <= kPinnedRays) return trace_few_rays(c, rays, n, cullMask, hits);
        if(n > c->rayCap) {
            c->rayCap = 0;
            dev_alloc(c->dRays, n);
            dev_alloc(c->dHits, n);
            c->rayCap = n;
        }
        if(!n) return RGRT_OK;
        check(hipMemcpyAsync(c->dRays, rays, n * sizeof(rgrt_ray), hipMemcpyHostToDevice, c->stream));
        launch_trace_rays_impl(c->stream, c->scene(), c->dRays, n, cullMask, c->dHits, c->dShade, c->spill, c->traceGrid,
                               4 * c->numCUs, c->rayFetch);
        check(hipMemcpyAsync(hits, c->dHits, n * sizeof(rgrt_hit), hipMemcpyDeviceToHost, c->stream));
        check(hipStreamSynchronize(c->stream));
        return traversal_errors(c);
    });
}

rgrt_status rgrt_trace(rgrt_ctx* c)
{
    return guarded(c, [&]() {
        c->timedRt = false;
        c->timedPost = false;
        return do_trace(c);
    });
}

rgrt_status rgrt_postprocess(rgrt_ctx* c, int32_t useFxaa)
{
    return guarded(c, [&]() {
        c->timedRt = false;
        return do_post(c, useFxaa);
    });
}

rgrt_status rgrt_render(rgrt_ctx* c, int32_t useFxaa)
{
    return guarded(c, [&]() {
        c->timedFrame = false;
        c->timedRt = false;
        c->timedPost = false;
        rgrt_status st = do_trace(c);
        if(st != RGRT_OK) return st;
        return do_post(c, useFxaa);
    });
}

} // extern "C"

namespace {

// Graph form of a frame, in three parts: everything that validates,
// allocates or waits (before a capture), the captured work on the context's
// stream, and the bookkeeping after the launch.
rgrt_status frame_prepare(rgrt_ctx* c, const rgrt_ubo* ubo, const rgrt_instance* in, uint32_t n, uint32_t flags)
{
    if(flags & ~(RGRT_FRAME_FXAA | RGRT_FRAME_REFIT_TLAS | RGRT_FRAME_GRAPH))
        return fail(c, RGRT_ERR_INVALID_ARG, "frame: unknown flags");
    rgrt_status st = rgrt_set_frame(c, ubo);
    if(st != RGRT_OK) return st;
    st = validate_instances(c, in, n, (flags & RGRT_FRAME_REFIT_TLAS) != 0, "frame");
    if(st != RGRT_OK) return st;
    if(!c->w || !c->h) return fail(c, RGRT_ERR_NOT_READY, "frame: zero-sized render target");
    stage_to_host(c, in, n);
    reserve_builder(c, std::max<uint32_t>(n, 1));
    prepare_sample_groups(c);
    c->passStride = chain_iters(c) + 2;
    ensure_host_counts(c, c->passStride * c->bands);
    ensure_band_streams(c);
    return RGRT_OK;
}

// Instance upload and TLAS build or refit of a graph frame.
void frame_enqueue_tlas(rgrt_ctx* c, uint32_t n, uint32_t flags)
{
    if(n)
        check(hipMemcpyAsync(c->dInstIn, c->hInstStage[c->stageIdx], n * sizeof(rgrt_instance), hipMemcpyHostToDevice,
                             c->stream));
    enqueue_tlas(c, n, (flags & RGRT_FRAME_REFIT_TLAS) != 0);
}

void frame_enqueue(rgrt_ctx* c, uint32_t n, uint32_t flags)
{
    frame_enqueue_tlas(c, n, flags);
    enqueue_trace_fixed(c);
    launch_post(c->stream, c->img, c->ubo, (flags & RGRT_FRAME_FXAA) ? 1 : 0, nullptr);
}

void frame_finish(rgrt_ctx* c, const rgrt_instance* in, uint32_t n, uint32_t flags)
{
    if(flags & RGRT_FRAME_FXAA) std::swap(c->img.base, c->img.final_); // raygun/render/raytracer.cpp:139
    finish_tlas(c, in, n);
    c->timedAs = c->timedRt = c->timedPost = false;
}

// Instantiates g into *exec, or updates *exec in place when the topology
// allows; destroys g.
void update_exec(hipGraphExec_t* exec, hipGraph_t g)
{
    bool updated = false;
    if(*exec) {
        hipGraphNode_t errNode = nullptr;
        hipGraphExecUpdateResult res = hipGraphExecUpdateError;
        updated = hipGraphExecUpdate(*exec, g, &errNode, &res) == hipSuccess && res == hipGraphExecUpdateSuccess;
        if(!updated) {
            (void)hipGetLastError(); // a refused update leaves nothing pending
            (void)hipGraphExecDestroy(*exec);
            *exec = nullptr;
        }
    }
    if(!updated) {
        const hipError_t e = hipGraphInstantiate(exec, g, nullptr, nullptr, 0);
        (void)hipGraphDestroy(g);
        check(e);
        return;
    }
    (void)hipGraphDestroy(g);
}

// Captures what f enqueues on stream s into *exec (update_exec).
template<typename F>
void capture_into(hipGraphExec_t* exec, hipStream_t s, F f)
{
    hipGraph_t g = nullptr;
    check(hipStreamBeginCapture(s, hipStreamCaptureModeThreadLocal));
    try {
        f();
    }
    catch(...) {
        (void)hipStreamEndCapture(s, &g);
        if(g) (void)hipGraphDestroy(g);
        throw;
    }
    check(hipStreamEndCapture(s, &g));
    update_exec(exec, g);
}

// A prepared frame (frame_prepare) captured on the context's stream and
// launched there as one hipGraph. With frameBands > 1 the frame is four
// kinds of graph instead: instance upload and TLAS on the context's stream,
// then every band's trace on a stream of its own (band 0 on the context's
// stream), then the post passes once every band has joined. The bands'
// passes run side by side, so one band's last, sparse passes overlap
// another's work instead of leaving the GPU idle; the images are those of
// the frame in one piece (each slot is traced by the same code either way).
// Separate graphs rather than one graph with a branch per band: the runtime
// was measured to run such branches one after another.
void launch_frame_graph(rgrt_ctx* c, const rgrt_instance* in, uint32_t n, uint32_t flags)
{
    hipStream_t s = c->stream;
    const bool timing = (c->flags & RGRT_CFG_TIMING) != 0;
    if(timing) {
        make_event(c->evFrameStart);
        make_event(c->evFrameEnd);
    }
    // the instance count and tables the captured kernels read
    const uint32_t prevInstances = c->numInstances;
    const bool prevHave = c->haveTlas;
    c->numInstances = n;
    c->haveTlas = true;
    const uint32_t bands = c->bands;
    try {
        if(bands == 1) {
            capture_into(&c->frameExec, s, [&]() { frame_enqueue(c, n, flags); });
        }
        else {
            capture_into(&c->preExec, s, [&]() { frame_enqueue_tlas(c, n, flags); });
            for(uint32_t b = 0; b < bands; ++b) {
                hipStream_t bs = b ? c->bandStream[b] : s;
                capture_into(&c->bandExec[b], bs, [&]() { enqueue_band(c, b, bands, bs); });
            }
            capture_into(&c->postExec, s, [&]() {
                launch_finalize_samples(s, shade_params(c));
                launch_post(s, c->img, c->ubo, (flags & RGRT_FRAME_FXAA) ? 1 : 0, nullptr);
            });
        }
    }
    catch(...) {
        c->numInstances = prevInstances;
        c->haveTlas = prevHave;
        throw;
    }
    if(timing) check(hipEventRecord(c->evFrameStart, s));
    if(bands == 1) {
        check(hipGraphLaunch(c->frameExec, s));
    }
    else {
        check(hipGraphLaunch(c->preExec, s));
        check(hipEventRecord(c->bandFork, s));
        for(uint32_t b = 1; b < bands; ++b) {
            check(hipStreamWaitEvent(c->bandStream[b], c->bandFork, 0));
            check(hipGraphLaunch(c->bandExec[b], c->bandStream[b]));
            check(hipEventRecord(c->bandJoin[b], c->bandStream[b]));
        }
        check(hipGraphLaunch(c->bandExec[0], s));
        for(uint32_t b = 1; b < bands; ++b) check(hipStreamWaitEvent(s, c->bandJoin[b], 0));
        check(hipGraphLaunch(c->postExec, s));
        const uint32_t passes = std::min<uint32_t>(c->tuning.wavefrontPasses, chain_iters(c));
        c->lastTraceLaunches = passes;
        c->lastDrained = true;
        c->lastWaves = passes;
        c->lastBands = bands;
    }
    if(timing) check(hipEventRecord(c->evFrameEnd, s));
    check(hipEventRecord(c->stageDone[c->stageIdx], s)); // this staging buffer is free after this frame
    frame_finish(c, in, n, flags);
    c->timedFrame = timing;
}
} // namespace

extern "C" {

rgrt_status rgrt_frame(rgrt_ctx* c, const rgrt_ubo* ubo, const rgrt_instance* in, uint32_t n, uint32_t flags)
{
    return guarded(c, [&]() {
        if(flags & ~(RGRT_FRAME_FXAA | RGRT_FRAME_REFIT_TLAS | RGRT_FRAME_GRAPH))
            return fail(c, RGRT_ERR_INVALID_ARG, "frame: unknown flags");
        const bool fxaa = (flags & RGRT_FRAME_FXAA) != 0;
        const bool refit = (flags & RGRT_FRAME_REFIT_TLAS) != 0;
        if(!(flags & RGRT_FRAME_GRAPH)) {
            // eager: the three calls of RenderSystem::render
            rgrt_status st = rgrt_set_frame(c, ubo);
            if(st != RGRT_OK) return st;
            st = refit ? rgrt_refit_tlas(c, in, n) : rgrt_build_tlas(c, in, n);
            if(st != RGRT_OK) return st;
            return rgrt_render(c, fxaa ? 1 : 0);
        }
        const rgrt_status st = frame_prepare(c, ubo, in, n, flags);
        if(st != RGRT_OK) return st;
        launch_frame_graph(c, in, n, flags);
        return RGRT_OK;
    });
}

} // extern "C"

struct rgrt_batch {
    std::vector<rgrt_ctx*> ctxs;
    hipGraphExec_t exec = nullptr;
    hipEvent_t fork = nullptr, done = nullptr;
    std::vector<hipEvent_t> join, pre;
    uint32_t mode = RGRT_BATCH_GRAPH_PER_SCENE;
    hipStream_t stream = nullptr; // ordered after every scene of each batch frame
    std::string err;
    // RGRT_BATCH_PERSISTENT: the scenes' kernel arguments in device memory
    // (two slots: a frame's slot is rewritten only after that frame ran),
    // the pass counters of the shared traversal launches, and the graph
    hipGraphExec_t pexec = nullptr;
    ShadeParams* dParams[2] = {nullptr, nullptr};
    TraceScene* dScenes[2] = {nullptr, nullptr};
    uint32_t* dStarts[2] = {nullptr, nullptr}; // block starts: raygen, rough/composite, FXAA (n + 1 each)
    hipEvent_t slotFree[2] = {nullptr, nullptr};
    int slot = 0;
    uint32_t* dCounters = nullptr;
    hipEvent_t fork2 = nullptr;
    std::vector<hipEvent_t> join2;
};

extern "C" {

rgrt_status rgrt_batch_create(rgrt_ctx* const* ctxs, uint32_t n, rgrt_batch** out)
{
    if(!out || !ctxs || n == 0) return RGRT_ERR_INVALID_ARG;
    *out = nullptr;
    for(uint32_t i = 0; i < n; ++i) {
        if(!ctxs[i]) return RGRT_ERR_INVALID_ARG;
        if(ctxs[i]->device != ctxs[0]->device) return RGRT_ERR_INVALID_ARG;
        for(uint32_t j = 0; j < i; ++j)
            if(ctxs[j] == ctxs[i]) return RGRT_ERR_INVALID_ARG;
    }
    auto* b = new rgrt_batch();
    b->ctxs.assign(ctxs, ctxs + n);
    try {
        check(hipSetDevice(ctxs[0]->device));
        check(hipEventCreateWithFlags(&b->fork, hipEventDisableTiming));
        check(hipEventCreateWithFlags(&b->done, hipEventDisableTiming));
        b->join.resize(n, nullptr);
        for(auto& e: b->join) check(hipEventCreateWithFlags(&e, hipEventDisableTiming));
        b->pre.resize(n, nullptr);
        for(auto& e: b->pre) check(hipEventCreateWithFlags(&e, hipEventDisableTiming));
        b->join2.resize(n, nullptr);
        for(auto& e: b->join2) check(hipEventCreateWithFlags(&e, hipEventDisableTiming));
        check(hipEventCreateWithFlags(&b->fork2, hipEventDisableTiming));
        check(hipStreamCreateWithFlags(&b->stream, hipStreamNonBlocking));
        if(n <= (uint32_t)kMaxBatchScenes) {
            for(int k = 0; k < 2; ++k) {
                check(hipMalloc((void**)&b->dParams[k], n * sizeof(ShadeParams)));
                check(hipMalloc((void**)&b->dScenes[k], n * sizeof(TraceScene)));
                check(hipMalloc((void**)&b->dStarts[k], 3 * (n + 1) * sizeof(uint32_t)));
                check(hipEventCreateWithFlags(&b->slotFree[k], hipEventDisableTiming));
            }
            check(hipMalloc((void**)&b->dCounters, 2 * sizeof(uint32_t)));
            check(hipMemsetAsync(b->dCounters, 0, 2 * sizeof(uint32_t), b->stream));
            check(hipStreamSynchronize(b->stream));
        }
    }
    catch(...) {
        rgrt_batch_destroy(b);
        return RGRT_ERR_HIP;
    }
    *out = b;
    return RGRT_OK;
}

void rgrt_batch_destroy(rgrt_batch* b)
{
    if(!b) return;
    for(rgrt_ctx* c: b->ctxs)
        if(c && c->stream) (void)hipStreamSynchronize(c->stream);
    if(b->exec) (void)hipGraphExecDestroy(b->exec);
    if(b->pexec) (void)hipGraphExecDestroy(b->pexec);
    for(int k = 0; k < 2; ++k) {
        if(b->dParams[k]) (void)hipFree(b->dParams[k]);
        if(b->dScenes[k]) (void)hipFree(b->dScenes[k]);
        if(b->dStarts[k]) (void)hipFree(b->dStarts[k]);
        if(b->slotFree[k]) (void)hipEventDestroy(b->slotFree[k]);
    }
    if(b->dCounters) (void)hipFree(b->dCounters);
    if(b->fork2) (void)hipEventDestroy(b->fork2);
    for(hipEvent_t e: b->join2)
        if(e) (void)hipEventDestroy(e);
    for(hipEvent_t e: b->join)
        if(e) (void)hipEventDestroy(e);
    for(hipEvent_t e: b->pre)
        if(e) (void)hipEventDestroy(e);
    if(b->stream) {
        (void)hipStreamSynchronize(b->stream);
        (void)hipStreamDestroy(b->stream);
    }
    if(b->fork) (void)hipEventDestroy(b->fork);
    if(b->done) (void)hipEventDestroy(b->done);
    delete b;
}

const char* rgrt_batch_last_error(const rgrt_batch* b) { return b ? b->err.c_str() : "null batch"; }

void* rgrt_batch_stream(rgrt_batch* b) { return b ? (void*)b->stream : nullptr; }

rgrt_status rgrt_batch_set_mode(rgrt_batch* b, uint32_t mode)
{
    if(!b || (mode != RGRT_BATCH_GRAPH_PER_SCENE && mode != RGRT_BATCH_ONE_GRAPH && mode != RGRT_BATCH_PERSISTENT))
        return RGRT_ERR_INVALID_ARG;
    if(mode == RGRT_BATCH_PERSISTENT && b->ctxs.size() > (size_t)kMaxBatchScenes) {
        b->err = "persistent batches hold at most " + std::to_string(kMaxBatchScenes) + " scenes";
        return RGRT_ERR_INVALID_ARG;
    }
    b->mode = mode;
    return RGRT_OK;
}

} // extern "C"

namespace {

// RGRT_BATCH_PERSISTENT: one graph on the first context's stream. Per scene
// (a branch on its own stream): instance upload and TLAS; then every scene
// together: ray generation, the passes (one traversal and one shading launch
// each, over every scene's queue), one drain launch, and the post passes
// (rough + composite, FXAA); per scene again only the sums of side-by-side
// samples and, with showAlpha, the post passes. The scenes' kernel
// arguments are in device memory (b->dParams / dScenes / dStarts, the slot of
// this frame).
rgrt_status batch_frame_persistent(rgrt_batch* b, const rgrt_frame_desc* descs)
{
    const uint32_t n = (uint32_t)b->ctxs.size();
    if(n > (uint32_t)kMaxBatchScenes || !b->dCounters) {
        b->err = "persistent batches hold at most " + std::to_string(kMaxBatchScenes) + " scenes";
        return RGRT_ERR_INVALID_ARG;
    }
    rgrt_ctx* c0 = b->ctxs[0];
    hipStream_t s0 = c0->stream;
    std::vector<uint32_t> prevN(n);
    std::vector<bool> prevHave(n);
    for(uint32_t i = 0; i < n; ++i) {
        prevN[i] = b->ctxs[i]->numInstances;
        prevHave[i] = b->ctxs[i]->haveTlas;
        b->ctxs[i]->numInstances = descs[i].numInstances;
        b->ctxs[i]->haveTlas = true;
    }
    try {
        check(hipSetDevice(c0->device));
        std::vector<ShadeParams> ps(n);
        std::vector<TraceScene> scs(n);
        uint32_t chain = 1;
        for(uint32_t i = 0; i < n; ++i) {
            ps[i] = shade_params(b->ctxs[i]);
            ps[i].st.segments = 1; // the merged launches take a scene's queue in one piece
            scs[i] = b->ctxs[i]->scene();
            chain = std::max(chain, chain_iters(b->ctxs[i]));
        }
        const uint32_t passes = std::min<uint32_t>(c0->tuning.wavefrontPasses, chain);
        // block starts of the merged launches
        std::vector<uint32_t> starts(3 * (n + 1), 0u);
        bool showAlpha = false, sampleSums = false;
        for(uint32_t i = 0; i < n; ++i) {
            const rgrt_ctx* c = b->ctxs[i];
            starts[i + 1] = starts[i] + (ps[i].st.npix + 255u) / 256u;
            starts[(n + 1) + i + 1] = starts[(n + 1) + i] + post_tiles(c->w, c->h);
            starts[2 * (n + 1) + i + 1] =
                starts[2 * (n + 1) + i] + ((descs[i].flags & RGRT_FRAME_FXAA) ? fxaa_tiles(c->w, c->h) : 0u);
            showAlpha = showAlpha || c->ubo.showAlpha;
            sampleSums = sampleSums || ps[i].st.groups > 1u;
        }
        const int slot = b->slot;
        b->slot ^= 1;
        check(hipEventSynchronize(b->slotFree[slot])); // the frame that used this slot has run
        check(hipMemcpy(b->dParams[slot], ps.data(), n * sizeof(ShadeParams), hipMemcpyHostToDevice));
        check(hipMemcpy(b->dScenes[slot], scs.data(), n * sizeof(TraceScene), hipMemcpyHostToDevice));
        check(hipMemcpy(b->dStarts[slot], starts.data(), starts.size() * sizeof(uint32_t), hipMemcpyHostToDevice));
        // work the scenes' own streams already hold comes before the batch
        for(uint32_t i = 1; i < n; ++i) {
            check(hipEventRecord(b->pre[i], b->ctxs[i]->stream));
            check(hipStreamWaitEvent(s0, b->pre[i], 0));
        }
        hipGraph_t g = nullptr;
        check(hipStreamBeginCapture(s0, hipStreamCaptureModeThreadLocal));
        uint32_t joined = 0, joined2 = 0;
        try {
            launch_zero_u32(s0, b->dCounters, 2);
            check(hipEventRecord(b->fork, s0));
            for(uint32_t i = 0; i < n; ++i) {
                rgrt_ctx* c = b->ctxs[i];
                hipStream_t s = c->stream;
                if(i) check(hipStreamWaitEvent(s, b->fork, 0));
                const uint32_t ni = descs[i].numInstances;
                if(ni)
                    check(hipMemcpyAsync(c->dInstIn, c->hInstStage[c->stageIdx], ni * sizeof(rgrt_instance),
                                         hipMemcpyHostToDevice, s));
                enqueue_tlas(c, ni, (descs[i].flags & RGRT_FRAME_REFIT_TLAS) != 0);
                if(i) {
                    check(hipEventRecord(b->join[i], s));
                    check(hipStreamWaitEvent(s0, b->join[i], 0));
                }
                joined = i + 1;
            }
            launch_raygen_multi(s0, b->dParams[slot], b->dStarts[slot], (int)n, starts[n]);
            bool oneSample = true;
            for(uint32_t i = 0; i < n; ++i) oneSample = oneSample && run_one_sample(ps[i]);
            int cur = 0;
            for(uint32_t it = 0; it < passes; ++it) {
                launch_trace_multi(s0, b->dParams[slot], b->dScenes[slot], (int)n, cur, c0->traceGrid, c0->spill, b->dCounters);
                launch_shade_multi(s0, b->dParams[slot], (int)n, cur, c0->shadeGrid, oneSample);
                cur ^= 1;
            }
            launch_drain_multi(s0, b->dParams[slot], b->dScenes[slot], (int)n, cur, c0->drainGrid, c0->spill, oneSample);
            if(sampleSums || showAlpha) {
                check(hipEventRecord(b->fork2, s0));
                for(uint32_t i = 0; i < n; ++i) {
                    rgrt_ctx* c = b->ctxs[i];
                    hipStream_t s = c->stream;
                    if(i) check(hipStreamWaitEvent(s, b->fork2, 0));
                    launch_finalize_samples(s, ps[i]);
                    if(showAlpha) launch_post(s, c->img, c->ubo, (descs[i].flags & RGRT_FRAME_FXAA) ? 1 : 0, nullptr);
                    if(i) {
                        check(hipEventRecord(b->join2[i], s));
                        check(hipStreamWaitEvent(s0, b->join2[i], 0));
                    }
                    joined2 = i + 1;
                }
            }
            if(!showAlpha)
                launch_post_multi(s0, b->dParams[slot], b->dStarts[slot] + (n + 1), (int)n, starts[2 * (n + 1) - 1],
                                  starts[3 * (n + 1) - 1]);
        }
        catch(...) {
            // join whatever branches were opened, then end the capture
            for(uint32_t i = 1; i < n && i <= joined; ++i) {
                (void)hipEventRecord(b->join[i], b->ctxs[i]->stream);
                (void)hipStreamWaitEvent(s0, b->join[i], 0);
            }
            for(uint32_t i = 1; i < n && i <= joined2; ++i) {
                (void)hipEventRecord(b->join2[i], b->ctxs[i]->stream);
                (void)hipStreamWaitEvent(s0, b->join2[i], 0);
            }
            (void)hipStreamEndCapture(s0, &g);
            if(g) (void)hipGraphDestroy(g);
            throw;
        }
        check(hipStreamEndCapture(s0, &g));
        update_exec(&b->pexec, g);
        check(hipGraphLaunch(b->pexec, s0));
        check(hipEventRecord(b->slotFree[slot], s0));
        check(hipEventRecord(b->done, s0));
        check(hipStreamWaitEvent(b->stream, b->done, 0));
        for(uint32_t i = 0; i < n; ++i) {
            rgrt_ctx* c = b->ctxs[i];
            check(hipEventRecord(c->stageDone[c->stageIdx], s0));
            if(i) check(hipStreamWaitEvent(c->stream, b->done, 0));
            frame_finish(c, descs[i].instances, descs[i].numInstances, descs[i].flags);
            c->timedFrame = false;
            c->lastTraceLaunches = passes;
            c->lastDrained = true;
            c->lastWaves = passes;
        }
    }
    catch(const std::exception& e) {
        for(uint32_t i = 0; i < n; ++i) {
            b->ctxs[i]->numInstances = prevN[i];
            b->ctxs[i]->haveTlas = prevHave[i];
        }
        b->err = e.what();
        return RGRT_ERR_HIP;
    }
    return RGRT_OK;
}

} // namespace

extern "C" {

rgrt_status rgrt_batch_frame(rgrt_batch* b, const rgrt_frame_desc* descs)
{
    if(!b || !descs) return RGRT_ERR_INVALID_ARG;
    const uint32_t n = (uint32_t)b->ctxs.size();
    // validation and staging, per context, before anything is captured
    for(uint32_t i = 0; i < n; ++i) {
        rgrt_ctx* c = b->ctxs[i];
        const rgrt_frame_desc& d = descs[i];
        const rgrt_status st =
            guarded(c, [&]() { return frame_prepare(c, d.ubo, d.instances, d.numInstances, d.flags | RGRT_FRAME_GRAPH); });
        if(st != RGRT_OK) {
            b->err = "scene " + std::to_string(i) + ": " + c->err;
            return st;
        }
    }
    rgrt_ctx* c0 = b->ctxs[0];
    hipStream_t s0 = c0->stream;
    if(b->mode == RGRT_BATCH_GRAPH_PER_SCENE) {
        // each scene's frame is one hipGraph on its own stream, after that
        // stream's earlier work only (no barrier between batch frames: a
        // scene's next frame starts while slower scenes still run); the
        // batch's stream then waits for all of them
        uint32_t i = 0;
        try {
            check(hipSetDevice(c0->device));
            for(; i < n; ++i) {
                rgrt_ctx* c = b->ctxs[i];
                launch_frame_graph(c, descs[i].instances, descs[i].numInstances, descs[i].flags | RGRT_FRAME_GRAPH);
                check(hipEventRecord(b->join[i], c->stream));
                check(hipStreamWaitEvent(b->stream, b->join[i], 0));
            }
        }
        catch(const std::exception& e) {
            b->err = "scene " + std::to_string(i) + ": " + e.what();
            return RGRT_ERR_HIP;
        }
        return RGRT_OK;
    }
    if(b->mode == RGRT_BATCH_PERSISTENT) return batch_frame_persistent(b, descs);
    std::vector<uint32_t> prevN(n);
    std::vector<bool> prevHave(n);
    for(uint32_t i = 0; i < n; ++i) {
        prevN[i] = b->ctxs[i]->numInstances;
        prevHave[i] = b->ctxs[i]->haveTlas;
        b->ctxs[i]->numInstances = descs[i].numInstances;
        b->ctxs[i]->haveTlas = true;
    }
    try {
        check(hipSetDevice(c0->device));
        // work the scenes' own streams already hold (vertex updates, BLAS
        // rebuilds) comes before the batch
        for(uint32_t i = 1; i < n; ++i) {
            check(hipEventRecord(b->pre[i], b->ctxs[i]->stream));
            check(hipStreamWaitEvent(s0, b->pre[i], 0));
        }
        // one graph, one branch per scene: the scenes' streams fork from and
        // join into the first scene's stream inside the capture
        hipGraph_t g = nullptr;
        check(hipStreamBeginCapture(s0, hipStreamCaptureModeThreadLocal));
        uint32_t joined = 0;
        try {
            check(hipEventRecord(b->fork, s0));
            for(uint32_t i = 0; i < n; ++i) {
                rgrt_ctx* c = b->ctxs[i];
                if(i) check(hipStreamWaitEvent(c->stream, b->fork, 0));
                frame_enqueue(c, descs[i].numInstances, descs[i].flags);
                if(i) {
                    check(hipEventRecord(b->join[i], c->stream));
                    check(hipStreamWaitEvent(s0, b->join[i], 0));
                }
                joined = i + 1;
            }
        }
        catch(...) {
            // join whatever branches were opened, then end the capture
            for(uint32_t i = 1; i < n && i <= joined; ++i) {
                (void)hipEventRecord(b->join[i], b->ctxs[i]->stream);
                (void)hipStreamWaitEvent(s0, b->join[i], 0);
            }
            (void)hipStreamEndCapture(s0, &g);
            if(g) (void)hipGraphDestroy(g);
            throw;
        }
        check(hipStreamEndCapture(s0, &g));
        update_exec(&b->exec, g);
        check(hipGraphLaunch(b->exec, s0));
        check(hipEventRecord(b->done, s0));
        check(hipStreamWaitEvent(b->stream, b->done, 0));
        for(uint32_t i = 0; i < n; ++i) {
            rgrt_ctx* c = b->ctxs[i];
            // the staging buffers are free and the scenes' later work is
            // ordered once the batch has run
            check(hipEventRecord(c->stageDone[c->stageIdx], s0));
            if(i) check(hipStreamWaitEvent(c->stream, b->done, 0));
            frame_finish(c, descs[i].instances, descs[i].numInstances, descs[i].flags);
            c->timedFrame = false;
        }
    }
    catch(const std::exception& e) {
        for(uint32_t i = 0; i < n; ++i) {
            b->ctxs[i]->numInstances = prevN[i];
            b->ctxs[i]->haveTlas = prevHave[i];
        }
        b->err = e.what();
        return RGRT_ERR_HIP;
    }
    return RGRT_OK;
}

static bool image_info(rgrt_ctx* c, rgrt_image which, void** ptr, uint64_t* bytes)
{
    const uint64_t npix = (uint64_t)c->w * c->h;
    Images& m = c->img;
    switch(which) {
    case RGRT_IMAGE_FINAL: *ptr = m.final_; *bytes = npix * 8; break;
    case RGRT_IMAGE_BASE: *ptr = m.base; *bytes = npix * 8; break;
    case RGRT_IMAGE_NORMAL: *ptr = m.normal; *bytes = npix * 8; break;
    case RGRT_IMAGE_ROUGH: *ptr = m.rough; *bytes = npix * 8; break;
    case RGRT_IMAGE_ROUGH_TRANSITIONS: *ptr = m.transitions; *bytes = npix; break;
    case RGRT_IMAGE_ROUGH_COLORS_A: *ptr = m.colorsA; *bytes = npix * 8; break;
    case RGRT_IMAGE_ROUGH_COLORS_B: *ptr = m.colorsB; *bytes = npix * 8; break;
    case RGRT_IMAGE_BASE_F32: *ptr = m.base32; *bytes = npix * 16; break;
    case RGRT_IMAGE_NORMAL_F32: *ptr = m.normal32; *bytes = npix * 16; break;
    case RGRT_IMAGE_ROUGH_F32: *ptr = m.rough32; *bytes = npix * 16; break;
    case RGRT_IMAGE_PRIMARY_HIT: *ptr = m.primary; *bytes = npix * sizeof(rgrt_hit); break;
    case RGRT_IMAGE_FEATURES: *ptr = m.features; *bytes = npix * 16; break;
    default: return false;
    }
    return *ptr != nullptr;
}

rgrt_status rgrt_read_image(rgrt_ctx* c, rgrt_image which, void* dst, uint64_t bytes)
{
    return guarded(c, [&]() {
        void* p = nullptr;
        uint64_t sz = 0;
        if(!image_info(c, which, &p, &sz)) return fail(c, RGRT_ERR_INVALID_ARG, "read_image: image not available");
        if(bytes != sz || !dst) return fail(c, RGRT_ERR_INVALID_ARG, "read_image: size mismatch");
        check(hipStreamSynchronize(c->stream));
        check(hipMemcpy(dst, p, sz, hipMemcpyDeviceToHost));
        return traversal_errors(c);
    });
}

} // extern "C"

struct rgrt_denoiser {
    rgrt_ctx* ctx;
    rgrt::Denoiser* d;
};

extern "C" {

rgrt_status rgrt_denoiser_create(rgrt_ctx* c, uint32_t seed, rgrt_denoiser** out)
{
    return guarded(c, [&]() {
        if(!out) return fail(c, RGRT_ERR_INVALID_ARG, "denoiser_create: null");
        *out = nullptr;
        auto* d = new Denoiser(seed);
        *out = new rgrt_denoiser{c, d};
        return RGRT_OK;
    });
}

void rgrt_denoiser_destroy(rgrt_denoiser* den)
{
    if(!den) return;
    (void)hipStreamSynchronize(den->ctx->stream);
    delete den->d;
    delete den;
}

rgrt_status rgrt_denoiser_num_params(rgrt_denoiser* den, uint64_t* count)
{
    if(!den || !count) return RGRT_ERR_INVALID_ARG;
    *count = den->d->num_params();
    return RGRT_OK;
}

rgrt_status rgrt_denoiser_get_params(rgrt_denoiser* den, float* params, uint64_t count)
{
    if(!den) return RGRT_ERR_INVALID_ARG;
    rgrt_ctx* c = den->ctx;
    return guarded(c, [&]() {
        if(!params || count != den->d->num_params()) return fail(c, RGRT_ERR_INVALID_ARG, "denoiser_get_params: count");
        den->d->get_params(c->stream, params);
        return RGRT_OK;
    });
}

rgrt_status rgrt_denoiser_set_params(rgrt_denoiser* den, const float* params, uint64_t count)
{
    if(!den) return RGRT_ERR_INVALID_ARG;
    rgrt_ctx* c = den->ctx;
    return guarded(c, [&]() {
        if(!params || count != den->d->num_params()) return fail(c, RGRT_ERR_INVALID_ARG, "denoiser_set_params: count");
        den->d->set_params(c->stream, params);
        return RGRT_OK;
    });
}

constexpr const char* kDenoiserBackwardOff =
    "the denoiser's backward pass is switched off: its weight-gradient kernel faulted the GPU and no cause has been "
    "found yet";

rgrt_status rgrt_denoiser_loss_and_grads(rgrt_denoiser* den, const uint16_t* x0, const float* target, uint32_t n,
                                         uint32_t h, uint32_t w, float* loss, float* grads, uint16_t* output)
{
    if(!den) return RGRT_ERR_INVALID_ARG;
    rgrt_ctx* c = den->ctx;
    return guarded(c, [&]() {
        if(!kDenoiserBackwardEnabled) return fail(c, RGRT_ERR_NOT_READY, kDenoiserBackwardOff);
        if(!x0 || !target || !loss || !n || !h || !w || h % 4 || w % 4 || (uint64_t)n * h * w > (1ull << 20))
            return fail(c, RGRT_ERR_INVALID_ARG, "denoiser_loss_and_grads: sizes (multiples of 4, at most 2^20 pixels)");
        *loss = den->d->loss_and_grads(c->stream, x0, target, (int)n, (int)h, (int)w, grads);
        if(output) den->d->read_output(c->stream, output);
        return RGRT_OK;
    });
}

rgrt_status rgrt_denoiser_infer(rgrt_denoiser* den, const uint16_t* x0, uint32_t n, uint32_t h, uint32_t w,
                                uint16_t* output)
{
    if(!den) return RGRT_ERR_INVALID_ARG;
    rgrt_ctx* c = den->ctx;
    return guarded(c, [&]() {
        if(!x0 || !output || !n || !h || !w || h % 4 || w % 4 || (uint64_t)n * h * w > (1ull << 22))
            return fail(c, RGRT_ERR_INVALID_ARG, "denoiser_infer: sizes (multiples of 4, at most 2^22 pixels)");
        den->d->infer(c->stream, x0, (int)n, (int)h, (int)w, output);
        return RGRT_OK;
    });
}

rgrt_status rgrt_denoiser_dataset_reserve(rgrt_denoiser* den, uint32_t count, uint32_t h, uint32_t w)
{
    if(!den) return RGRT_ERR_INVALID_ARG;
    rgrt_ctx* c = den->ctx;
    return guarded(c, [&]() {
        if(!count || !h || !w || h % 4 || w % 4) return fail(c, RGRT_ERR_INVALID_ARG, "denoiser_dataset_reserve: sizes");
        check(hipStreamSynchronize(c->stream));
        den->d->dataset_reserve(count, (int)h, (int)w);
        return RGRT_OK;
    });
}

rgrt_status rgrt_denoiser_dataset_add_input(rgrt_denoiser* den, uint32_t slot)
{
    if(!den) return RGRT_ERR_INVALID_ARG;
    rgrt_ctx* c = den->ctx;
    return guarded(c, [&]() {
        den->d->dataset_add_input(c->stream, c->img, slot);
        return RGRT_OK;
    });
}

rgrt_status rgrt_denoiser_dataset_add_target(rgrt_denoiser* den, uint32_t slot, float weight, int32_t accumulate)
{
    if(!den) return RGRT_ERR_INVALID_ARG;
    rgrt_ctx* c = den->ctx;
    return guarded(c, [&]() {
        den->d->dataset_add_target(c->stream, c->img, slot, weight, accumulate != 0);
        return RGRT_OK;
    });
}

rgrt_status rgrt_denoiser_dataset_read(rgrt_denoiser* den, uint32_t first, uint32_t count, uint32_t h, uint32_t w,
                                       uint16_t* x0, float* target)
{
    if(!den) return RGRT_ERR_INVALID_ARG;
    rgrt_ctx* c = den->ctx;
    return guarded(c, [&]() {
        den->d->dataset_read(c->stream, first, count, (int)h, (int)w, x0, target);
        return RGRT_OK;
    });
}

rgrt_status rgrt_denoiser_train(rgrt_denoiser* den, uint32_t steps, uint32_t batch, float lr, uint32_t seed, uint32_t used,
                                float* loss)
{
    if(!den) return RGRT_ERR_INVALID_ARG;
    rgrt_ctx* c = den->ctx;
    return guarded(c, [&]() {
        if(!kDenoiserBackwardEnabled) return fail(c, RGRT_ERR_NOT_READY, kDenoiserBackwardOff);
        if(!(lr > 0.0f)) return fail(c, RGRT_ERR_INVALID_ARG, "denoiser_train: learning rate");
        const float l = den->d->train(c->stream, steps, batch, lr, seed, used);
        if(loss) *loss = l;
        return RGRT_OK;
    });
}

rgrt_status rgrt_denoise(rgrt_denoiser* den, float fallbackA, float fallbackB, uint32_t* fallbackTiles, uint32_t* tiles)
{
    if(!den) return RGRT_ERR_INVALID_ARG;
    rgrt_ctx* c = den->ctx;
    return guarded(c, [&]() {
        if(!c->w || !c->h || c->w % 4 || c->h % 4)
            return fail(c, RGRT_ERR_INVALID_ARG, "denoise: render size must be a multiple of 4 in each direction");
        if(c->sampling.mode != RGRT_SAMPLING_STOCHASTIC)
            return fail(c, RGRT_ERR_NOT_READY, "denoise: the frame must be traced with RGRT_SAMPLING_STOCHASTIC");
        if(!den->d->has_trained_params())
            return fail(c, RGRT_ERR_NOT_READY,
                        "denoise: the network has no trained parameters (load them with rgrt_denoiser_set_params or "
                        "train it with rgrt_denoiser_train first)");
        const uint32_t nt = den->d->denoise(c->stream, c->img, fallbackA, fallbackB);
        if(tiles) *tiles = nt;
        if(fallbackTiles) *fallbackTiles = den->d->count_fallback(c->stream, nt);
        return RGRT_OK;
    });
}

rgrt_status rgrt_read_image_rgba8(rgrt_ctx* c, rgrt_image which, rgrt_format format, void* dst, uint64_t bytes)
{
    return guarded(c, [&]() {
        if(which != RGRT_IMAGE_FINAL && which != RGRT_IMAGE_BASE && which != RGRT_IMAGE_NORMAL && which != RGRT_IMAGE_ROUGH &&
           which != RGRT_IMAGE_ROUGH_COLORS_A && which != RGRT_IMAGE_ROUGH_COLORS_B)
            return fail(c, RGRT_ERR_INVALID_ARG, "read_image_rgba8: not an rgba16f image");
        if((uint32_t)format > (uint32_t)RGRT_FORMAT_BGRA8_SRGB) return fail(c, RGRT_ERR_INVALID_ARG, "read_image_rgba8: format");
        void* p = nullptr;
        uint64_t sz = 0;
        if(!image_info(c, which, &p, &sz)) return fail(c, RGRT_ERR_INVALID_ARG, "read_image_rgba8: image not available");
        const uint64_t npix = (uint64_t)c->w * c->h;
        if(bytes != npix * 4 || !dst) return fail(c, RGRT_ERR_INVALID_ARG, "read_image_rgba8: size mismatch");
        if(c->rgba8Cap < npix) {
            c->rgba8Cap = 0;
            dev_alloc(c->dRgba8, npix * 4);
            c->rgba8Cap = npix;
        }
        const int bgra = (format == RGRT_FORMAT_BGRA8_UNORM || format == RGRT_FORMAT_BGRA8_SRGB) ? 1 : 0;
        const int srgb = (format == RGRT_FORMAT_RGBA8_SRGB || format == RGRT_FORMAT_BGRA8_SRGB) ? 1 : 0;
        launch_to_rgba8(c->stream, static_cast<const uint16_t*>(p), c->dRgba8, npix, bgra, srgb);
        check(hipStreamSynchronize(c->stream));
        check(hipMemcpy(dst, c->dRgba8, npix * 4, hipMemcpyDeviceToHost));
        return traversal_errors(c);
    });
}

rgrt_status rgrt_write_image(rgrt_ctx* c, rgrt_image which, const void* src, uint64_t bytes)
{
    return guarded(c, [&]() {
        void* p = nullptr;
        uint64_t sz = 0;
        if(!image_info(c, which, &p, &sz)) return fail(c, RGRT_ERR_INVALID_ARG, "write_image: image not available");
        if(bytes != sz || !src) return fail(c, RGRT_ERR_INVALID_ARG, "write_image: size mismatch");
        check(hipStreamSynchronize(c->stream));
        check(hipMemcpy(p, src, sz, hipMemcpyHostToDevice));
        return RGRT_OK;
    });
}

rgrt_status rgrt_image_device_ptr(rgrt_ctx* c, rgrt_image which, void** dptr, uint64_t* bytes)
{
    return guarded(c, [&]() {
        void* p = nullptr;
        uint64_t sz = 0;
        if(!dptr || !image_info(c, which, &p, &sz)) return fail(c, RGRT_ERR_INVALID_ARG, "image_device_ptr: not available");
        *dptr = p;
        if(bytes) *bytes = sz;
        return RGRT_OK;
    });
}

rgrt_status rgrt_get_stats(rgrt_ctx* c, rgrt_stats* out)
{
    return guarded(c, [&]() {
        if(!out) return fail(c, RGRT_ERR_INVALID_ARG, "get_stats: null");
        check(hipStreamSynchronize(c->stream));
        std::memset(out, 0, sizeof(*out));
        if(c->st.counters) {
            // the counter blocks of the last frame's bands
            for(uint32_t b = 0; b < c->lastBands; ++b) {
                uint64_t cnt[3];
                check(hipMemcpy(cnt, c->st.counters + (size_t)kCounterBlock * b + 4, sizeof(cnt), hipMemcpyDeviceToHost));
                out->rays += cnt[0];
                out->skyLookups += cnt[1];
                out->zeroDirRays += cnt[2];
            }
        }
        out->waves = c->lastWaves;
        out->traceLaunches = c->lastTraceLaunches;
        out->drained = c->lastDrained ? 1u : 0u;
        if(c->timedAs) out->asBuildMs = elapsed(c->evAsStart, c->evAsEnd);
        if(c->timedRt) {
            out->rtOnlyMs = elapsed(c->evRtStart, c->evRtOnlyEnd);
            float tk = 0.0f, sk = 0.0f;
            for(uint32_t i = 0; i < c->lastTraceLaunches; ++i) {
                tk += elapsed(c->traceEvents[2 * i], c->traceEvents[2 * i + 1]);
                sk += elapsed(c->shadeEvents[2 * i], c->shadeEvents[2 * i + 1]);
            }
            out->traceKernelMs = tk;
            out->shadeKernelMs = sk;
            if(c->lastDrained) out->drainKernelMs = elapsed(c->evDrainStart, c->evDrainEnd);
        }
        if(c->timedPost) {
            out->roughMs = elapsed(c->evRtOnlyEnd, c->evRoughEnd);
            out->postprocMs = elapsed(c->evRtOnlyEnd, c->evPostEnd);
            out->rtTotalMs = elapsed(c->evRtStart, c->evPostEnd);
            if(c->timedAs) out->frameMs = elapsed(c->evAsStart, c->evPostEnd);
        }
        if(c->timedFrame) out->frameMs = elapsed(c->evFrameStart, c->evFrameEnd);
        return RGRT_OK;
    });
}

rgrt_status rgrt_set_tuning(rgrt_ctx* c, const rgrt_tuning* t)
{
    return guarded(c, [&]() {
        if(!t) return fail(c, RGRT_ERR_INVALID_ARG, "set_tuning: null");
        for(uint32_t v: {t->traceBlocksPerCU, t->shadeBlocksPerCU, t->drainBlocksPerCU})
            if(v < 1 || v > 32) return fail(c, RGRT_ERR_INVALID_ARG, "set_tuning: blocks per CU outside 1..32");
        if(t->hostLag < 1 || t->hostLag > 16) return fail(c, RGRT_ERR_INVALID_ARG, "set_tuning: hostLag outside 1..16");
        if(t->frameBands > kMaxBands) return fail(c, RGRT_ERR_INVALID_ARG, "set_tuning: frameBands outside 0..4");
        c->tuning = *t;
        c->apply_tuning();
        return RGRT_OK;
    });
}

rgrt_status rgrt_set_sample_groups(rgrt_ctx* c, uint32_t maxGroups)
{
    return guarded(c, [&]() {
        if(maxGroups > 32) return fail(c, RGRT_ERR_INVALID_ARG, "set_sample_groups: more than 32");
        c->sampleGroups = maxGroups;
        return RGRT_OK;
    });
}

rgrt_status rgrt_get_tuning(rgrt_ctx* c, rgrt_tuning* t)
{
    return guarded(c, [&]() {
        if(!t) return fail(c, RGRT_ERR_INVALID_ARG, "get_tuning: null");
        *t = c->tuning;
        return RGRT_OK;
    });
}

rgrt_status rgrt_get_pass_counts(rgrt_ctx* c, uint32_t* counts, uint32_t capacity, uint32_t* count)
{
    return guarded(c, [&]() {
        check(hipStreamSynchronize(c->stream));
        const uint32_t stride = c->lastBands > 1 ? c->passStride : 0u;
        const uint32_t n = std::min(c->lastTraceLaunches, c->hostCountsCap);
        if(count) *count = n;
        if(counts)
            for(uint32_t i = 0; i < std::min(n, capacity); ++i) {
                uint32_t v = 0;
                for(uint32_t b = 0; b < c->lastBands; ++b) v += c->hostCounts[(size_t)stride * b + i];
                counts[i] = v;
            }
        return RGRT_OK;
    });
}

} // extern "C"
