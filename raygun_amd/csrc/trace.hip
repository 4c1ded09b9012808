// trace.hip — traversal kernels: the wavefront queue pass and plain
// closest-hit queries (rgrt_trace_rays).
#pragma clang fp contract(off)

#include "rgrt_internal.h"
#include "traverse.h"

namespace rgrt {

namespace {

constexpr int kTraceBlock = 256;
constexpr int kLdsStack = 16;
constexpr int kSpill = 368; // with the 16 LDS entries: the 382-entry worst case of two wide LBVH levels

// Wavefront trace pass: rays [0, count) of queue `cur` -> hit records, and
// the rays queued ahead -> the frames that will need their hits. Waves fetch
// 64 rays at a time from a global counter (persistent grid).
// Waves per SIMD the traversal pass is compiled for: the register budget is
// 512 / waves VGPRs, its loop needs 94. At 6 waves (80, twelve spilled) 3,000
// small instances take 3.52 ms against 3.32 at 5, a 640x360 frame 0.466 against
// 0.446, 1080p over 2M triangles 7.47 against 7.17, 4K at 4 samples 86.2
// against 84.3.
#ifndef RGRT_TRACE_WAVES
#define RGRT_TRACE_WAVES 5
#endif

template<bool kAhead>
__global__ __launch_bounds__(kTraceBlock) __attribute__((amdgpu_waves_per_eu(RGRT_TRACE_WAVES))) void k_trace_queue(
    TraceScene sc, WavefrontState st, int cur, int32_t* __restrict__ spillBase, uint32_t* hostSlot)
{
    __shared__ int32_t ldsStack[kLdsStack * kTraceBlock];
    __shared__ QueueMap queue;
    uint32_t* counters = st.counters;
    const float* __restrict__ rays = st.rays[cur];
    float* __restrict__ hits = st.hits;
    const size_t npix = st.npix;
    const size_t aheadCap = npix * kAheadPerSlot;
    queue.load(st, cur);
    const uint32_t ahead = kAhead ? (uint32_t)min((size_t)counters[kAheadCountWord + cur], aheadCap) : 0u;
    if(blockIdx.x == 0 && threadIdx.x < kMaxSegments) { // the output queue of the shading pass that follows
        segment_counts(st, 1 - cur, threadIdx.x)[0] = 0;
        segment_counts(st, 1 - cur, threadIdx.x)[1] = 0;
    }
    if(blockIdx.x == 0 && threadIdx.x == 0) {
        *hostSlot = queue.count() + ahead; // host-visible: lets the host stop once the queues drain
        counters[kAheadCountWord + (1 - cur)] = 0;
        counters[2 + (1 - cur)] = 0; // the fetch counter of the next traversal pass
        // ray statistics (64-bit) at counters[4..5]
        atomicAdd(reinterpret_cast<unsigned long long*>(counters + 4), (unsigned long long)queue.count() + ahead);
    }
    const int lane = threadIdx.x & 63;
    const uint32_t gtid = blockIdx.x * kTraceBlock + threadIdx.x;
    __shared__ float boxRay[kBoxRayWords * kTraceBlock];
    TraversalStack<kLdsStack, kTraceBlock, kSpill> stack{ldsStack, spillBase + (size_t)gtid * kSpill, (int)threadIdx.x, boxRay};
    uint32_t* fetch = counters + 2 + cur;
    // The work is cut into chunks of 64 rays: the queue's, then those of the
    // rays queued ahead. Wave w first takes chunks w, w + waves, ... (three
    // quarters of its share, at least one); the rest are fetched from a counter,
    // which evens out the waves. A pass with fewer rays than the grid has lanes
    // does no atomics at all.
    const uint32_t wavesInGrid = gridDim.x * (kTraceBlock / 64);
    const uint32_t mainChunks = queue.chunks();
    const uint32_t chunks = mainChunks + (ahead + 63u) / 64u;
    const uint32_t rounds = max(1u, chunks * 3u / (wavesInGrid * 4u));
    uint32_t k = blockIdx.x * (kTraceBlock / 64) + (threadIdx.x >> 6);
    for(uint32_t round = 1; k < chunks; ++round) {
        const bool isAhead = kAhead && k >= mainChunks;
        uint32_t i;
        bool mine;
        if(isAhead) {
            i = (k - mainChunks) * 64u + lane;
            mine = i < ahead;
        }
        else {
            uint32_t within = k;
            const uint32_t s = queue.segment((uint32_t)lane, within);
            mine = queue.span(st, s).entry(within, (uint32_t)lane, i);
        }
        if(mine) {
            RayIn r;
            uint32_t mask, slot = 0;
            if(isAhead) {
                const float* q = st.ahead + i;
                r.ox = q[0 * aheadCap];
                r.oy = q[1 * aheadCap];
                r.oz = q[2 * aheadCap];
                r.dx = q[3 * aheadCap];
                r.dy = q[4 * aheadCap];
                r.dz = q[5 * aheadCap];
                slot = __float_as_uint(q[6 * aheadCap]);
                r.tmin = kAheadTmin;
                r.tmax = kAheadTmax;
                mask = 0xffu;
            }
            else {
                r.ox = rays[0 * npix + i];
                r.oy = rays[1 * npix + i];
                r.oz = rays[2 * npix + i];
                r.tmin = rays[3 * npix + i];
                r.dx = rays[4 * npix + i];
                r.dy = rays[5 * npix + i];
                r.dz = rays[6 * npix + i];
                r.tmax = rays[7 * npix + i];
                mask = (__float_as_uint(rays[9 * npix + i]) >> kMaskShift) & 0xffu;
            }
            const HitRec h = traverse<RGRT_INST_EVERY>(sc, r, mask, stack);
            if(isAhead) { // into the frame that waits for it (store_frame)
                const uint32_t level = (slot >> kAheadLevelShift) & 7u, kind = slot >> kAheadKindShift;
                float* b = st.frames + ((size_t)level * st.frameSlots + (slot & (kAheadMaxSlots - 1u))) * kFrameStrideAhead;
                reinterpret_cast<float4*>(b)[3 + kind] = make_float4(h.t, h.u, h.v, __uint_as_float(h.inst));
                b[20 + kind] = __uint_as_float(h.prim);
            }
            else {
                hits[0 * npix + i] = h.t;
                hits[1 * npix + i] = h.u;
                hits[2 * npix + i] = h.v;
                hits[3 * npix + i] = __uint_as_float(h.inst);
                hits[4 * npix + i] = __uint_as_float(h.prim);
            }
        }
        if(chunks <= wavesInGrid) break; // no rays beyond the first chunks
        if(round < rounds) {
            k += wavesInGrid;
            continue;
        }
        uint32_t b = 0;
        if(lane == 0) b = rounds * wavesInGrid + atomicAdd(fetch, 1u);
        k = __shfl(b, 0);
    }
}

// Traversal pass of a whole batch: the queues `cur` of every scene in one
// launch. The work is cut into 64-ray chunks per scene (a chunk never spans
// two scenes, so a wave traces one scene at a time); wave w first takes
// chunk w, then chunks from the batch's counter. Block 0 does each scene's
// bookkeeping of a pass: clears the output queue and the drain's fetch
// counter, adds the queue to the ray statistics, and clears the batch
// counter of the next pass.
__global__ __launch_bounds__(kTraceBlock) __attribute__((amdgpu_waves_per_eu(RGRT_TRACE_WAVES))) void k_trace_multi(
    const ShadeParams* __restrict__ ps, const TraceScene* __restrict__ scs, int numScenes, int cur,
    int32_t* __restrict__ spillBase, uint32_t* __restrict__ batchCounters)
{
    __shared__ int32_t ldsStack[kLdsStack * kTraceBlock];
    __shared__ uint32_t chunkEnd[kMaxBatchScenes];
    const int lane = threadIdx.x & 63;
    if(threadIdx.x < 64) {
        uint32_t count = 0, v = 0;
        if(lane < numScenes) {
            const QueueSpan queue(ps[lane].st, cur, 0u);
            count = queue.count();
            v = queue.chunks;
        }
        for(int off = 1; off < 64; off <<= 1) {
            const uint32_t u = __shfl_up(v, off);
            if(lane >= off) v += u;
        }
        if(lane < numScenes) chunkEnd[lane] = v;
        if(blockIdx.x == 0) {
            if(lane < numScenes) {
                uint32_t* counters = ps[lane].st.counters;
                segment_counts(ps[lane].st, 1 - cur, 0u)[0] = 0; // the output queue of the shading pass that follows
                segment_counts(ps[lane].st, 1 - cur, 0u)[1] = 0;
                counters[2 + (1 - cur)] = 0; // the fetch counter of the drain
                atomicAdd(reinterpret_cast<unsigned long long*>(counters + 4), (unsigned long long)count);
            }
            if(lane == 0) batchCounters[1 - cur] = 0;
        }
    }
    __syncthreads();
    const uint32_t chunks = chunkEnd[numScenes - 1];
    const uint32_t gtid = blockIdx.x * kTraceBlock + threadIdx.x;
    __shared__ float boxRay[kBoxRayWords * kTraceBlock];
    TraversalStack<kLdsStack, kTraceBlock, kSpill> stack{ldsStack, spillBase + (size_t)gtid * kSpill, (int)threadIdx.x, boxRay};
    const uint32_t wavesInGrid = gridDim.x * (kTraceBlock / 64);
    uint32_t k = blockIdx.x * (kTraceBlock / 64) + (threadIdx.x >> 6);
    for(;;) {
        if(k >= chunks) break;
        const int s = __builtin_amdgcn_readfirstlane(__popcll(__ballot(lane < numScenes && chunkEnd[lane < numScenes ? lane : 0] <= k)));
        const uint32_t first = s ? chunkEnd[s - 1] : 0u;
        const WavefrontState& st = ps[s].st;
        uint32_t i;
        if(QueueSpan(st, cur, 0u).entry(k - first, (uint32_t)lane, i)) {
            const size_t npix = st.npix;
            const float* __restrict__ rays = st.rays[cur];
            float* __restrict__ hits = st.hits;
            const TraceScene sc = scs[s];
            RayIn r;
            r.ox = rays[0 * npix + i];
            r.oy = rays[1 * npix + i];
            r.oz = rays[2 * npix + i];
            r.tmin = rays[3 * npix + i];
            r.dx = rays[4 * npix + i];
            r.dy = rays[5 * npix + i];
            r.dz = rays[6 * npix + i];
            r.tmax = rays[7 * npix + i];
            const uint32_t flags = __float_as_uint(rays[9 * npix + i]);
            const HitRec h = traverse<RGRT_INST_EVERY>(sc, r, (flags >> kMaskShift) & 0xffu, stack);
            hits[0 * npix + i] = h.t;
            hits[1 * npix + i] = h.u;
            hits[2 * npix + i] = h.v;
            hits[3 * npix + i] = __uint_as_float(h.inst);
            hits[4 * npix + i] = __uint_as_float(h.prim);
        }
        if(chunks <= wavesInGrid) break; // no chunks beyond the static share
        uint32_t b = 0;
        if(lane == 0) b = wavesInGrid + atomicAdd(batchCounters + cur, 1u);
        k = __shfl(b, 0);
    }
}

// Closest-hit queries over a persistent grid (the spill region is sized per
// launched thread); a hit's instance is reported by its customIndex. Chunks of
// `lanes` rays: the first rounds by position, the rest (calls of more rays than
// the grid has lanes) from the counter `fetch`, as in the queue pass.
template<int kInstEvery>
__global__ __launch_bounds__(kTraceBlock) __attribute__((amdgpu_waves_per_eu(RGRT_TRACE_WAVES))) void k_trace_rays(
    TraceScene sc, const rgrt_ray* __restrict__ rays, uint32_t n, uint32_t cullMask, rgrt_hit* __restrict__ hits,
    const InstanceShade* __restrict__ inst, int32_t* __restrict__ spillBase, uint32_t lanes, uint32_t* __restrict__ fetch)
{
    __shared__ int32_t ldsStack[kLdsStack * kTraceBlock];
    const uint32_t gtid = blockIdx.x * kTraceBlock + threadIdx.x;
    __shared__ float boxRay[kBoxRayWords * kTraceBlock];
    TraversalStack<kLdsStack, kTraceBlock, kSpill> stack{ldsStack, spillBase + (size_t)gtid * kSpill, (int)threadIdx.x, boxRay};
    const uint32_t lane = threadIdx.x & 63u;
    const uint32_t waves = gridDim.x * (kTraceBlock / 64);
    const uint32_t chunks = (n + lanes - 1u) / lanes;
    const uint32_t rounds = max(1u, (uint32_t)((uint64_t)chunks * 3u / (waves * 4u)));
    uint32_t k = blockIdx.x * (kTraceBlock / 64) + (threadIdx.x >> 6);
    for(uint32_t round = 1; k < chunks; ++round) {
        const uint32_t i = k * lanes + lane;
        if(lane < lanes && i < n) {
            const rgrt_ray rr = rays[i];
            RayIn r{rr.origin[0], rr.origin[1], rr.origin[2], rr.tmin, rr.dir[0], rr.dir[1], rr.dir[2], rr.tmax};
            const HitRec h = traverse<kInstEvery>(sc, r, cullMask & 0xffu, stack);
            rgrt_hit o;
            o.t = h.t;
            o.u = h.u;
            o.v = h.v;
            o.instance = h.inst < sc.numInstances ? inst[h.inst].customIndex : kNoHit;
            o.primitive = h.prim;
            hits[i] = o;
        }
        if(chunks <= waves) break; // no rays beyond the first chunks
        if(round < rounds) {
            k += waves;
            continue;
        }
        uint32_t b = 0;
        if(lane == 0) b = rounds * waves + atomicAdd(fetch, 1u);
        k = __shfl(b, 0);
    }
}

} // namespace

uint32_t trace_spill_words_per_thread() { return kSpill; }
uint32_t trace_block_size() { return kTraceBlock; }
// Blocks of the traversal pass a CU holds.
uint32_t trace_resident_blocks()
{
    int n = 0;
    check(hipOccupancyMaxActiveBlocksPerMultiprocessor(&n, k_trace_queue<false>, kTraceBlock, 0));
    return (uint32_t)std::max(1, n);
}

void launch_trace_queue_impl(hipStream_t s, const TraceScene& sc, const WavefrontState& st, int cur, uint32_t gridBlocks,
                             int32_t* spill, uint32_t* hostSlot, bool ahead)
{
    if(ahead) k_trace_queue<true><<<gridBlocks, kTraceBlock, 0, s>>>(sc, st, cur, spill, hostSlot);
    else k_trace_queue<false><<<gridBlocks, kTraceBlock, 0, s>>>(sc, st, cur, spill, hostSlot);
}

void launch_trace_multi(hipStream_t s, const ShadeParams* ps, const TraceScene* scs, int numScenes, int cur, uint32_t gridBlocks,
                        int32_t* spill, uint32_t* batchCounters)
{
    k_trace_multi<<<gridBlocks, kTraceBlock, 0, s>>>(ps, scs, numScenes, cur, spill, batchCounters);
}

namespace {
__global__ void k_zero_u32(uint32_t* p, uint32_t n)
{
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if(i < n) p[i] = 0u;
}
} // namespace

// Clears n words with a kernel (capturable into a graph, unlike a memset node).
void launch_zero_u32(hipStream_t s, uint32_t* p, uint32_t n)
{
    if(n) k_zero_u32<<<(n + 255) / 256, 256, 0, s>>>(p, n);
}

// Few rays are spread over the SIMDs, down to one per wave: a wave's loop then
// runs only the kind of step its rays are at, and entering an instance need not
// wait for other lanes' nodes. Alone, 100 rays over 64 instances take 134 -> 96
// us, 1024 rays 186 -> 123, 10,000 150 -> 133; 60,000 and more fill the waves.
// (The same in the passes of a frame changed nothing.) With the chunks past the
// first rounds fetched, 1M rays take 815 -> 715 us.
void launch_trace_rays_impl(hipStream_t s, const TraceScene& sc, const rgrt_ray* rays, uint32_t n, uint32_t cullMask,
                            rgrt_hit* hits, const InstanceShade* inst, int32_t* spill, uint32_t gridBlocks, uint32_t simds,
                            uint32_t* fetch)
{
    if(!n) return;
    uint32_t lanes = 64;
    while(lanes > 1 && n <= (uint64_t)simds * (lanes / 2)) lanes /= 2;
    const uint32_t chunks = (n + lanes - 1) / lanes;
    const uint32_t blocks = std::min<uint32_t>(gridBlocks, (chunks + kTraceBlock / 64 - 1) / (kTraceBlock / 64));
    if(chunks > blocks * (kTraceBlock / 64)) launch_zero_u32(s, fetch, 1);
    if(lanes < 8) k_trace_rays<1><<<blocks, kTraceBlock, 0, s>>>(sc, rays, n, cullMask, hits, inst, spill, lanes, fetch);
    else k_trace_rays<RGRT_INST_EVERY><<<blocks, kTraceBlock, 0, s>>>(sc, rays, n, cullMask, hits, inst, spill, lanes, fetch);
}

} // namespace rgrt
