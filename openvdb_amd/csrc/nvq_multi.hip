// Persistent multi-grid ray query: one launch (after those that build the grids' slot maps) answers the
// rays of up to kMaxGrids grids of mixed leaf codecs and classes.  Wavefronts pull 8x8 ray tiles from a
// device work queue
// (forEachQueuedTile: chunks interleaved over one counter per XCD), costliest tiles first (a
// per-tile estimate, counting-sorted before the launch; the no-allocation variant keeps grid
// and image order), until every grid's tiles are taken (the persistent-warp pattern of the reference's iso-surface renderer,
// examples/ex_raytrace_iso_surface/common.h:79-110, 166-189), so small and large grids share
// the machine without per-grid launches or tail effects.  Level-set
// grids run zeroCrossing, fog volumes run the emission-absorption march.
#include "nvq_device.h"
#include "nvq_internal.h"
#include "nvq_profile.h"
#include "nvq_rays.h"
#include "nvq_rules.h"

#include <hip/hip_runtime.h>

#include <mutex>

// Work-queue counters of nvq_multi_query_noalloc (kQueueBands counters, kQueueStride words apart:
// 2 KiB).  Each device holds its own copy until the process ends; host code reaches it only
// through the device address hipGetSymbolAddress returns for that device.
static __device__ __align__(256) uint32_t scratch[nvq::kQueueBands * nvq::kQueueStride];

namespace nvq {
namespace {

template<uint32_t GT>
__device__ __forceinline__ void runRay(const GridView& g, uint32_t op, const float* eye, const float* dir, uint64_t i,
                                       float dt, float sigma, const CrossingOut& o)
{
    if (op == kOpZeroCrossing) zeroCrossingRay<GT>(g, eye, dir, i, 0.0f, o);
    else fogMarchRay<GT>(g, eye, dir, i, dt, sigma, o.t, o.v);
}

__device__ __forceinline__ void runTile(const MultiArgs& A, uint32_t t, const float* eye, const float* dir, float dt,
                                        float sigma, const CrossingOut& o)
{
    const uint32_t lane = threadIdx.x & 63u;
    uint32_t j = 0;
    while (j + 1 < A.k && A.slot[j + 1].tileBase <= t) ++j;
    const MultiSlot& S = A.slot[j];
    const uint32_t local = t - S.tileBase;
    const uint32_t tx = local % S.tilesX, ty = local / S.tilesX;
    const uint32_t px = tx * 8 + (lane & 7u), py = ty * 8 + (lane >> 3);
    const uint64_t i = S.rayBase + uint64_t(py) * S.width + px;
    // lanes outside the image or past a ragged last row idle; the wave stays together
    if (px < S.width && py < S.height && i < S.rayEnd) {
        const GridView g = *S.view;
        switch (g.type) {
        case GT_FLOAT: runRay<GT_FLOAT>(g, S.op, eye, dir, i, dt, sigma, o); break;
        case GT_FP4: runRay<GT_FP4>(g, S.op, eye, dir, i, dt, sigma, o); break;
        case GT_FP8: runRay<GT_FP8>(g, S.op, eye, dir, i, dt, sigma, o); break;
        case GT_FP16: runRay<GT_FP16>(g, S.op, eye, dir, i, dt, sigma, o); break;
        case GT_FPN: runRay<GT_FPN>(g, S.op, eye, dir, i, dt, sigma, o); break;
        default: runRay<GT_ONINDEX>(g, S.op, eye, dir, i, dt, sigma, o); break;
        }
    }
}

__global__ __launch_bounds__(kBlock) void k_multi_query(MultiArgs A, const float* __restrict__ eye,
                                                        const float* __restrict__ dir, float dt, float sigma,
                                                        uint32_t* __restrict__ counters,
                                                        const uint32_t* __restrict__ order, CrossingOut o)
{
    forEachQueuedTile<true>(counters, A.totalTiles, [&](uint32_t q) { runTile(A, order ? order[q] : q, eye, dir, dt, sigma, o); });
}

// The same over slot maps: one march and one crossing body for every codec.  A tile with a ray its map
// leaves open, or of a grid without a map, goes to the list `again`, which k_multi_again answers
// through the accessor.
// One step in flight and 7 wavefronts per SIMD (72 VGPRs): with both bodies in one kernel the crossings
// gain more from wavefronts than the marches from batches.  Sixteen Fp16 grids, 16.8 M rays: accessor
// 5.65 ms; 4 steps and 3 wavefronts 2.83, 4 and 4 2.51, 2 and 4 2.31, 2 and 6 2.24, 1 and 7 2.17.
// Marches alone, three fogs of 64^2, 256^2 and 1024^2 rays each: 0.86, 0.69 and 1.24 ms (accessor 3.8, 2.9, 5.3).
// Sixteen Fp16 grids: the VALU issues in 86 % of the slots of busy CUs, 21 % of wavefront
// cycles wait to issue.
__global__ __launch_bounds__(kBlock) __attribute__((amdgpu_waves_per_eu(7, 8))) void k_multi_slots(MultiArgs A, const SlotMap* __restrict__ maps,
                                                        const float* __restrict__ eye, const float* __restrict__ dir,
                                                        float dt, float sigma, uint32_t* __restrict__ counters,
                                                        const uint32_t* __restrict__ order,
                                                        uint32_t* __restrict__ again, uint32_t* __restrict__ count,
                                                        CrossingOut o)
{
    const uint32_t lane = threadIdx.x & 63u;
    forEachQueuedTile(counters, A.totalTiles, [&](uint32_t q) {
        const uint32_t t = __builtin_amdgcn_readfirstlane(order ? order[q] : q);
        uint32_t j = 0;
        while (j + 1 < A.k && A.slot[j + 1].tileBase <= t) ++j;
        const MultiSlot& S = A.slot[j];
        const uint32_t local = t - S.tileBase;
        const uint32_t tx = local % S.tilesX, ty = local / S.tilesX;
        const uint32_t px = tx * 8 + (lane & 7u), py = ty * 8 + (lane >> 3);
        const uint64_t i = S.rayBase + uint64_t(py) * S.width + px;
        bool open = false;
        if (px < S.width && py < S.height && i < S.rayEnd) {
            const SlotMap& M = maps[j];
            const GridView& g = *S.view;
            if (!M.entry) open = true;
            else if (S.op == kOpZeroCrossing) open = !zeroCrossingSlots(M, g, eye, dir, i, 0.0f, o);
            else open = !fogMarchSlots<1>(M, g, eye, dir, i, dt, sigma, o.t, o.v);
        }
        if (__any(open) && lane == 0) again[atomicAdd(count, 1u)] = t;
    });
}

__global__ __launch_bounds__(kBlock) void k_multi_again(MultiArgs A, const float* __restrict__ eye,
                                                        const float* __restrict__ dir, float dt, float sigma,
                                                        uint32_t* __restrict__ counters,
                                                        const uint32_t* __restrict__ again,
                                                        const uint32_t* __restrict__ count, CrossingOut o)
{
    const uint32_t n = *count;
    if (n == 0) return;
    forEachQueuedTile(counters, n, [&](uint32_t q) { runTile(A, again[q], eye, dir, dt, sigma, o); });
}

// Cost of a tile of the multi-grid launch for the longest-first queue order: the longest of its
// four corner rays inside its grid's bbox, a sixteenth of that for zeroCrossing.  A march steps every half voxel
// with a trilinear sample per step; zeroCrossing moves by nodes and leaves to the surface and
// stops at the first crossing, at far fewer probes per unit length.
// Four lanes per tile, one per corner: with one tile per wavefront, 262K tiles took 107 us.
__global__ __launch_bounds__(kBlock) void k_multi_tile_cost(MultiArgs A, const float* __restrict__ eye,
                                                            const float* __restrict__ dir, uint32_t* __restrict__ key)
{
    const uint32_t corner = threadIdx.x & 3u;
    const uint64_t tile = tileOfQuad(blockIdx.x, blockIdx.y, threadIdx.x, kBlock);
    if (tile >= A.totalTiles) return; // whole quads
    const uint32_t t = uint32_t(tile);
    float c = 0.0f;
    uint32_t j = 0;
    while (j + 1 < A.k && A.slot[j + 1].tileBase <= t) ++j;
    const MultiSlot& S = A.slot[j];
    const uint32_t local = t - S.tileBase;
    const uint32_t tx = local % S.tilesX, ty = local / S.tilesX;
    const uint32_t px = tx * 8 + (corner & 1u) * 7u, py = ty * 8 + (corner >> 1) * 7u;
    const uint64_t i = S.rayBase + uint64_t(py) * S.width + px;
    if (px < S.width && py < S.height && i < S.rayEnd) {
        c = clippedLength(*S.view, eye + 3 * i, dir + 3 * i);
        if (S.op == kOpZeroCrossing) c *= 0.0625f;
    }
    c = fmaxf(c, __shfl_xor(c, 1));
    c = fmaxf(c, __shfl_xor(c, 2));
    if (corner == 0) key[t] = costKey(c, t);
}

constexpr int kMaxDevices = 64;
std::mutex gScratchLock;
uint32_t* gScratch[kMaxDevices]; // device address of `scratch` on each device, set on first use

// Device address of `scratch` on device `dev`, which must be current: looked up once per device.
int scratchOn(int dev, uint32_t** out)
{
    if (dev < 0 || dev >= kMaxDevices) return -1;
    std::lock_guard<std::mutex> lock(gScratchLock);
    if (!gScratch[dev]) {
        void* p = nullptr;
        if (hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)) != hipSuccess || !p) return -1;
        gScratch[dev] = static_cast<uint32_t*>(p);
    }
    *out = gScratch[dev];
    return 0;
}

uint32_t queryBlocks(const MultiArgs& A, int cus)
{
    const uint64_t waves = A.totalTiles; // one wave per tile is the most that can be busy
    uint32_t blocks = uint32_t(cus) * 8u;
    if (uint64_t(blocks) * (kBlock / 64) > waves) blocks = uint32_t((waves + (kBlock / 64) - 1) / (kBlock / 64));
    return blocks == 0 ? 1 : blocks;
}

} // namespace

int multiQueryNoAlloc(const MultiArgs& A, const float* eye, const float* dir, float dt, float sigma, uint8_t* hit,
                      int32_t* ijk, float* a, float* b, float* normal, hipStream_t s)
{
    int dev = 0, cus = 0;
    if (hipGetDevice(&dev) != hipSuccess || hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess)
        return -1;
    uint32_t* counter = nullptr;
    if (scratchOn(dev, &counter) != 0) return -2;
    // the counters keep the previous call's values: clear them with a kernel (no memset node)
    hipLaunchKernelGGL(k_queue_reset, dim3(1), dim3(kQueueBands), 0, s, counter);
    hipLaunchKernelGGL(k_multi_query, dim3(queryBlocks(A, cus)), dim3(kBlock), 0, s, A, eye, dir, dt, sigma, counter,
                       nullptr, CrossingOut{hit, ijk, a, b, normal});
    return hipGetLastError() == hipSuccess ? 0 : -4;
}

int multiQuery(const MultiArgs& A, const GridView* const* views, const float* eye, const float* dir, float dt, float sigma,
               uint8_t* hit, int32_t* ijk, float* a, float* b, float* normal, hipStream_t s)
{
    int dev = 0, cus = 0;
    if (hipGetDevice(&dev) != hipSuccess || hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess)
        return -1;
    // queue counters (and those of the second launch), then the tile cost keys and the longest-first
    // order (4 bytes per tile each; none up to kOrderMinTiles tiles, which are all resident at once),
    // the list of tiles to answer again, and the grids' maps
    const bool ordered = A.totalTiles > kOrderMinTiles;
    auto up = [](size_t x) { return (x + 255) & ~size_t(255); };
    const size_t keyBytes = ordered ? up(size_t(A.totalTiles) * 4) : 0;
    const size_t countBytes = ordered ? up(orderScratchBytes(A.totalTiles)) : 0;
    const size_t need = 2 * kQueueBytes + 2 * keyBytes + countBytes;
    const size_t againBytes = 256 + up(size_t(A.totalTiles) * 4), mapBytes = up(sizeof(SlotMap) * kMaxGrids);
    MapJob jobs[kMaxGrids];
    size_t total = need + againBytes + mapBytes, at[kMaxGrids], bytes[kMaxGrids];
    // maps for all grids where one of them pays on its own: three level sets of 64 rays each 137 us with three
    // maps, 147 with none, 217 with two
    bool any = false;
    for (uint32_t j = 0; j < A.k; ++j) {
        const MultiSlot& S = A.slot[j];
        jobs[j] = MapJob{views[j], S.view, nullptr, S.op == kOpFogMarch ? kMapBricks : kMapSigns};
        any = any || (S.rayEnd > S.rayBase && slotMapBytes(*views[j], S.rayEnd - S.rayBase, jobs[j].parts));
    }
    for (uint32_t j = 0; j < A.k; ++j) {
        const uint64_t rays = A.slot[j].rayEnd - A.slot[j].rayBase;
        bytes[j] = any && rays ? slotMapBytes(*views[j], rays, jobs[j].parts, true) : 0;
    }
    boundMaps(bytes, A.k);
    for (uint32_t j = 0; j < A.k; ++j) {
        at[j] = total;
        total += bytes[j];
    }
    // no map on a captured stream, nor where the scratch cannot grow
    any = any && !isCapturing(s);
    WorkspaceLease lease;
    char* base = any ? lease.acquire(total, s, true) : nullptr;
    if (!base) {
        any = false;
        base = lease.acquire(need, s);
    }
    const CrossingOut o{hit, ijk, a, b, normal};
    const dim3 blocks(queryBlocks(A, cus));
    if (!base) {
        if (!lease.capturing()) return -2;
        // recorded without scratch: the tiles in turn
        hipLaunchKernelGGL(k_multi_query, blocks, dim3(kBlock), 0, s, A, eye, dir, dt, sigma, nullptr, nullptr, o);
        return hipGetLastError() == hipSuccess ? 0 : -4;
    }
    uint32_t* counter = reinterpret_cast<uint32_t*>(base);
    uint32_t* second = reinterpret_cast<uint32_t*>(base + kQueueBytes);
    uint32_t* key = reinterpret_cast<uint32_t*>(base + 2 * kQueueBytes);
    uint32_t* order = ordered ? reinterpret_cast<uint32_t*>(base + 2 * kQueueBytes + keyBytes) : nullptr;
    hipLaunchKernelGGL(k_queue_reset, dim3(1), dim3(kQueueBands), 0, s, counter);
    if (ordered) {
        ProfScope prof("tile_order", s);
        const LaunchRows rows = quadRows(A.totalTiles, kBlock);
        hipLaunchKernelGGL(k_multi_tile_cost, dim3(rows.x, rows.y), dim3(kBlock), 0, s, A, eye, dir, key);
        launchTileOrder(key, uint64_t(A.totalTiles), order,
                        reinterpret_cast<uint32_t*>(base + 2 * kQueueBytes + 2 * keyBytes), s);
    }
    if (any) {
        uint32_t* count = reinterpret_cast<uint32_t*>(base + need);
        uint32_t* again = reinterpret_cast<uint32_t*>(base + need + 256);
        SlotMap* maps = reinterpret_cast<SlotMap*>(base + need + againBytes);
        hipLaunchKernelGGL(k_queue_reset, dim3(1), dim3(kQueueBands), 0, s, second);
        hipLaunchKernelGGL(k_queue_reset, dim3(1), dim3(1), 0, s, count);
        for (uint32_t j = 0; j < A.k; ++j)
            if (bytes[j]) jobs[j].mem = base + at[j];
        if (launchSlotMaps(jobs, A.k, maps, s) != 0) return -4;
        ProfScope prof("k_multi_query", s);
        hipLaunchKernelGGL(k_multi_slots, blocks, dim3(kBlock), 0, s, A, maps, eye, dir, dt, sigma, counter, order, again,
                           count, o);
        hipLaunchKernelGGL(k_multi_again, blocks, dim3(kBlock), 0, s, A, eye, dir, dt, sigma, second, again, count, o);
    } else {
        ProfScope prof("k_multi_query", s);
        hipLaunchKernelGGL(k_multi_query, blocks, dim3(kBlock), 0, s, A, eye, dir, dt, sigma, counter, order, o);
    }
    return hipGetLastError() == hipSuccess ? 0 : -4;
}

} // namespace nvq
