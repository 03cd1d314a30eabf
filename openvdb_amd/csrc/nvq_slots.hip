// Slot maps (nvq_slots.h): the flattened view of a grid that the ray queries read.
//   k_slot_entries : one tree walk per 8^3 slot of the bbox
//   k_slot_bricks  : one wavefront per leaf decodes its 9^3 brick (marches)
//   k_slot_signs   : one wavefront per leaf sets its active and sign bits (crossings)
#include "nvq_slots.h"
#include "nvq_internal.h"
#include "nvq_profile.h"

#include <hip/hip_runtime.h>

#include <algorithm>
#include <type_traits>

namespace nvq {
namespace {

constexpr int kThreads = 256;
constexpr uint64_t kSignBytes = 256; // per leaf

// Where one map is built.
struct MapMem {
    uint32_t *entry, *tileIndex, *slotOf, *leafOff, *leaves;
    float *value, *brick;
    uint8_t* signs;
    uint32_t count;
};

template<uint32_t GT>
__device__ __forceinline__ void slotEntries(const GridView& g, const SlotMap& M, const MapMem& W, uint32_t i)
{
    if (i >= W.count) return;
    const uint32_t z = i % M.n[2], r = i / M.n[2], y = r % M.n[1], x = r / M.n[1];
    Accessor<GT> acc(g);
    const Probe p = acc.probe((M.lo[0] + int32_t(x)) << 3, (M.lo[1] + int32_t(y)) << 3, (M.lo[2] + int32_t(z)) << 3);
    uint32_t e;
    if (!p.leaf) {
        e = kSlotTile | (p.active ? kSlotTileOn : 0u) | (p.dim == 8u ? 3u : (p.dim == 128u ? 7u : 12u));
    } else if (p.dim != 1u || x + 1u >= M.n[0] || y + 1u >= M.n[1] || z + 1u >= M.n[2]) {
        e = kSlotOther;
    } else {
        // bricks are numbered as the leaves are, where these have one size; FpN's are numbered as
        // the threads come (any order gives the same outputs).  A leaf outside the leaf array
        // (not laid out breadth first) has no number.
        const uint64_t off = uint64_t(p.leaf - g.leaf0);
        if constexpr (GT == GT_FPN) {
            e = kSlotOther;
            if ((off & 31u) == 0 && off < (uint64_t(1) << 37)) {
                const uint32_t b = atomicAdd(W.leaves, 1u);
                if (b < g.leafCount) {
                    W.leafOff[b] = uint32_t(off >> 5);
                    e = b;
                }
            }
        } else {
            const uint64_t b = off / g.leafSize;
            e = b < g.leafCount && b * g.leafSize == off ? uint32_t(b) : kSlotOther;
        }
    }
    W.entry[i] = e;
    W.value[i] = p.value;
    if (!(e & kSlotTile)) W.slotOf[e] = i;
    if constexpr (GT == GT_ONINDEX) W.tileIndex[i] = uint32_t(p.index); // used by the adjoint: < 2^31 values
}

// One wavefront per brick.  Lane l decodes row (x, y) = (l / 8, l % 8) of the leaf, one voxel of
// each facing layer of the three upper neighbours and, lanes 0..24, one of the layers' edges and
// corner; the brick is put together in LDS and written as whole 16-byte words.  All loads of a
// lane are independent.  Bound by HBM: the leaves are read and the bricks written once.
// One wavefront for the leaves of 16 slots in turn, each voxel on its own: 548 us for the
// 141,950 leaves of a 512^3 fog.
template<uint32_t GT>
__device__ __forceinline__ void slotBrick(const GridView& g, const SlotMap& M, const MapMem& W, uint32_t b, float* out)
{
    const uint32_t lane = threadIdx.x & 63u;
    if (b >= g.leafCount) return; // whole wavefronts; no barrier follows
    const uint32_t slot = __builtin_amdgcn_readfirstlane(W.slotOf[b]);
    // a number no slot was given (its leaf lies outside the table) holds what was there before
    if (slot >= W.count || M.entry[slot] != b) return;
    auto leafOf = [&](uint32_t e) {
        return g.leaf0 + (GT == GT_FPN ? uint64_t(W.leafOff[e]) << 5 : uint64_t(e) * g.leafSize);
    };
    // voxel (x, y, z) of the brick that lies in the neighbour slot above on the axes given
    auto beyond = [&](uint32_t x, uint32_t y, uint32_t z) -> float {
        // leaves on the table's rim are kSlotOther: the slot above exists on every axis
        const uint32_t s = slot + ((x >> 3) * M.n[1] + (y >> 3)) * M.n[2] + (z >> 3);
        const uint32_t e = M.entry[s];
        if (!(e & kSlotTile)) return Codec<GT>::get(leafOf(e), ((x & 7u) << 6) | ((y & 7u) << 3) | (z & 7u), g.channel);
        if (e != kSlotOther) return M.value[s];
        // a neighbour the table does not resolve: through the tree
        Accessor<GT> acc(g);
        const uint32_t sz = slot % M.n[2], r = slot / M.n[2], sy = r % M.n[1], sx = r / M.n[1];
        return acc.getValue(((M.lo[0] + int32_t(sx)) << 3) + int32_t(x), ((M.lo[1] + int32_t(sy)) << 3) + int32_t(y),
                            ((M.lo[2] + int32_t(sz)) << 3) + int32_t(z));
    };
    const uint32_t h = lane >> 3, l = lane & 7u;
    float row[8];
    leafRow<GT>(leafOf(b), lane, g.channel, row);
    const float fx = beyond(8u, h, l), fy = beyond(h, 8u, l), fz = beyond(h, l, 8u);
    // lanes 0..7: (8, l, 8); 8..15: (l, 8, 8); 16..23: (8, 8, l); 24: (8, 8, 8)
    const uint32_t ex = h == 1 ? l : 8u, ey = h == 0 ? l : 8u, ez = h == 2 ? l : 8u;
    const float fe = lane < 25u ? beyond(ex, ey, ez) : 0.0f;
#pragma unroll
    for (int k = 0; k < 8; ++k) out[h * 81u + l * 9u + k] = row[k];
    out[8u * 81u + h * 9u + l] = fx;
    out[h * 81u + 8u * 9u + l] = fy;
    out[h * 81u + l * 9u + 8u] = fz;
    if (lane < 25u) out[ex * 81u + ey * 9u + ez] = fe;
    __builtin_amdgcn_wave_barrier(); // the wavefront reads what its own lanes wrote, in LDS order
    const float4* src = reinterpret_cast<const float4*>(out);
    float4* dst = reinterpret_cast<float4*>(W.brick + uint64_t(b) * kBrickFloats);
#pragma unroll
    for (uint32_t j = 0; j < 3; ++j) {
        const uint32_t k = j * 64u + lane;
        if (k < (kBrickEdge * kBrickEdge * kBrickEdge + 3u) / 4u) dst[k] = src[k];
    }
}

// One wavefront per leaf.  Lane l takes byte l % 8 of block l / 8: voxels x & 3 = k / 2, y & 3 =
// 2 (k & 1) + {0, 1}, z & 3 = 0..3, as two rows of four.
template<uint32_t GT>
__device__ __forceinline__ void slotSigns(const GridView& g, const SlotMap& M, const MapMem& W, uint32_t b, float iso)
{
    const uint32_t lane = threadIdx.x & 63u;
    if (b >= g.leafCount) return;
    const uint32_t slot = __builtin_amdgcn_readfirstlane(W.slotOf[b]);
    if (slot >= W.count || M.entry[slot] != b) return; // as in slotBrick
    const uint8_t* leaf = g.leaf0 + (GT == GT_FPN ? uint64_t(M.leafOff[b]) << 5 : uint64_t(b) * g.leafSize);
    const uint32_t block = lane >> 3, k = lane & 7u;
    const uint32_t x = (block >> 2) * 4u + (k >> 1), y = ((block >> 1) & 1u) * 4u + (k & 1u) * 2u, z = (block & 1u) * 4u;
    const uint64_t word = ld_u64(leaf + kLeafVMask + 8u * x);
    uint32_t on = 0, below = 0, above = 0;
#pragma unroll
    for (uint32_t r = 0; r < 2; ++r) {
        const uint32_t n = (x << 6) | ((y + r) << 3) | z;
        on |= (uint32_t(word >> ((y + r) * 8u + z)) & 15u) << (4u * r);
        float v[4];
        if constexpr (GT == GT_FLOAT) {
            const float4 f = *reinterpret_cast<const float4*>(leaf + kLeafData + 4u * n);
            v[0] = f.x; v[1] = f.y; v[2] = f.z; v[3] = f.w;
        } else {
#pragma unroll
            for (uint32_t j = 0; j < 4; ++j) v[j] = Codec<GT>::get(leaf, n + j, g.channel);
        }
#pragma unroll
        for (uint32_t j = 0; j < 4; ++j) {
            const float d = v[j] - iso;
            below |= (d < 0.0f ? 1u : 0u) << (4u * r + j);
            above |= (d > 0.0f ? 1u : 0u) << (4u * r + j);
        }
    }
    uint8_t* out = W.signs + (uint64_t(b) * 8u + block) * 32u + k;
    out[0] = uint8_t(on);
    out[8] = uint8_t(below);
    out[16] = uint8_t(on);
    out[24] = uint8_t(above);
}

__device__ __forceinline__ uint32_t waveNumber() { return __builtin_amdgcn_readfirstlane(blockIdx.x * (kThreads / 64) + (threadIdx.x >> 6)); }

template<uint32_t GT>
__global__ __launch_bounds__(kThreads) void k_slot_entries(GridView g, SlotMap M, MapMem W)
{
    slotEntries<GT>(g, M, W, blockIdx.x * kThreads + threadIdx.x);
}
template<uint32_t GT>
__global__ __launch_bounds__(kThreads) void k_slot_bricks(GridView g, SlotMap M, MapMem W)
{
    __shared__ __align__(16) float stage[kThreads / 64][kBrickFloats];
    slotBrick<GT>(g, M, W, waveNumber(), stage[threadIdx.x >> 6]);
}
template<uint32_t GT>
__global__ __launch_bounds__(kThreads) void k_slot_signs(GridView g, SlotMap M, MapMem W, float iso)
{
    slotSigns<GT>(g, M, W, waveNumber(), iso);
}

// The maps of several grids, blockIdx.y the grid, its codec chosen at run time (scalar branches).
constexpr uint32_t kJobs = 8;
struct MapJobs {
    const GridView* view[kJobs];
    SlotMap map[kJobs];
    MapMem mem[kJobs];
};

__global__ void k_maps_store(MapJobs J, uint32_t n, SlotMap* __restrict__ maps)
{
    const uint32_t j = threadIdx.x;
    if (j >= n) return;
    maps[j] = J.map[j];
    if (J.mem[j].leaves) *J.mem[j].leaves = 0u;
}

template<class F>
__device__ __forceinline__ void byCodec(uint32_t type, F&& f)
{
    switch (type) {
    case GT_FLOAT: f(std::integral_constant<uint32_t, GT_FLOAT>{}); break;
    case GT_FP4: f(std::integral_constant<uint32_t, GT_FP4>{}); break;
    case GT_FP8: f(std::integral_constant<uint32_t, GT_FP8>{}); break;
    case GT_FP16: f(std::integral_constant<uint32_t, GT_FP16>{}); break;
    case GT_FPN: f(std::integral_constant<uint32_t, GT_FPN>{}); break;
    default: f(std::integral_constant<uint32_t, GT_ONINDEX>{}); break;
    }
}

__global__ __launch_bounds__(kThreads) void k_maps_entries(MapJobs J)
{
    const uint32_t j = blockIdx.y;
    if (blockIdx.x * kThreads >= J.mem[j].count) return;
    const GridView& g = *J.view[j];
    byCodec(g.type, [&](auto GT) {
        slotEntries<decltype(GT)::value>(g, J.map[j], J.mem[j], blockIdx.x * kThreads + threadIdx.x);
    });
}

__global__ __launch_bounds__(kThreads) void k_maps_leaves(MapJobs J)
{
    __shared__ __align__(16) float stage[kThreads / 64][kBrickFloats];
    const uint32_t j = blockIdx.y;
    const GridView& g = *J.view[j];
    if (!J.mem[j].count || blockIdx.x * (kThreads / 64) >= g.leafCount) return;
    byCodec(g.type, [&](auto GT) {
        if (J.mem[j].brick) slotBrick<decltype(GT)::value>(g, J.map[j], J.mem[j], waveNumber(), stage[threadIdx.x >> 6]);
        if (J.mem[j].signs) slotSigns<decltype(GT)::value>(g, J.map[j], J.mem[j], waveNumber(), 0.0f);
    });
}

__global__ void k_zero_word(uint32_t* p) { *p = 0u; }

size_t up256(size_t x) { return (x + 255) & ~size_t(255); }

template<uint32_t GT>
void launchMap(const GridView& g, const SlotMap& M, const MapMem& W, float iso, hipStream_t s)
{
    if (GT == GT_FPN) hipLaunchKernelGGL(k_zero_word, dim3(1), dim3(1), 0, s, W.leaves);
    hipLaunchKernelGGL(k_slot_entries<GT>, dim3((W.count + kThreads - 1) / kThreads), dim3(kThreads), 0, s, g, M, W);
    const dim3 waves((g.leafCount + kThreads / 64 - 1) / (kThreads / 64));
    if (g.leafCount && W.brick) hipLaunchKernelGGL(k_slot_bricks<GT>, waves, dim3(kThreads), 0, s, g, M, W);
    if (g.leafCount && W.signs) hipLaunchKernelGGL(k_slot_signs<GT>, waves, dim3(kThreads), 0, s, g, M, W, iso);
}

// Lays the map of g out in mem (slotMapBytes of it).
bool layMap(const GridView& g, char* mem, uint32_t parts, SlotMap& M, MapMem& W)
{
    const SlotBox box = slotBoxOf(g.bbox);
    const uint64_t count = box.count;
    if (!count) return false;
    for (int a = 0; a < 3; ++a) {
        M.lo[a] = box.lo[a];
        M.n[a] = box.n[a];
    }
    const uint64_t leaves = std::max<uint64_t>(g.leafCount, 1);
    auto take = [&](size_t bytes) {
        char* p = mem;
        mem += up256(bytes);
        return p;
    };
    W.count = uint32_t(count);
    W.entry = reinterpret_cast<uint32_t*>(take(4 * count));
    W.value = reinterpret_cast<float*>(take(4 * count));
    W.tileIndex = g.type == GT_ONINDEX ? reinterpret_cast<uint32_t*>(take(4 * count)) : nullptr;
    W.slotOf = reinterpret_cast<uint32_t*>(take(4 * leaves));
    W.leafOff = reinterpret_cast<uint32_t*>(take(4 * leaves));
    W.leaves = reinterpret_cast<uint32_t*>(take(4));
    W.brick = parts & kMapBricks ? reinterpret_cast<float*>(take(4ull * kBrickFloats * leaves)) : nullptr;
    W.signs = parts & kMapSigns ? reinterpret_cast<uint8_t*>(take(kSignBytes * leaves)) : nullptr;
    M.entry = W.entry;
    M.value = W.value;
    M.brick = W.brick;
    M.tileIndex = W.tileIndex;
    M.signs = reinterpret_cast<const uint4*>(W.signs);
    M.leafOff = W.leafOff;
    return true;
}

} // namespace

size_t slotMapBytes(const GridView& g, uint64_t rays, uint32_t parts, bool besides)
{
    const uint64_t count = slotBoxOf(g.bbox).count;
    if (!count) return 0;
    if (g.leafCount > kMaxMapLeaves) return 0;
    if (((parts & kMapBricks) || besides) &&
        (count > kMapSlotsPerRay * rays + kMapSlotsFree || g.leafCount > kMapLeavesPerRay * rays + kMapLeavesFree))
        return 0;
    const uint32_t leafBytes = g.type == GT_ONINDEX ? 96u + 2048u : g.leafSize; // with its channel's values
    if ((parts & kMapSigns) && !besides && !crossingMapPays(count, g.leafCount, leafBytes, g.type == GT_FPN, rays)) return 0;
    const uint64_t leaves = std::max<uint64_t>(g.leafCount, 1);
    return up256(4 * count) * (g.type == GT_ONINDEX ? 3 : 2) + up256(4 * leaves) * 2 + 256 +
           (parts & kMapBricks ? up256(4ull * kBrickFloats * leaves) : 0) + (parts & kMapSigns ? up256(kSignBytes * leaves) : 0);
}

int launchSlotMap(const GridView& g, char* mem, SlotMap& M, uint32_t parts, float iso, hipStream_t s)
{
    MapMem W;
    if (!layMap(g, mem, parts, M, W)) return -1;
    ProfScope prof("slot_map", s);
    switch (g.type) {
    case GT_FLOAT: launchMap<GT_FLOAT>(g, M, W, iso, s); break;
    case GT_FP4: launchMap<GT_FP4>(g, M, W, iso, s); break;
    case GT_FP8: launchMap<GT_FP8>(g, M, W, iso, s); break;
    case GT_FP16: launchMap<GT_FP16>(g, M, W, iso, s); break;
    case GT_FPN: launchMap<GT_FPN>(g, M, W, iso, s); break;
    case GT_ONINDEX: launchMap<GT_ONINDEX>(g, M, W, iso, s); break;
    default: return -3;
    }
    return hipGetLastError() == hipSuccess ? 0 : -4;
}

int launchSlotMaps(const MapJob* jobs, uint32_t n, SlotMap* maps, hipStream_t s)
{
    ProfScope prof("slot_map", s);
    for (uint32_t j0 = 0; j0 < n; j0 += kJobs) {
        const uint32_t m = std::min(kJobs, n - j0);
        MapJobs J{};
        uint32_t slots = 0, leaves = 0;
        for (uint32_t j = 0; j < m; ++j) {
            const MapJob& job = jobs[j0 + j];
            J.view[j] = job.device;
            if (!job.mem) continue;
            if (!layMap(*job.host, job.mem, job.parts, J.map[j], J.mem[j])) return -1;
            slots = std::max(slots, J.mem[j].count);
            leaves = std::max(leaves, job.host->leafCount);
        }
        hipLaunchKernelGGL(k_maps_store, dim3(1), dim3(64), 0, s, J, m, maps + j0);
        if (!slots) continue;
        hipLaunchKernelGGL(k_maps_entries, dim3((slots + kThreads - 1) / kThreads, m), dim3(kThreads), 0, s, J);
        if (leaves)
            hipLaunchKernelGGL(k_maps_leaves, dim3((leaves + kThreads / 64 - 1) / (kThreads / 64), m), dim3(kThreads), 0, s, J);
    }
    return hipGetLastError() == hipSuccess ? 0 : -4;
}

} // namespace nvq
