// Flattened view of a grid's tree for the ray queries, built per call in the stream's scratch.
//
// A ray crosses a leaf every few steps and samples two cells per voxel.  Through the accessor each
// of the eight corners of a cell is its own guarded lookup (cached leaf, else lower, upper, root),
// so a step waits for up to eight loads one after the other.  The slot map answers the same
// lookups with one table load per leaf-sized slot and independent loads at constant offsets per
// cell:
//   entry[slot] : for every 8^3 slot of the grid's bbox (one slot wider below, two above) the leaf
//                 that holds it, or the getDim and state of the tile that covers it
//   value[slot] : the value every voxel of a slot without a leaf reads (tile or background)
//   brick[leaf] (marches) : 9^3 decoded floats, the leaf's voxels and the next one of its upper
//                 neighbours, so that the eight corners of any cell that starts in the leaf are four 8-byte loads
//                 from one base address, whatever the codec
//   signs[leaf] (crossings) : per 4^3 block of the leaf the active bits of its voxels and the bits
//                 of those below and above the iso value, so that a ray walking through the narrow
//                 band reads 16 bytes per block instead of a value, a mask word and a flag per voxel
// All values are ReadAccessor::getValue results, so the queries' outputs keep their bits.
#pragma once
#include "nvq_device.h"
#include "nvq_rules.h"

#include <hip/hip_runtime.h>

namespace nvq {

// Entries: the brick number of the slot's leaf (ReadAccessor::getDim 1), or a tile (bit 31) with its
// getDim and state, or kSlotOther: a leaf under a render-skip flag, or on the rim of the table.
// Queries that meet kSlotOther, or leave the table, are answered through the accessor instead.
// A tile's bits: log2 of its getDim (3, 7 or 12) in 0..3, its state in 4.
constexpr uint32_t kSlotTile = 0x80000000u, kSlotTileOn = 16u, kSlotOther = 0xffffffffu;
constexpr uint32_t kBrickEdge = 9, kBrickFloats = 736; // 729 used: 23 whole 128-byte lines

struct SlotMap {
    int32_t lo[3];  // first slot per axis
    uint32_t n[3];  // slots per axis
    const uint32_t* entry;
    const float* value;
    const float* brick;
    const uint32_t* tileIndex; // index grids: the channel index of a slot without a leaf
    const uint4* signs;        // [leaf][block][2]: {active, below}, {active, above}
    const uint32_t* leafOff;   // FpN: offset of each leaf, in units of 32 bytes
};

constexpr uint32_t kMapBricks = 1u, kMapSigns = 2u; // what a map holds besides its table

// One slot as a march or crossing meets it.
struct SlotCell {
    int32_t ox, oy, oz; // slot origin (voxels)
    uint32_t entry;
    int32_t dim;        // getDim of its voxels: 1 in a leaf
};

__device__ __forceinline__ bool slotAt(const SlotMap& M, int32_t x, int32_t y, int32_t z, uint32_t& i)
{
    const uint32_t a = uint32_t((x >> 3) - M.lo[0]), b = uint32_t((y >> 3) - M.lo[1]), c = uint32_t((z >> 3) - M.lo[2]);
    i = (a * M.n[1] + b) * M.n[2] + c;
    return a < M.n[0] && b < M.n[1] && c < M.n[2];
}

__device__ __forceinline__ int32_t slotDim(uint32_t entry) { return (entry & kSlotTile) ? 1 << (entry & 15u) : 1; }

__device__ __forceinline__ bool slotCell(const SlotMap& M, int32_t x, int32_t y, int32_t z, SlotCell& c)
{
    uint32_t i;
    if (!slotAt(M, x, y, z, i)) return false;
    c.ox = x & ~7;
    c.oy = y & ~7;
    c.oz = z & ~7;
    c.entry = M.entry[i];
    c.dim = slotDim(c.entry);
    return c.entry != kSlotOther;
}

typedef float v2f __attribute__((ext_vector_type(2)));
__device__ __forceinline__ v2f loadPair(const float* p)
{
    v2f v;
    __builtin_memcpy(&v, p, 8); // one 8-byte load at 4-byte alignment
    return v;
}

// Decoded values of the eight voxels (x, y, 0..7) of a leaf, row = 8 x + y: one or two wide loads.
template<uint32_t GT>
__device__ __forceinline__ void leafRow(const uint8_t* leaf, uint32_t row, const float* channel, float v[8])
{
    if constexpr (GT == GT_FLOAT) {
        const float4* p = reinterpret_cast<const float4*>(leaf + kLeafData + 32u * row);
        const float4 a = p[0], b = p[1];
        v[0] = a.x; v[1] = a.y; v[2] = a.z; v[3] = a.w;
        v[4] = b.x; v[5] = b.y; v[6] = b.z; v[7] = b.w;
    } else if constexpr (GT == GT_FP16 || GT == GT_FP8 || GT == GT_FP4) {
        constexpr int kBits = GT == GT_FP16 ? 16 : (GT == GT_FP8 ? 8 : 4), kWords = kBits / 4;
        uint32_t w[kWords];
        __builtin_memcpy(w, leaf + kLeafData + row * uint32_t(kBits), sizeof(w));
#pragma unroll
        for (int k = 0; k < 8; ++k)
            v[k] = dequant(leaf, (w[k * kBits / 32] >> (k * kBits % 32)) & ((1u << kBits) - 1u));
    } else if constexpr (GT == GT_ONINDEX) {
        // the row is one byte of the value mask: its active voxels have consecutive indices
        const uint32_t w = row >> 3, shift = 8u * (row & 7u);
        const uint64_t word = ld_u64(leaf + kLeafVMask + 8u * w);
        uint64_t at = ld_u64(leaf + kIdxLeafOffset) + uint64_t(__popcll(word & ((uint64_t(1) << shift) - 1u)));
        if (w) at += (ld_u64(leaf + kIdxLeafPrefix) >> (9u * (w - 1u))) & 511u;
        const uint32_t bits = uint32_t(word >> shift) & 255u;
#pragma unroll
        for (int k = 0; k < 8; ++k) {
            const bool on = (bits >> k) & 1u;
            v[k] = channel[on ? at : 0u];
            at += on ? 1u : 0u;
        }
    } else {
#pragma unroll
        for (int k = 0; k < 8; ++k) v[k] = Codec<GT>::get(leaf, 8u * row + k, channel);
    }
}

// Corners of the cell at brick offset `at` (brick * kBrickFloats + (x * 9 + y) * 9 + z)
__device__ __forceinline__ void brickCell(const SlotMap& M, uint32_t at, Cell& c)
{
    const float* p = M.brick + at;
#pragma unroll
    for (int a = 0; a < 2; ++a)
#pragma unroll
        for (int b = 0; b < 2; ++b) {
            const v2f v = loadPair(p + (a * 9 + b) * 9);
            c.v[a][b][0] = v.x;
            c.v[a][b][1] = v.y;
        }
}

// trilerp of any cell, each corner through its own slot, one x layer at a time (the rare path: its
// registers count against the common one).  False when a corner lies outside the table or in a
// slot the table does not resolve.
__device__ __forceinline__ bool slotTrilinear(const SlotMap& M, float px, float py, float pz, float& out)
{
    const float fx = floorf(px), fy = floorf(py), fz = floorf(pz);
    const int32_t x = int32_t(fx), y = int32_t(fy), z = int32_t(fz);
    const float u = px - fx, v = py - fy, w = pz - fz;
    float layer[2] = {0.0f, 0.0f};
    bool ok = true;
#pragma unroll 1
    for (int a = 0; a < 2; ++a) {
        float c[4];
#pragma unroll
        for (int s = 0; s < 4; ++s) {
            uint32_t i;
            if (!slotAt(M, x + a, y + (s >> 1), z + (s & 1), i)) {
                i = 0;
                ok = false;
            }
            const uint32_t e = M.entry[i];
            ok = ok && e != kSlotOther;
            const uint32_t lx = uint32_t(x + a) & 7u, ly = uint32_t(y + (s >> 1)) & 7u, lz = uint32_t(z + (s & 1)) & 7u;
            c[s] = *((e & kSlotTile) ? M.value + i : M.brick + (e * kBrickFloats + (lx * 9u + ly) * 9u + lz));
        }
        layer[1] = lerpf(lerpf(c[0], c[1], w), lerpf(c[2], c[3], w), v);
        layer[0] = a ? layer[0] : layer[1];
    }
    out = lerpf(layer[0], layer[1], u);
    return ok;
}

// When a map pays.  Marches: it costs about 45 us per million slots and 1.1 us per 1000 leaves (142 us for the
// 141,950 leaves of a 512^3 fog, 5 TB/s of leaves read and bricks written).  Against that stands the
// accessor's latency: one ray through that fog takes 0.39 to 0.49 ms, as its lookups wait for each other,
// and 0.30 to 0.36 with the map; 64 rays 6.4 and 0.8 ms.  So small launches take a map too, up to these sizes per
// launch and per ray; beyond them, and where a brick's offset would leave 32 bits, the accessor
// answers.  (A launch whose rays all miss pays the map for nothing: 15 us and 166.)
// Crossings: crossingMapPays (nvq_rules.h).
constexpr uint64_t kMapSlotsPerRay = 256, kMapSlotsFree = 1u << 20;
constexpr uint64_t kMaxMapLeaves = 1400000, kMapLeavesPerRay = 64, kMapLeavesFree = 1u << 18;

// ------------------------------------------------------------------ crossings
__device__ __forceinline__ const uint8_t* slotLeaf(const SlotMap& M, const GridView& g, uint32_t e)
{
    return g.leaf0 + (g.type == GT_FPN ? uint64_t(M.leafOff[e]) << 5 : uint64_t(e) * g.leafSize);
}

// Voxel n of a leaf, the codec chosen at run time (the type is the same for the whole launch or
// ray tile, so the branch is scalar).
__device__ __forceinline__ float leafValue(const GridView& g, const uint8_t* leaf, uint32_t n)
{
    switch (g.type) {
    case GT_FLOAT: return Codec<GT_FLOAT>::get(leaf, n, g.channel);
    case GT_FP4: return Codec<GT_FP4>::get(leaf, n, g.channel);
    case GT_FP8: return Codec<GT_FP8>::get(leaf, n, g.channel);
    case GT_FP16: return Codec<GT_FP16>::get(leaf, n, g.channel);
    case GT_FPN: return Codec<GT_FPN>::get(leaf, n, g.channel);
    default: return Codec<GT_ONINDEX>::get(leaf, n, g.channel);
    }
}

// Value of voxel (x, y, z) in slot i with entry e (not kSlotOther).
__device__ __forceinline__ float slotVoxel(const SlotMap& M, const GridView& g, uint32_t i, uint32_t e, int32_t x,
                                           int32_t y, int32_t z)
{
    if (e & kSlotTile) return M.value[i];
    return leafValue(g, slotLeaf(M, g, e), Accessor<GT_FLOAT>::leafOffset(x, y, z));
}

// The corners of a cell, all lookups of a stage in flight together.  False: not resolved.
template<uint32_t GT>
__device__ __forceinline__ bool slotCornersOf(const SlotMap& M, const GridView& g, int32_t x, int32_t y, int32_t z, Cell& c)
{
    uint32_t i[8], e[8];
    bool ok = true;
#pragma unroll
    for (int s = 0; s < 8; ++s)
        if (!slotAt(M, x + (s >> 2), y + ((s >> 1) & 1), z + (s & 1), i[s])) {
            i[s] = 0;
            ok = false;
        }
#pragma unroll
    for (int s = 0; s < 8; ++s) {
        e[s] = M.entry[i[s]];
        ok = ok && e[s] != kSlotOther;
    }
#pragma unroll
    for (int s = 0; s < 8; ++s) {
        float v;
        if (e[s] & kSlotTile)
            v = M.value[i[s]];
        else
            v = Codec<GT>::get(slotLeaf(M, g, e[s]),
                               Accessor<GT>::leafOffset(x + (s >> 2), y + ((s >> 1) & 1), z + (s & 1)), g.channel);
        c.v[s >> 2][(s >> 1) & 1][s & 1] = v;
    }
    return ok;
}
__device__ __forceinline__ bool slotCorners(const SlotMap& M, const GridView& g, int32_t x, int32_t y, int32_t z, Cell& c)
{
    switch (g.type) {
    case GT_FLOAT: return slotCornersOf<GT_FLOAT>(M, g, x, y, z, c);
    case GT_FP4: return slotCornersOf<GT_FP4>(M, g, x, y, z, c);
    case GT_FP8: return slotCornersOf<GT_FP8>(M, g, x, y, z, c);
    case GT_FP16: return slotCornersOf<GT_FP16>(M, g, x, y, z, c);
    case GT_FPN: return slotCornersOf<GT_FPN>(M, g, x, y, z, c);
    default: return slotCornersOf<GT_ONINDEX>(M, g, x, y, z, c);
    }
}

// isoCrossingCore over a slot map: the same HDDA steps, states and comparisons.  `open` is set when
// the ray meets a slot the map does not resolve; it must then be answered through the accessor.
// Bound by the VALU (incoherent rays) or by the slowest tile's chain of iterations (images): reading
// the map into L2 first changed nothing.  So the walk keeps nothing but the HDDA and two bit words, and
// candidates are looked at outside of it.  1,000,003 scattered rays at a Fp16 torus: accessor 1177 us
// (475 M wavefront instructions with the walk and the look at candidates in one loop), 750 us (286 M).
// 512^2 image of a sphere 227 -> 141 us.  Selects in place of stepOnce's branches: 768 us.
__device__ __forceinline__ bool isoCrossingSlots(const SlotMap& M, const GridView& g, Ray& ray, float iso, int32_t c[3],
                                                 float& v, float& t, bool& open)
{
    if (!rayClip(ray, g.bbox) || double(ray.t1) > 1e20) return false;
    const float Delta = 1.0001f;
    float p[3];
    rayAt(ray, ray.t0, p);
    int32_t x = ifloor(p[0]), y = ifloor(p[1]), z = ifloor(p[2]);
    uint32_t i = 0, e = kSlotOther;
    if (slotAt(M, x, y, z, i)) e = M.entry[i];
    open = e == kSlotOther;
    if (open) return false;
    HDDA h;
    h.init(ray, ray.t0, ray.t1, slotDim(e));
    const float v0 = slotVoxel(M, g, i, e, x, y, z) - iso;
    // candidates are the active voxels on the other side of iso; the crossing itself is decided by
    // the product of the values, as it may underflow
    const uint4* signs = M.signs + (v0 > 0.0f ? 0 : 1);
    const bool some = v0 > 0.0f || v0 < 0.0f;
    // active and candidate bits of the 4^3 block (leaves) or the slot (tiles) of voxel (kx, ky, kz)
    uint32_t on0, on1, other0, other1;
    int32_t kx = x, ky = y, kz = z, dim = slotDim(e);
    auto block = [&]() {
        const uint32_t b = (uint32_t(kx) & 4u) | ((uint32_t(ky) & 4u) >> 1) | ((uint32_t(kz) & 4u) >> 2);
        const uint4 w = signs[(e * 8u + b) * 2u];
        on0 = w.x;
        on1 = w.y;
        other0 = w.z;
        other1 = w.w;
    };
    on0 = on1 = other0 = other1 = (e & kSlotTileOn) ? ~0u : 0u;
    if (!(e & kSlotTile)) block();
    bool band = false;
    for (;;) {
        bool candidate = false;
        while (h.stepOnce()) {
            rayAt(ray, h.t0 + Delta, p);
            x = band ? h.vx : ifloor(p[0]);
            y = band ? h.vy : ifloor(p[1]);
            z = band ? h.vz : ifloor(p[2]);
            const uint32_t dirty = uint32_t((x ^ kx) | (y ^ ky) | (z ^ kz));
            if (dirty & ~3u) {
                kx = x;
                ky = y;
                kz = z;
                if (dirty & ~7u) {
                    e = kSlotOther;
                    if (slotAt(M, x, y, z, i)) e = M.entry[i];
                    if (e == kSlotOther) break;
                    dim = slotDim(e);
                    on0 = on1 = other0 = other1 = (e & kSlotTileOn) ? ~0u : 0u; // of a tile
                }
                if (!(e & kSlotTile)) block();
            }
            const uint32_t n = ((uint32_t(x) & 1u) << 4) | ((uint32_t(y) & 3u) << 2) | (uint32_t(z) & 3u);
            const bool high = x & 2, active = ((high ? on1 : on0) >> n) & 1u;
            if (band) {
                candidate = active && (((high ? other1 : other0) >> n) & 1u) != 0;
                band = active; // the narrow band ends at an inactive voxel
                if (candidate) break;
            } else {
                if (h.dim != dim) h.update(ray, dim);
                band = dim == 1 && active;
            }
        }
        open = e == kSlotOther;
        if (!candidate || !some) return false;
        v = slotVoxel(M, g, i, e, x, y, z) - iso;
        if (v * v0 < 0) {
            c[0] = x;
            c[1] = y;
            c[2] = z;
            t = h.t0;
            return true;
        }
    }
}

// Host side (nvq_slots.hip).  slotMapBytes: the scratch a map of grid g takes, or 0 when the call
// should go through the accessor: a bbox or leaf count out of proportion to its rays, or beyond
// the table's 32-bit offsets.  launchSlotMap builds it in `mem` (256-byte aligned).
// `parts`: kMapBricks, kMapSigns (against `iso`).  `besides`: the call builds maps of other grids; a crossing's
// map then has a march's limits, as its tiles would otherwise wait for the launch after the others'.
size_t slotMapBytes(const GridView& g, uint64_t rays, uint32_t parts, bool besides = false);
// One map of a multi-grid call: the grid's view on the host and on the device, and the memory its map
// is built in (nullptr: none, and maps[j].entry is null).
struct MapJob {
    const GridView* host;
    const GridView* device;
    char* mem;
    uint32_t parts;
};
// Builds the maps of `n` grids (iso 0) with a few launches and stores them in maps[n], device memory.
int launchSlotMaps(const MapJob* jobs, uint32_t n, SlotMap* maps, hipStream_t s);
int launchSlotMap(const GridView& g, char* mem, SlotMap& M, uint32_t parts, float iso, hipStream_t s);

} // namespace nvq
