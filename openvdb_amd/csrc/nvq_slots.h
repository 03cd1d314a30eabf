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
//   brick[leaf] : 9^3 decoded floats, the leaf's voxels and the next one of its upper neighbours, so
//                 that the eight corners of any cell that starts in the leaf are four 8-byte loads
//                 from one base address, whatever the codec
// All values are ReadAccessor::getValue results, so the queries' outputs keep their bits.
#pragma once
#include "nvq_device.h"

#include <hip/hip_runtime.h>

namespace nvq {

// Entries: the brick number of the slot's leaf (ReadAccessor::getDim 1), or a tile (bit 31) with its
// getDim and state, or kSlotOther: a leaf under a render-skip flag, or on the rim of the table.
// Queries that meet kSlotOther, or leave the table, are answered through the accessor instead.
constexpr uint32_t kSlotTile = 0x80000000u, kSlotTileOn = 4u, kSlotOther = 0xffffffffu;
constexpr uint32_t kBrickEdge = 9, kBrickFloats = 736; // 729 used: 23 whole 128-byte lines

struct SlotMap {
    int32_t lo[3];  // first slot per axis
    uint32_t n[3];  // slots per axis
    const uint32_t* entry;
    const float* value;
    const float* brick;
    const uint32_t* tileIndex; // index grids: the channel index of a slot without a leaf
};

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

__device__ __forceinline__ bool slotCell(const SlotMap& M, int32_t x, int32_t y, int32_t z, SlotCell& c)
{
    uint32_t i;
    if (!slotAt(M, x, y, z, i)) return false;
    c.ox = x & ~7;
    c.oy = y & ~7;
    c.oz = z & ~7;
    c.entry = M.entry[i];
    // getDim of a tile: 8, 128 or 4096
    c.dim = (c.entry & kSlotTile) ? int32_t(8u << (4u * (c.entry & 3u) + ((c.entry & 3u) >> 1))) : 1;
    return c.entry != kSlotOther;
}

typedef float v2f __attribute__((ext_vector_type(2)));
__device__ __forceinline__ v2f loadPair(const float* p)
{
    v2f v;
    __builtin_memcpy(&v, p, 8); // one 8-byte load at 4-byte alignment
    return v;
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

// When a map pays: it costs about 45 us per million slots and 1.1 us per 1000 leaves (142 us for the
// 141,950 leaves of a 512^3 fog, 5 TB/s of leaves read and bricks written).  Against that stands the
// accessor's latency: one ray through that fog takes milliseconds, as its lookups wait for each other.
// So small launches take a map too, up to these sizes per launch and per ray; beyond them, and
// where a brick's offset would leave 32 bits, the accessor answers.
constexpr uint64_t kMaxMapSlots = uint64_t(1) << 24, kMapSlotsPerRay = 256, kMapSlotsFree = 1u << 20;
constexpr uint64_t kMaxMapLeaves = 1400000, kMapLeavesPerRay = 64, kMapLeavesFree = 1u << 18;

// Host side (nvq_slots.hip).  slotMapBytes: the scratch a map of grid g takes, or 0 when the call
// should go through the accessor: a bbox or leaf count out of proportion to its rays, or beyond
// the table's 32-bit offsets.  launchSlotMap builds it in `mem` (256-byte aligned).
size_t slotMapBytes(const GridView& g, uint64_t rays);
int launchSlotMap(const GridView& g, char* mem, SlotMap& M, hipStream_t s);

} // namespace nvq
