// Rules on sizes and indices that host code decides by: plain C++, so that tests/test_rules_cpu.py runs them
// without a GPU.  constexpr functions are callable from kernels too.
#pragma once
#include <cmath>
#include <stddef.h>
#include <stdint.h>

namespace nvq {

// ------------------------------------------------------------------ launches of four threads per tile
// Rows of at most 2^22 workgroups: a launch dimension of 2^32 threads or more is refused, which four
// threads per tile reach at 2^30 tiles, while a multi-grid call admits 2^31 - 1.
constexpr uint32_t kRowBlocks = 1u << 22;
struct LaunchRows {
    uint32_t x, y;
};
constexpr LaunchRows quadRows(uint32_t tiles, uint32_t threads)
{
    const uint64_t blocks = (uint64_t(tiles) + threads / 4u - 1u) / (threads / 4u);
    const uint64_t y = (blocks + kRowBlocks - 1u) / kRowBlocks;
    return y <= 1u ? LaunchRows{uint32_t(blocks), 1u} : LaunchRows{kRowBlocks, uint32_t(y)};
}
// The tile of a thread's quad: in 64 bits, as the thread's number in the launch passes 2^32.
constexpr uint64_t tileOfQuad(uint32_t blockX, uint32_t blockY, uint32_t thread, uint32_t threads)
{
    return (uint64_t(blockY) * kRowBlocks + blockX) * (threads / 4u) + (thread >> 2);
}

// ------------------------------------------------------------------ slot tables
// The 8^3 slots of a grid's bbox, one slot wider below and two above, so that a cell's eight corners and a
// brick's upper neighbours stay inside.
constexpr uint64_t kMaxMapSlots = uint64_t(1) << 24;
struct SlotBox {
    int32_t lo[3];  // first slot per axis
    uint32_t n[3];  // slots per axis
    uint64_t count; // 0: no table (an empty grid, coordinates whose neighbours could leave the int32 range, too many)
};
inline SlotBox slotBoxOf(const int32_t bbox[6])
{
    SlotBox b{};
    uint64_t count = 1;
    for (int a = 0; a < 3; ++a) {
        if (bbox[a] > bbox[3 + a] || bbox[a] < -(1 << 30) || bbox[3 + a] > (1 << 30)) return b;
        const int64_t l = (int64_t(bbox[a]) >> 3) - 1, h = (int64_t(bbox[3 + a]) >> 3) + 2;
        b.lo[a] = int32_t(l);
        b.n[a] = uint32_t(h - l + 1);
        count *= b.n[a];
        if (count > kMaxMapSlots) return b;
    }
    b.count = count;
    return b;
}

// The scratch that one call may take for maps and what goes with them (the adjoint's blocks): a stream keeps
// its block until the process ends.  A march's map is 2.9 KB per leaf, the adjoint's and its blocks 7 KB:
// 1.4 M and 2^20 leaves, the most they are built for, stay within it; of a multi-grid call's maps those that
// still fit are built, in order, and the other grids' tiles go through the accessor.
constexpr uint64_t kMaxMapBytes = uint64_t(8) << 30;
inline void boundMaps(size_t* bytes, uint32_t n, uint64_t most = kMaxMapBytes)
{
    for (uint32_t j = 0; j < n; ++j) {
        if (bytes[j] > most) bytes[j] = 0;
        most -= bytes[j];
    }
}

// Whether a crossing's rays pay for a map with sign bits.  A crossing through the accessor takes some hundred
// microseconds at most, however large its grid, so its map may cost no more than what its walk saves; all in
// microseconds, fitted to spheres of radius 30, 100, 400 and 800 and a torus (300, 80), 64 to 2^20 rays:
//   cost: 4 of launches, 45 per million slots, 0.55 per thousand Float leaves read and written (FpN: 1.5, its
//         leaves being numbered by an atomic)
//   saved: the grid's extent in slots (cube root of the table) times a factor that grows with the rays: 0.4 at
//         64 (one 8x8 tile at the torus: 72 us through the accessor, 83 with a map), 1 at 1000, 1.6 at
//         16,384, 3.1 at 2^18, 5.9 at 2^20
// Fewer than 64 rays go through the accessor: 17 to 20 us for one, 22 to 31 with a map (FpN torus: 73).
// 65,536 rays at the sphere of radius 800 (8.5 M slots): 590 us, 609 with a map; 2^18: 760 and 650.
inline bool crossingMapPays(uint64_t slots, uint64_t leaves, uint32_t leafBytes, bool fpn, uint64_t rays)
{
    if (rays < 64) return false;
    const double perLeaf = fpn ? 1.5e-3 : 0.55e-3 * (leafBytes + 256) / 2400.0;
    const double cost = 4.0 + 45e-6 * double(slots) + perLeaf * double(leaves);
    const double saved = std::cbrt(double(slots)) * (0.4 + 0.15 * std::log2(double(rays) / 64.0) + 3.3e-6 * double(rays));
    return cost <= saved;
}

// ------------------------------------------------------------------ block cache of the march's adjoint
constexpr uint32_t kCacheBlocks = 128;
constexpr uint32_t kNoBlock = 0xffffffffu;
// A block's tag is its linear position in the table's box, bx * sx + by * sy + bz.
struct BlockBox {
    uint32_t sx, sy;
};
// Strides of a block tag, at least the box's extents, with the low bits that spread best.  False: no cache (a
// position, slot * 64 + block, times 8 words would leave 32 bits, or a tag would).
inline bool blockBoxOf(const SlotBox& b, BlockBox& x)
{
    auto atLeast = [](uint64_t n, uint32_t low) {
        const uint64_t r = (n & ~uint64_t(kCacheBlocks - 1)) | low;
        return r < n ? r + kCacheBlocks : r;
    };
    if (b.count == 0 || b.count > (1u << 23)) return false;
    const uint64_t sy = atLeast(4ull * b.n[2], 19u), sx = atLeast(4ull * b.n[1] * sy, 45u);
    x.sy = uint32_t(sy);
    x.sx = uint32_t(sx);
    return 4ull * b.n[0] * sx < kNoBlock;
}

} // namespace nvq
