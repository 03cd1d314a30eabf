// Rules on sizes and indices that host code decides by: plain C++, so that tests/test_rules_cpu.py runs them
// without a GPU.  constexpr functions are callable from kernels too.
#pragma once
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

} // namespace nvq
