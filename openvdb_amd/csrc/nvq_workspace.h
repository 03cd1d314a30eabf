// When a stream's scratch block is reused, replaced or refused: plain C++, so that tests/test_workspace_cpu.py
// runs the rules without a GPU.
#pragma once
#include <stddef.h>

namespace nvq {

struct ScratchBlock {
    char* ptr = nullptr;
    size_t bytes = 0;
    bool captured = false; // recorded into a graph, whose replays use it at any later time
};

// The block, at least `bytes` long, or nullptr.  Mem: alloc(bytes) (nullptr on failure) and free(ptr), both in
// stream order.
// `capturing`: the launches to come are recorded into a graph.  They use the block only as it is: memory
// allocated during a capture belongs to the graph, and a free would become part of it.  From then on the
// block is never freed; a call that needs more takes another one beside it.
template<class Mem>
char* scratchAcquire(ScratchBlock& b, size_t bytes, bool capturing, Mem&& mem)
{
    if (!b.ptr || b.bytes < bytes) {
        if (capturing) return nullptr;
        if (b.ptr && !b.captured) mem.free(b.ptr);
        b = ScratchBlock{};
        const size_t grown = bytes + bytes / 8, least = size_t(1) << 20, want = grown > least ? grown : least;
        b.ptr = mem.alloc(want);
        if (!b.ptr) return nullptr;
        b.bytes = want;
    }
    b.captured = b.captured || capturing;
    return b.ptr;
}

} // namespace nvq
