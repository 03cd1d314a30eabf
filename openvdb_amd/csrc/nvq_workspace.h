// When a stream's scratch block is reused, replaced or refused: plain C++, so that tests/test_workspace_cpu.py
// runs the rules without a GPU.
#pragma once
#include <stddef.h>

namespace nvq {

struct ScratchBlock {
    char* ptr = nullptr;
    size_t bytes = 0;
    bool captured = false; // recorded into a graph, whose replays use it at any later time
    size_t refused = 0;    // the smallest optional size that could not be had, 0: none
    unsigned asked = 0;    // optional requests of at least that size since
};

// A refused size is asked for again at every kRefusedAgain-th request: memory may have been given back.
constexpr unsigned kRefusedAgain = 64;

// The block, at least `bytes` long, or nullptr.  Mem: alloc(bytes) (nullptr on failure) and free(ptr), both in
// stream order.
// `capturing`: the launches to come are recorded into a graph.  They use the block only as it is: memory
// allocated during a capture belongs to the graph, and a free would become part of it.  From then on the
// block is never freed; a call that needs more takes another one beside it.
// `optional`: the caller does without.  The old block is then given up only once the larger one is there, and
// a size that was refused is not asked for on every call: where memory is short, each call would
// otherwise exchange the block for a large one in vain and back, and a stream-ordered free waits for
// the stream.
template<class Mem>
char* scratchAcquire(ScratchBlock& b, size_t bytes, bool capturing, bool optional, Mem&& mem)
{
    if (!b.ptr || b.bytes < bytes) {
        if (capturing) return nullptr;
        if (optional && b.refused && bytes >= b.refused && ++b.asked % kRefusedAgain) return nullptr;
        // room to grow: an eighth, at most 256 MiB
        const size_t eighth = bytes / 8, most = size_t(256) << 20, least = size_t(1) << 20;
        const size_t grown = bytes + (eighth < most ? eighth : most), want = grown > least ? grown : least;
        auto drop = [&]() {
            if (b.ptr && !b.captured) mem.free(b.ptr);
            b.ptr = nullptr;
            b.bytes = 0;
            b.captured = false;
        };
        if (!optional) drop();
        char* p = mem.alloc(want);
        if (!p) {
            if (optional && (!b.refused || bytes < b.refused)) {
                b.refused = bytes;
                b.asked = 0;
            }
            return nullptr;
        }
        if (optional) drop();
        b.ptr = p;
        b.bytes = want;
        if (bytes >= b.refused) b.refused = 0;
    }
    b.captured = b.captured || capturing;
    return b.ptr;
}

} // namespace nvq
