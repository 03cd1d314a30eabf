"""The rules by which a stream's scratch block is reused, replaced and refused (nvq_workspace.h), on the host."""
from test_rules_cpu import run_cpp

MEM = """
    struct Mem {
        size_t room = ~size_t(0), held = 0;
        int allocs = 0, frees = 0;
        std::vector<char*> freed;
        char* alloc(size_t n) { ++allocs; return n <= room ? (held = n, new char[1]) : nullptr; }
        void free(char* p) { ++frees; freed.push_back(p); }
    } m;
    ScratchBlock b;
    const size_t MB = 1u << 20;
    auto say = [&](bool x) { std::printf("%d", x ? 1 : 0); };
"""


def check(tmp_path, body):
    out = run_cpp(tmp_path, MEM + body + 'std::printf("\\n");', ("nvq_workspace.h",))
    assert set(out[0]) == {"1"}, out[0]


def test_block_is_reused_and_grows(tmp_path):
    check(tmp_path, """
    char* p = scratchAcquire(b, 100, false, m);
    say(p && b.bytes == MB);
    say(scratchAcquire(b, MB, false, m) == p && m.allocs == 1);
    char* q = scratchAcquire(b, 16 * MB, false, m);
    say(q && q != p && b.bytes == 18 * MB && m.frees == 1 && m.freed[0] == p);
    say(scratchAcquire(b, 5, false, m) == q && m.allocs == 2);
    """)


def test_capture_neither_allocates_nor_frees(tmp_path):
    check(tmp_path, """
    say(!scratchAcquire(b, 100, true, m) && m.allocs == 0 && !b.captured);
    char* p = scratchAcquire(b, 100, false, m);
    say(!scratchAcquire(b, 2 * MB, true, m) && m.allocs == 1 && m.frees == 0 && b.ptr == p && !b.captured);
    say(scratchAcquire(b, MB, true, m) == p && b.captured);
    """)


def test_block_of_a_capture_is_never_freed(tmp_path):
    check(tmp_path, """
    char* p = scratchAcquire(b, 100, false, m);
    say(scratchAcquire(b, 100, true, m) == p);
    say(scratchAcquire(b, 100, false, m) == p); // eager calls go on sharing it, in stream order
    char* q = scratchAcquire(b, 4 * MB, false, m);
    say(q && q != p && m.frees == 0 && !b.captured);
    char* r = scratchAcquire(b, 8 * MB, false, m); // the new one was in no capture
    say(r && m.frees == 1 && m.freed[0] == q);
    """)
