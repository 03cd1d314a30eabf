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
    char* p = scratchAcquire(b, 100, false, false, m);
    say(p && b.bytes == MB);
    say(scratchAcquire(b, MB, false, false, m) == p && m.allocs == 1);
    char* q = scratchAcquire(b, 16 * MB, false, false, m);
    say(q && q != p && b.bytes == 18 * MB && m.frees == 1 && m.freed[0] == p);
    say(scratchAcquire(b, 5, false, false, m) == q && m.allocs == 2);
    say(scratchAcquire(b, 8192 * MB, false, false, m) && b.bytes == 8448 * MB); // an eighth, at most 256 MiB
    """)


def test_capture_neither_allocates_nor_frees(tmp_path):
    check(tmp_path, """
    say(!scratchAcquire(b, 100, true, false, m) && m.allocs == 0 && !b.captured);
    char* p = scratchAcquire(b, 100, false, false, m);
    say(!scratchAcquire(b, 2 * MB, true, false, m) && m.allocs == 1 && m.frees == 0 && b.ptr == p && !b.captured);
    say(scratchAcquire(b, MB, true, false, m) == p && b.captured);
    """)


def test_block_of_a_capture_is_never_freed(tmp_path):
    check(tmp_path, """
    char* p = scratchAcquire(b, 100, false, false, m);
    say(scratchAcquire(b, 100, true, false, m) == p);
    say(scratchAcquire(b, 100, false, false, m) == p); // eager calls go on sharing it, in stream order
    char* q = scratchAcquire(b, 4 * MB, false, false, m);
    say(q && q != p && m.frees == 0 && !b.captured);
    char* r = scratchAcquire(b, 8 * MB, false, false, m); // the new one was in no capture
    say(r && m.frees == 1 && m.freed[0] == q);
    """)


def test_optional_request_keeps_the_block_when_it_is_refused(tmp_path):
    check(tmp_path, """
    char* p = scratchAcquire(b, 100, false, false, m);
    m.room = 64 * MB;
    say(!scratchAcquire(b, 100 * MB, false, true, m) && b.ptr == p && b.bytes == MB && m.frees == 0);
    say(scratchAcquire(b, 100, false, false, m) == p && m.allocs == 2);
    // the same size, or more, is not asked for again on the next calls; less is
    for (int i = 1; i < 64; ++i) say(!scratchAcquire(b, (100 + i) * MB, false, true, m));
    say(m.allocs == 2 && m.frees == 0);
    char* q = scratchAcquire(b, 8 * MB, false, true, m);
    say(q && q != p && m.allocs == 3 && m.frees == 1 && m.freed[0] == p);
    """)


def test_refused_size_is_asked_for_again_in_time(tmp_path):
    check(tmp_path, """
    m.room = MB;
    say(!scratchAcquire(b, 100 * MB, false, true, m) && m.allocs == 1);
    m.room = ~size_t(0);
    int calls = 0;
    while (!scratchAcquire(b, 100 * MB, false, true, m)) ++calls;
    say(calls == int(kRefusedAgain) - 1 && m.allocs == 2 && b.refused == 0);
    """)


def test_needed_request_frees_first_and_ignores_refusals(tmp_path):
    check(tmp_path, """
    char* p = scratchAcquire(b, 100, false, false, m);
    m.room = 64 * MB;
    say(!scratchAcquire(b, 60 * MB, false, true, m) && b.ptr == p);
    say(scratchAcquire(b, 50 * MB, false, false, m) && m.frees == 1);
    m.room = 80 * MB;
    say(scratchAcquire(b, 60 * MB, false, false, m) && b.refused == 0);
    say(!scratchAcquire(b, 90 * MB, false, false, m) && !b.ptr && m.frees == 3);
    """)


def test_optional_growth_beside_a_captured_block(tmp_path):
    check(tmp_path, """
    char* p = scratchAcquire(b, 100, false, false, m);
    say(scratchAcquire(b, 100, true, false, m) == p && b.captured);
    m.room = MB;
    say(!scratchAcquire(b, 4 * MB, false, true, m) && b.ptr == p && b.captured);
    m.room = ~size_t(0);
    say(scratchAcquire(b, 3 * MB, false, true, m) != p && m.frees == 0 && !b.captured);
    """)
