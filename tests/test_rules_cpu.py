"""The rules of openvdb_amd/csrc/nvq_rules.h (launch shapes, indices), compiled for the host and run at the
ends of the ranges that the entry points admit."""
import os
import subprocess

import numpy as np
import pytest

from conftest import ROOT

CSRC = os.path.join(ROOT, "openvdb_amd", "csrc")


def run_cpp(tmp_path, body, headers=("nvq_rules.h",)):
    """Compiles `body` as main() and returns what it printed, line by line."""
    src, exe = tmp_path / "t.cpp", tmp_path / "t"
    src.write_text("".join(f'#include "{h}"\n' for h in headers) + "#include <cstdio>\n#include <vector>\n"
                   "using namespace nvq;\nint main() {\n" + body + "\nreturn 0; }\n")
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-Wextra", "-Werror", "-I", CSRC, str(src), "-o", str(exe)],
                   check=True)
    return subprocess.run([str(exe)], check=True, capture_output=True, text=True, timeout=60).stdout.split("\n")[:-1]


@pytest.mark.parametrize("tiles", [1, 63, 64, 65, 262144, (1 << 28) - 1, 1 << 28, (1 << 28) + 1, 1 << 30,
                                   (1 << 30) + 77, (1 << 31) - 1])
def test_every_tile_has_one_quad(tmp_path, tiles):
    """Last and first tile of each row of the launch, and every row's threads below 2^32."""
    out = run_cpp(tmp_path, f"""
    const LaunchRows r = quadRows({tiles}u, 256u);
    std::printf("%u %u\\n", r.x, r.y);
    for (uint32_t y = 0; y < r.y; ++y)
        std::printf("%llu %llu %llu\\n", (unsigned long long)tileOfQuad(0, y, 0, 256u),
                    (unsigned long long)tileOfQuad(0, y, 3, 256u),
                    (unsigned long long)tileOfQuad(r.x - 1, y, 255, 256u));""")
    x, rows = map(int, out[0].split())
    assert x * 256 < 1 << 32 and rows < 65536
    expect = 0
    for line in out[1:]:
        first, same, last = map(int, line.split())
        assert first == same == expect
        assert last == first + 64 * x - 1
        expect = last + 1
    assert expect - 64 * x < tiles <= expect and expect - tiles < max(64 * x if rows > 1 else 64, 64)


BOXES = [(1, 1, 1), (4, 4, 4), (67, 67, 67), (203, 203, 203), (204, 204, 204), (255, 255, 255), (1, 1, 1 << 23),
         (1 << 23, 1, 1), (1, 1 << 23, 1), (4096, 64, 32), (4097, 64, 32), (3, 5, 7), (32, 33, 31), (256, 256, 256)]


@pytest.mark.parametrize("n", BOXES)
def test_block_tags_are_distinct_and_positions_fit(tmp_path, n):
    """blockBoxOf says before anything is built whether the adjoint's block cache can serve a box."""
    out = run_cpp(tmp_path, f"""
    SlotBox b{{}};
    const uint32_t n[3] = {{{n[0]}u, {n[1]}u, {n[2]}u}};
    b.count = 1;
    for (int a = 0; a < 3; ++a) {{ b.n[a] = n[a]; b.count *= n[a]; }}
    BlockBox x{{}};
    const bool ok = blockBoxOf(b, x);
    std::printf("%d %u %u\\n", ok ? 1 : 0, x.sx, x.sy);""")
    ok, sx, sy = map(int, out[0].split())
    slots = n[0] * n[1] * n[2]
    assert not ok or slots <= 1 << 23
    if ok:
        assert sy >= 4 * n[2] and sx >= 4 * n[1] * sy     # distinct tags
        assert (4 * n[0] - 1) * sx + (4 * n[1] - 1) * sy + 4 * n[2] - 1 < (1 << 32) - 2
        assert ((slots - 1) * 64 + 63) * 8 + 7 < 1 << 32  # positions
        assert sy % 128 == 19 and sx % 128 == 45
    else:
        assert slots > 1 << 22 or max(n) > 4096  # only large or very long boxes are turned away


@pytest.mark.parametrize("bbox,n", [((0, 0, 0, 0, 0, 0), (4, 4, 4)), ((-1, 0, 7, 8, 7, 8), (6, 4, 5)),
                                    ((5, 0, 0, 4, 9, 9), None), ((-(1 << 30), 0, 0, -(1 << 30) + 7, 7, 7), (4, 4, 4)),
                                    ((-(1 << 30) - 1, 0, 0, 0, 7, 7), None), ((0, 0, 0, (1 << 30) + 1, 7, 7), None),
                                    ((0, 0, 0, 2015, 2015, 2015), (255, 255, 255)),
                                    ((0, 0, 0, 2023, 2023, 2023), (256, 256, 256)),
                                    ((0, 0, 0, 2031, 2023, 2023), None)])
def test_slot_box(tmp_path, bbox, n):
    out = run_cpp(tmp_path, f"""
    const int32_t bbox[6] = {{{", ".join(map(str, bbox))}}};
    const SlotBox b = slotBoxOf(bbox);
    std::printf("%llu %u %u %u %d %d %d\\n", (unsigned long long)b.count, b.n[0], b.n[1], b.n[2], b.lo[0], b.lo[1], b.lo[2]);""")
    count, *rest = map(int, out[0].split())
    if n is None:
        assert count == 0
    else:
        assert tuple(rest[:3]) == n and count == n[0] * n[1] * n[2]
        assert [8 * x for x in rest[3:]] == [(x & ~7) - 8 for x in bbox[:3]]


def test_fd6_samples_below_2_23_stay_near_their_block():
    """fd6Near: for |p| < 2^23, floor(p + 1) and floor(p - 1) in FP32 are the next cells or one further up, so
    that the samples' corners lie in [cell-1, cell+3]; and those slots are the ones the block itself overlaps."""
    whole = np.unique(np.concatenate([np.arange(0, 4200), 2 ** np.arange(0, 24), 2 ** np.arange(1, 24) - 1,
                                      2 ** np.arange(0, 23) + 1, np.random.default_rng(0).integers(0, 1 << 23, 20000)]))
    at = np.concatenate([whole, -whole]).astype(np.float32)
    bits = at.view(np.int32)[:, None] + np.arange(-40, 41, dtype=np.int32)
    p = np.concatenate([bits.view(np.float32).reshape(-1), np.float32(2.0) ** -np.arange(1, 140, dtype=np.float32),
                        -(np.float32(2.0) ** -np.arange(1, 140, dtype=np.float32))]).astype(np.float32)
    p = p[np.isfinite(p) & (np.abs(p) < 8388608.0)]
    cell = np.floor(p).astype(np.int64)
    up, down = (np.floor(p + np.float32(d)).astype(np.int64) - cell for d in (1, -1))
    assert set(np.unique(up)) == {1, 2} and set(np.unique(down)) == {-1, 0}
    off = (up == 2) | (down == 0)
    assert off.sum() > 100
    first, last, far = (cell - 1) >> 3, (cell + 2) >> 3, (cell + up + 1) >> 3
    assert np.all((far == first) | (far == last))


# (slots, leaves, bytes per leaf, FpN), rays, whether the crossing was measured faster with the map
LEVEL_SETS = {"sphere30": (1728, 345, 2144, 0), "sphere100": (24389, 4025, 2144, 0), "torus300": (235224, 30249, 2144, 0),
              "torus300fp16": (235224, 30249, 1120, 0), "torus300fpn": (235224, 30249, 0, 1),
              "sphere400": (1124864, 64800, 2144, 0), "sphere800": (8489664, 259616, 2144, 0)}


@pytest.mark.parametrize("name,rays,pays", [
    ("sphere30", 1, 0), ("sphere30", 8, 0), ("sphere30", 64, 1), ("sphere30", 1000, 1), ("sphere30", 1 << 20, 1),
    ("sphere100", 4, 0), ("sphere100", 16, 0), ("sphere100", 64, 1), ("sphere100", 16384, 1),
    ("torus300", 1, 0), ("torus300", 16, 0), ("torus300", 64, 0), ("torus300", 256, 1), ("torus300", 1 << 18, 1),
    ("torus300fp16", 1000, 1), ("torus300fpn", 64, 0), ("torus300fpn", 128, 0), ("torus300fpn", 1 << 20, 1),
    ("sphere400", 64, 0), ("sphere400", 1000, 1), ("sphere400", 1 << 18, 1),
    ("sphere800", 16384, 0), ("sphere800", 65536, 0), ("sphere800", 1 << 18, 1), ("sphere800", 1 << 20, 1)])
def test_crossing_maps_are_built_where_they_were_faster(tmp_path, name, rays, pays):
    slots, leaves, size, fpn = LEVEL_SETS[name]
    out = run_cpp(tmp_path, f'std::printf("%d\\n", crossingMapPays({slots}u, {leaves}u, {size}u, {"true" if fpn else "false"}, {rays}u));')
    assert int(out[0]) == pays


@pytest.mark.parametrize("wanted,built", [([3, 4, 1], [3, 4, 1]), ([9], [0]), ([8], [8]), ([5, 4, 3, 1], [5, 0, 3, 0]),
                                          ([0, 0, 8, 1], [0, 0, 8, 0])])
def test_maps_of_a_call_are_bounded(tmp_path, wanted, built):
    """In GiB, against the 8 that one call may take."""
    sizes = ", ".join(f"size_t({w}) << 30" for w in wanted)
    out = run_cpp(tmp_path, f"""
    size_t b[] = {{{sizes}}};
    boundMaps(b, {len(wanted)}u);
    for (size_t x : b) std::printf("%zu\\n", x >> 30);
    // the largest map of a march and of an adjoint fit, with a slot table of 2^24
    std::printf("%d\\n", 1400000ull * (2944 + 8) + (12ull << 24) + 4096 <= kMaxMapBytes &&
                         (1ull << 20) * (2944 + 8 + 4096) + (12ull << 23) + 4096 <= kMaxMapBytes ? 1 : 0);""")
    assert [int(x) for x in out] == built + [1]
