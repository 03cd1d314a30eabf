"""The rules of openvdb_amd/csrc/nvq_rules.h (launch shapes, indices), compiled for the host and run at the
ends of the ranges that the entry points admit."""
import os
import subprocess

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
