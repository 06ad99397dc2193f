"""The regions of the layer launch's exchange buffer (nanollama_amd/csrc/nl_layers_map.h), compiled by itself: a line of 128 bytes belongs to one region and to
one XCD's copy, and no region reaches into the next."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
# q|k|v tiles, heads, records a head, tiles of WO, tiles of gate
SHAPES = [(108, 9, 16, 36, 92), (16, 2, 2, 8, 12), (144, 24, 16, 96, 256), (192, 32, 16, 128, 256), (44, 11, 3, 44, 17), (12, 3, 1, 12, 1)]


@pytest.fixture(scope="module")
def maps(tmp_path_factory):
    d = tmp_path_factory.mktemp("map")
    calls = "".join("p(nl::layers_map(%d, %d, %d, %d, %d));" % s for s in SHAPES)
    (d / "m.cpp").write_text('#include <cstdio>\n#include "nl_layers_map.h"\nvoid p(nl::LayersMap m) { std::printf("%d %d %d %d %d %d %d %d %d %d\\n", '
                             "m.gq, m.gr, m.go, m.gp, m.gh, m.gx, m.loc, m.loc_n, m.tickets, m.total); }\nint main() { " + calls + " }\n")
    subprocess.check_call(["g++", "-std=c++17", "-Wall", "-Werror", "-I", os.path.join(ROOT, "nanollama_amd", "csrc"), str(d / "m.cpp"), "-o", str(d / "m")])
    return [[int(w) for w in line.split()] for line in subprocess.check_output([str(d / "m")], text=True).splitlines()]


@pytest.mark.parametrize("i", range(len(SHAPES)))
def test_regions(maps, i):
    t_qkv, heads, rec, t_d, t_i = SHAPES[i]
    gq, gr, go, gp, gh, gx, loc, loc_n, tickets, total = maps[i]
    sizes = [t_qkv * 6, heads * rec * 22, heads * 22, t_d * 6, t_i * 6, t_d * 6, 8 * loc_n, 8 * 8]
    starts = [gq, gr, go, gp, gh, gx, loc, tickets]
    assert all(s % 8 == 0 for s in starts + [loc_n])
    assert starts[0] == 0 and all(a + n <= b for a, n, b in zip(starts, sizes, starts[1:] + [total]))
    assert loc_n >= 12 * t_d + 6 * t_i
