"""Decode attention: where its workgroups do their work (cogstream_amd/csrc/mla_place.h), counted on the host."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
PROGRAM = r"""
#include <cstdio>
#include <cstdlib>
#include <map>
#include <tuple>
#include "mla_place.h"
// arguments: tiles of 32 keys a split, head tiles, groups, contexts; prints the workgroups with work of every engine, or why not
int main(int argc, char** argv) {
    const int tiles = atoi(argv[1]), nht = atoi(argv[2]), groups = atoi(argv[3]), n = argc - 4;
    int longest = 0;
    for (int b = 0; b < n; ++b) { const int t = (atoi(argv[4 + b]) + 31) / 32; if (t > longest) longest = t; }
    const int grid_x = ((longest + tiles - 1) / tiles + 7) / 8 * 8 * nht;
    long engine[8][4] = {}, in_front = 0;
    for (int b = 0; b < n; ++b) {
        const int ctx = atoi(argv[4 + b]), parts = ((ctx - 1) / 32 + tiles) / tiles;
        const long first = in_front / (32 * tiles) + b;
        in_front += ctx;
        for (int y = b * groups; y < (b + 1) * groups; ++y) {
            std::map<std::pair<int, int>, int> xcd;
            for (int x = 0; x < grid_x; ++x) {
                const MlaPlace p = mla_place(x, y, grid_x, nht, first);
                if (p.split < 0 || p.head_tile < 0 || p.head_tile >= nht) return puts("out of range"), 1;
                if (!xcd.emplace(std::make_pair(p.split, p.head_tile), x & 7).second) return puts("taken twice"), 1;
                if (p.split < parts) ++engine[x & 7][((long)y * grid_x + x) / 8 % 4];
            }
            for (int s = 0; s < parts; ++s)
                for (int h = 0; h < nht; ++h) {
                    const auto i = xcd.find({s, h});
                    if (i == xcd.end()) return puts("not taken"), 1;
                    if (i->second != xcd[{s, 0}]) return puts("head tiles of a split on two XCDs"), 1;
                }
        }
    }
    for (auto& x : engine) for (long e : x) printf("%ld ", e);
    return 0;
}
"""


@pytest.fixture(scope="module")
def program(tmp_path_factory):
    if shutil.which("g++") is None:
        pytest.skip("no g++")
    d = tmp_path_factory.mktemp("place")
    (d / "place.cpp").write_text(PROGRAM)
    subprocess.run(["g++", "-std=c++17", "-O1", "-I", os.path.join(ROOT, "cogstream_amd", "csrc"), str(d / "place.cpp"), "-o", str(d / "place")], check=True)
    return str(d / "place")


@pytest.mark.parametrize("tiles,head_tiles,groups,contexts", [
    (9, 1, 1, [256 * (i + 1) for i in range(32)]),          # four places a block and XCD
    (12, 1, 1, [256 * (i + 1) for i in range(32)]),         # three
    (17, 1, 1, [256 * (i + 1) for i in range(32)]),         # two
    (3, 1, 1, [256 * (i + 1) for i in range(16)]),
    (3, 2, 1, [256 * (i + 1) for i in range(16)]),
    (2, 1, 32, [64 * (i + 1) for i in range(32)]),          # one place, many blocks: few splits, not always of the first XCDs
    (2, 1, 4, [300] * 64),
    (4, 8, 1, [2000] * 8),
    (4, 1, 1, [50] * 20 + [8000] * 4),
    (5, 1, 4, [128 * (i + 1) for i in range(24)]),
    (3, 2, 3, [700] * 7),
    (2, 4, 1, [1, 100, 4000]),
    (2, 1, 1, [16000]),
    (1, 1, 1, [1]),
])
def test_decode_workgroups_reach_every_engine(program, tiles, head_tiles, groups, contexts):
    """every (split, head tile) of a block once, head tiles of a split on one XCD; no shader engine has more than a quarter above its share of
    the workgroups with work, and three for what does not come out even (each of the two moves, and the rounding)"""
    r = subprocess.run([program, *map(str, (tiles, head_tiles, groups, *contexts))], capture_output=True, text=True)
    assert r.returncode == 0, r.stdout
    engines = [int(v) for v in r.stdout.split()]
    assert len(engines) == 32 and max(engines) <= 1.25 * sum(engines) / 32 + 3, engines
