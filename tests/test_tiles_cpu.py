"""Which tiles of a persistent GEMM go out as quarters (csrc/pq_tiles.h, compiled here with the host compiler), against the
same rule stated in Python, which the GPU tests use to say what their shapes reach."""
import os
import subprocess

import pytest

from dispatch_rules import whole_tiles

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "pyraquant_amd", "csrc")


@pytest.fixture(scope="module")
def rule(tmp_path_factory):
    d = tmp_path_factory.mktemp("tiles")
    src, exe = str(d / "rule.cpp"), str(d / "rule")
    with open(src, "w") as f:
        f.write('#include "pq_tiles.h"\n#include <cstdio>\nint main() { int t, w, k; while (scanf("%d %d %d", &t, &w, &k) == 3) {'
                ' const pq::WholeTiles r = pq::whole_tiles(t, w, k); printf("%d %d\\n", r.lo, r.hi); } }\n')
    subprocess.run(["g++", "-std=c++17", "-O1", "-I", CSRC, src, "-o", exe], check=True)

    def run(cases):
        text = "".join("%d %d %d\n" % c for c in cases)
        out = subprocess.run([exe], input=text, capture_output=True, text=True, check=True).stdout.split("\n")
        return [tuple(map(int, l.split())) for l in out if l]

    return run


def test_whole_tiles(rule):
    cases = [(t, w, K) for w in (32, 4) for t in range(8 * w + 1, 8 * w * 11) for K in (64, 640, 1984, 2048, 4032, 4096, 15360)]
    for (t, w, K), (lo, hi) in zip(cases, rule(cases)):
        lengths, whole = whole_tiles(t, K, w)
        assert lo == whole[0] and (t % 8 == 0 or hi == whole[1]), (t, w, K, lo, hi)
        for n, m in zip(lengths, (lo, hi if t % 8 else lo)):
            assert w <= m <= n and 4 * (n - m) <= w, (t, w, K, lo, hi)   # a whole tile each first; one wave of quarters


def test_quarters_only_where_they_gain(rule):
    """Products that were slower with quarters stay whole (256 CUs; times alone, whole against quarters): 8 tiles past the
    round at short K (29440 x 640 x 1280 72.7 against 82.9 us), lists with quarters beside lists without (95129 x 2752 x 1152
    418 and 439, 11296 x 3392 x 11904 402 and 433), many rounds (26406 x 1280 x 5120 200 and 208); those that gain keep them."""
    whole = [(29440, 640, 1280), (9216, 1280, 3968), (95129, 2752, 1152), (11296, 3392, 11904), (26406, 1280, 5120),
             (17152, 1280, 5120), (10496, 640, 5120)]
    quartered = [(4352, 3072, 12288), (16640, 3072, 3072), (16640, 12288, 3072), (6656, 640, 5120), (13120, 1280, 5120),
                 (52736, 5120, 1280), (9948, 1280, 5120)]
    tiles = {s: -(-s[0] // 256) * -(-s[2] // 256) for s in whole + quartered}
    for shape, (lo, hi) in zip(tiles, rule([(t, 32, s[1]) for s, t in tiles.items()])):
        t = tiles[shape]
        some = lo < t // 8 or (t % 8 and hi < t // 8 + 1)
        assert bool(some) == (shape in quartered), (shape, t, lo, hi)
