"""The strip kernel's layout (csrc/hipclaw_strip_shape.h), compiled as host code:
every column of every patch lies in exactly one strip, strips of a wave do not
share lanes, and the strips' rows cover the patch."""
import json
import os
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "forestclaw_amd", "csrc")
MAIN = r"""
#include <cstdio>
#include "hipclaw_strip_shape.h"
using namespace hipclaw;
int main() {
    for (int mx = 8; mx <= 640; mx++)
        for (int whole = 0; whole < 2; whole++) {
            StripShape s;
            const bool ok = strip_pattern(mx, whole, s);
            std::printf("[%d, %d, %d, %d, %d, [", mx, whole, ok, ok ? s.waves : 0, ok ? s.patches : 0);
            for (int w = 0; ok && w < s.waves && w < StripShape::WAVES; w++)
                for (int k = 0; k < StripShape::SEGS; k++)
                    std::printf("%s%u", w + k ? ", " : "", s.seg[w][k]);
            std::printf("], [");
            const int n[4] = {1, 37, 800, 20000};
            for (int i = 0; ok && i < 4; i++)
                for (int my = 8; my <= 64; my += 7) {
                    strip_rows(my, n[i], 1024, my % 2, whole, s);
                    std::printf("%s[%d, %d, %d]", i + my > 8 ? ", " : "", my, s.H, s.nsy);
                }
            std::printf("]]\n");
        }
}
"""


@pytest.fixture(scope="module")
def layouts(tmp_path_factory):
    d = tmp_path_factory.mktemp("strips")
    (d / "main.cpp").write_text(MAIN)
    subprocess.run(["g++", "-std=c++17", "-I", CSRC, str(d / "main.cpp"), "-o", str(d / "main")], check=True)
    out = subprocess.run([str(d / "main")], check=True, capture_output=True, text=True).stdout
    return [json.loads(line) for line in out.splitlines()]


def test_every_column_once(layouts):
    assert len(layouts) == 2 * 633
    for mx, whole, ok, waves, patches, seg, _ in layouts:
        if not ok:
            assert whole and mx > 60
            continue
        if waves > 8:                      # listed by width alone
            assert not whole and patches == 1 and 60 * (waves - 1) < mx <= 60 * waves
            continue
        seen = set()
        for w in range(waves):
            free = 0
            assert seg[6 * w] != 0         # the first strip says which patch a wave begins with
            for k in range(6):
                s = seg[6 * w + k]
                if s == 0:
                    continue
                lane, n, patch, col = s & 63, (s >> 6) & 63, (s >> 12) & 15, s >> 16
                assert lane >= free and n >= 1 and lane + n + 4 <= 64 and patch < patches
                free = lane + n + 4
                if whole:
                    assert n == mx
                for c in range(col, col + n):
                    assert (patch, c) not in seen
                    seen.add((patch, c))
        assert seen == {(p, c) for p in range(patches) for c in range(mx)}, (mx, whole)
        # no worse than strips of one patch's equal parts
        parts = -(-mx // 60)
        if not whole:
            assert patches / waves >= 1.0 / parts - 1e-12, mx


def test_rows_cover_the_patch(layouts):
    for mx, whole, ok, _, _, _, rows in layouts:
        for my, h, nsy in rows:
            assert 1 <= h <= my and h * nsy >= my and h * (nsy - 1) < my
            if whole:
                assert nsy == 1
