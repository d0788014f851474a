"""The rows of a strip (csrc/hipclaw_strip_shape.h: strip_rows), compiled as host
code: among all cuts of a patch none takes less by the rule's own measure, rounds of
waves over the SIMDs times row steps, when the waves are those the launch starts.
(The last pattern's waves are started whether its patches are there or not.)"""
import json
import os
import subprocess

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "forestclaw_amd", "csrc")
SIMDS = 1024
MAIN = r"""
#include <cstdio>
#include "hipclaw_strip_shape.h"
using namespace hipclaw;
int main() {
    const int mxs[] = {8, 9, 16, 20, 32, 33, 48, 61, 64, 100, 128, 500};
    for (int mx : mxs) {
        StripShape s;
        strip_pattern(mx, false, s);
        for (int my : {8, 17, 32, 61, 100})
            for (int n = 1; n < 40000; n += 1 + n / 7)
                for (int pairs = 0; pairs < 2; pairs++) {
                    strip_rows(my, n, SIMDS, pairs, false, s);
                    std::printf("[%d, %d, %d, %d, %d, %d, %d, %d]\n", mx, my, n, pairs, s.waves, s.patches, s.H, s.nsy);
                }
    }
}
""".replace("SIMDS", str(SIMDS))


def test_no_cut_is_shorter(tmp_path):
    (tmp_path / "main.cpp").write_text("#include <initializer_list>\n" + MAIN)
    subprocess.run(["g++", "-std=c++17", "-I", CSRC, str(tmp_path / "main.cpp"), "-o", str(tmp_path / "main")], check=True)
    out = subprocess.run([str(tmp_path / "main")], check=True, capture_output=True, text=True).stdout
    seen = 0
    for line in out.splitlines():
        mx, my, n, pairs, waves, patches, H, nsy = json.loads(line)

        def cost(cut):
            h = -(-my // cut)
            rounds = -(-(-(-n // patches) * waves * cut) // SIMDS)
            return rounds * (h + 3) * (1.2 if pairs and rounds == 1 else 1.0)

        cuts = [c for c in range(1, my + 1) if -(-my // -(-my // c)) == c]
        assert cost(nsy) <= min(map(cost, cuts)) * (1 + 1e-12), (mx, my, n, pairs, H, nsy)
        seen += 1
    assert seen > 5000
