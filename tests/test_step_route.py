"""Which launches the tile kernel takes (csrc/hipclaw_strip_shape.h: tiles_pay),
compiled as host code: small launches and small ones in place, and none once the
strips' waves fill the chip; more patches never send a launch back to the tiles."""
import json
import os
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "forestclaw_amd", "csrc")
SIMDS = 1024
MAIN = r"""
#include <cstdio>
#include "hipclaw_strip_shape.h"
int main() {
    const int waves[6] = {1 * 4, 1 * 8, 9 * 4, 9 * 8, 16 * 4, 16 * 8};
    for (int tile = 8; tile <= 32; tile *= 2)
        for (int w = 0; w < 6; w++)
            for (int mx = tile; mx <= 200; mx += 7)
                for (int regs = 0; regs < 3; regs++)
                    for (int here = 0; here < (mx == tile ? 2 : 1); here++) {
                        const int across = (mx + tile - 1) / tile;
                        std::printf("[%d, %d, %d, %d, %d, %d, [", tile, waves[w], mx, regs, here, across * across);
                        for (int n = 1; n <= (1 << 20); n *= 2)
                            std::printf("%s%d", n > 1 ? ", " : "",
                                        (int) hipclaw::tiles_pay(waves[w], tile, mx, mx, n, across * across, SIMDS, regs, here));
                        std::printf("]]\n");
                    }
}
""".replace("SIMDS", str(SIMDS))


@pytest.fixture(scope="module")
def routes(tmp_path_factory):
    d = tmp_path_factory.mktemp("routes")
    (d / "main.cpp").write_text(MAIN)
    subprocess.run(["g++", "-std=c++17", "-I", CSRC, str(d / "main.cpp"), "-o", str(d / "main")], check=True)
    out = subprocess.run([str(d / "main")], check=True, capture_output=True, text=True).stdout
    return [json.loads(line) for line in out.splitlines()]


def test_one_switch_from_tiles_to_strips(routes):
    for *_, tiles in routes:
        assert tiles == sorted(tiles, reverse=True)
        assert not tiles[-1]


def test_in_place_steps_of_few_patches_take_tiles(routes):
    """One wave per patch would march its rows alone."""
    seen = 0
    for tile, wave_bytes, mx, regs, here, per, tiles in routes:
        if here:
            seen += 1
            assert all(tiles[:9])            # up to 256 patches, a quarter of the SIMDs
    assert seen == 54


def test_small_launches_take_tiles(routes):
    """8 x 8 tiles: one per CU for any solver, four for shallow water FP32-bulk, eight
    for FP64 (four with time-sync registers, two where they add up); 16 x 16 tiles two
    per CU (one), only where an interface has 72 bytes of waves; 32 x 32 tiles in
    place only.  Tiles that overlap count by the cells they compute."""
    cus = SIMDS // 4
    for tile, wave_bytes, mx, regs, here, per, tiles in routes:
        if here:
            continue
        heavy = wave_bytes >= 72
        limit = {8: (((8, 4, 2) if heavy else (max(1, wave_bytes / 9), 1, 1))[regs]) * cus,
                 16: (2, 2, 1)[regs] * cus if heavy else 0, 32: 0}[tile]
        load = per * per * tile * tile / (mx * mx)
        assert [bool(t) for t in tiles] == [2 ** k * load <= limit for k in range(len(tiles))], (tile, wave_bytes, mx, regs)
