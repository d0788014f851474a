// How a launch of the strip kernel (hipclaw_strips.h) lays the patches of its
// work list on waves of 64 lanes, and which launches the tile kernel takes instead.
// Host code, without HIP.
#pragma once

namespace hipclaw {

// `waves` waves hold `patches` patches side by side, and the pattern repeats;
// segment k of wave w of the pattern is a strip of one patch (strip_segment),
// 0 past the last segment.  A strip of w columns takes w + 4 lanes, its halo
// among them.  Patches of more columns than a pattern holds take `waves` waves
// of 60 columns each (the last one fewer), computed instead of listed.  In y a
// patch is cut into nsy strips of H rows, the last one moved back to end at the
// patch edge: it overlaps the one before it, and both write the same bits.
struct StripShape {
    static constexpr int WAVES = 8, SEGS = 6, LANES = 64, HALO = 4, PATCHES = 15;
    int H, nsy;
    int waves, patches;
    unsigned seg[WAVES][SEGS];
};

// first lane | columns << 6 | patch of the pattern << 12 | first column (0-based) << 16
constexpr unsigned strip_segment(int lane, int n, int patch, int col) {
    return (unsigned) lane | (unsigned) n << 6 | (unsigned) patch << 12 | (unsigned) col << 16;
}

// Packs patches of mx columns.  A patch that does not fit into what is left of
// a wave is cut and goes on in the next one (11 % more columns per wave at
// mx = 32, 37 % at mx = 40, than whole strips of equal width), unless `whole`:
// an update in place needs the patch in one wave, which then reads every cell
// before it writes it.  Of the patterns of at most WAVES waves, the one with the
// most columns per wave; false if `whole` patches have no room.
inline bool strip_pattern(int mx, bool whole, StripShape& sh) {
    constexpr int MOST = StripShape::LANES - StripShape::HALO;
    if (whole && mx > MOST) return false;
    StripShape t{};
    int col = 0, patch = 0;      // the next column to lay out
    double best = 0.0;
    sh = t;
    for (int w = 0; w < StripShape::WAVES; w++) {
        int lane = 0;
        for (int k = 0; k < StripShape::SEGS; k++) {
            const int room = MOST - lane, left = mx - col;
            if (room < 1 || (whole && left > room) || patch >= StripShape::PATCHES) break;
            const int n = left < room ? left : room;
            t.seg[w][k] = strip_segment(lane, n, patch, col);
            lane += n + StripShape::HALO;
            col += n;
            if (col == mx) { col = 0; patch++; }
        }
        // the pattern that ends with this wave, less the patch only begun
        const double cols = (double) patch * mx / (w + 1);
        if (patch > 0 && cols > best * 1.0001) {
            best = cols;
            sh = t;
            sh.waves = w + 1;
            sh.patches = patch;
            for (int v = 0; v <= w; v++)
                for (int k = 0; k < StripShape::SEGS; k++)
                    if ((int) ((sh.seg[v][k] >> 12) & 15) >= patch) sh.seg[v][k] = 0;
        }
    }
    if (best == 0.0) {           // wider than WAVES waves
        sh.waves = (mx + MOST - 1) / MOST;
        sh.patches = 1;
    }
    return true;
}

// Rows per strip.  One wave keeps a SIMD's issue slots nearly full, so a launch
// takes as long as the SIMD with the most waves: ceil(waves / SIMDs) strips of
// H + 3 row steps each (three rows lead in).  Alone on its SIMD a wave waits for
// its own results a sixth of the time, which a second one would use (`pairs`:
// the kernel's registers leave room for it).  Kernel times, us: shallow water
// FP64, 700 patches of 32 x 32 (420 waves of columns), H = 4, 8, 16, 32: 71, 62,
// 66, 110; 256 of 16 x 16 (86), H = 1, 2, 4, 8, 16: 23, 20, 25, 36, 59; Euler
// FP32-bulk, 2800 of 16 x 16 (934), H = 4, 8, 16: 50, 42, 45.  The waves of a last
// pattern with fewer patches are started all the same and count: 134 of 61 x 61, 153
// waves of columns in 20 patterns of 8, are three rounds at H = 5 (2,080 waves, 63 us)
// and one at H = 11 (49).
inline void strip_rows(int my, int nwork, int simds, bool pairs, bool whole, StripShape& sh) {
    const long long cols = ((long long) nwork + sh.patches - 1) / sh.patches * sh.waves;
    double best = 0.0;
    sh.nsy = 1;
    for (int nsy = 1; nsy <= (whole ? 1 : my); nsy++) {
        const int H = (my + nsy - 1) / nsy;
        if ((my + H - 1) / H != nsy) continue;   // (the same H as fewer strips)
        const long long rounds = (cols * nsy + simds - 1) / simds;
        const double cost = (double) rounds * (H + 3) * (pairs && rounds == 1 ? 1.2 : 1.0);
        if (nsy == 1 || cost < best) { best = cost; sh.nsy = nsy; }
    }
    sh.H = (my + sh.nsy - 1) / sh.nsy;
}

// Whether a launch takes less time on the tile kernel, whose waves share a tile's
// rows: a strip's wave, alone on its SIMD, issues one instruction per four cycles
// and leads in with five row steps, so strips win once their waves fill the SIMDs.
// Kernel times in us, tiles and strips:
//   T = 8   shallow water FP64 24 x 20 (9 tiles each), 16 patches 7.9 / 14.6, 133
//           15.7 / 18.4, 266 29.1 / 22.0; FP32-bulk 16 5.6 / 7.5, 66 8.1 / 8.2, 133
//           10.6 / 9.5; advection FP64 16 4.5 / 5.8, 66 6.6 / 6.1
//   T = 16  shallow water FP64 16 x 16, 15 patches 12.4 / 14.6, 500 18.4 / 22.1, 1000
//           39.7 / 32.2; Euler FP64 250 16.8 / 24.5, 1000 43.3 / 44.2; lighter solvers
//           and the FP32-bulk form 0.7 to 1.0 times as long with strips
//   T = 32  shallow water FP64 32 x 32, 1 patch 29.5 / 14.6, 700 85 / 62
// and with time-sync registers, which the tiles store at the end of a tile,
//   T = 8   shallow water FP64 24 x 24, strips 1.24 times as long with 88 patches and
//           0.8 with 333; FP32-bulk 1.07 with 28, 0.91 with 44
// and where these add up over substeps, which the strips leave to the L2 (one level's
// copy, step, ghost fill and synchronisation),
//   T = 8   shallow water FP64 12 x 12, 100 patches 23.7 / 25.6, 256 27.7 / 26.5
//   T = 16  16 x 16, 256 patches 28.1 / 30.8, 288 32.7 / 31.4
// Tiles that overlap (a patch the tile does not divide) compute cells twice, and
// count as much more.
// In place a patch is one strip of all its rows, a serial chain: tiles until the
// strips' waves fill three quarters of the SIMDs (half of them for a solver of few
// wave components).  Shallow water FP64 8 x 8, 1 patch 6.6 / 30.7, 2000 17.1 / 32.9,
// 4000 29.1 / 33.9, 8000 52.8 / 51.7; 16 x 16, 1 patch 11.6 / 52.6, 2000 53.6 / 56.8,
// 3000 76 / 64; 32 x 32 (T = 32) 28.5 / 96, 700 80 / 101; advection FP64 8 x 8, 1000
// 6.9 / 9.4, 2000 9.9 / 9.7.
// wave_bytes: of one interface's waves (meqn x mwaves values).
enum { TILES_PLAIN = 0, TILES_REGISTERS = 1, TILES_ACCUMULATE = 2 };
inline bool tiles_pay(int wave_bytes, int tile, int mx, int my, int nwork, int tiles_per_patch, int simds, int regs,
                      bool inplace) {
    const long long cus = simds / 4;
    if (inplace) {
        const int across = StripShape::LANES / (mx + StripShape::HALO);
        const int per_wave = across < 1 ? 1 : across < StripShape::SEGS ? across : StripShape::SEGS;
        return 4LL * nwork <= (wave_bytes >= 24 ? 3LL : 2LL) * simds * per_wave;
    }
    const bool heavy = wave_bytes >= 72;
    double most;                 // tiles per CU
    if (tile == 8) most = regs ? (!heavy ? 1 : regs == TILES_ACCUMULATE ? 2 : 4) : heavy ? 8 : wave_bytes < 9 ? 1 : wave_bytes / 9.0;
    else most = tile == 16 && heavy ? (regs == TILES_ACCUMULATE ? 1 : 2) : 0;
    const double ntiles = (double) nwork * tiles_per_patch, twice = (double) tiles_per_patch * tile * tile / ((double) mx * my);
    return ntiles * twice <= most * cus;
}

}  // namespace hipclaw
