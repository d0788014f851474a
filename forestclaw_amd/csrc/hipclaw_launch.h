// Launch dispatch of the step kernel for one Riemann functor: the strip kernel
// (step_strips), or for small launches and for solvers with more wave components
// than a lane can keep the LDS tile kernel (step_tiles); time-sync registers and the
// compile-time method pick the instantiation.  Shared by the built-in solvers' two
// translation units (FP64 compiled without FMA contraction, FP32-bulk with it)
// and by solvers an application compiles itself (hipclaw_user_solver.h); the
// instantiations take the contraction mode of the unit that includes this.
#pragma once

#include <atomic>
#include <type_traits>

#include <hip/hip_ext.h>
#include <hip/hip_runtime.h>

#include "hipclaw_strips.h"

namespace hipclaw {

// The stream of a step launch and, for a timed launch, two events that
// hipExtLaunchKernelGGL binds to the kernel's own start and end, so their
// elapsed time is the kernel's execution without the gaps around it.
struct StepLaunch {
    hipStream_t st;
    hipEvent_t start, stop;
    StepLaunch(hipStream_t s, hipEvent_t a = nullptr, hipEvent_t b = nullptr) : st(s), start(a), stop(b) {}
};

// Workgroups of `kernel` (block size `block`, static LDS only) that the
// current device holds at once: the grid of a persistent launch.
inline int resident_blocks(const void* kernel, int block) {
    int dev = 0, cus = 0, per_cu = 0;
    if (hipGetDevice(&dev) != hipSuccess) return 0;
    if (hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess) return 0;
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, kernel, block, 0) != hipSuccess) return 0;
    return per_cu * cus;
}

// Launch a persistent step kernel: min(tiles, resident workgroups) of them.
// `resident` caches the occupancy query; each kernel instantiation owns one.
// Host threads may race to fill it: they compute the same value, and the
// atomic makes the store and the loads well defined.
template <typename K>
inline int launch_persistent(K kernel, int block, const StepArgs& a, const StepLaunch& L,
                             std::atomic<int>& resident) {
    const int ntiles = a.nwork * a.ntx * a.nty;
    if (ntiles <= 0) return 0;
    int nres = resident.load(std::memory_order_relaxed);
    if (nres <= 0) {
        nres = resident_blocks((const void*) kernel, block);
        resident.store(nres, std::memory_order_relaxed);
    }
    if (nres <= 0) return (int) hipErrorInvalidDeviceFunction;
    const int nblocks = ntiles < nres ? ntiles : nres;
    if (L.start || L.stop)
        hipExtLaunchKernelGGL(kernel, dim3(nblocks), dim3(block), 0, L.st, L.start, L.stop, 0, a);
    else
        hipLaunchKernelGGL(kernel, dim3(nblocks), dim3(block), 0, L.st, a);
    return (int) hipGetLastError();
}

// Every wave family uses the MC limiter (mthlim 4), so the step may take the
// instantiation with the limiter fixed at compile time.
template <class RP>
inline bool all_mc_limiter(const StepArgs& a) {
    for (int mw = 0; mw < RP::MWAVES; mw++)
        if (a.mthlim[mw] != 4) return false;
    return true;
}

// Whether the functor provides the conservative flux the time-sync registers
// store (consflux<IXY>); without it a solver runs without time sync.
template <class RP, class = void>
struct has_consflux : std::false_type {};
template <class RP>
struct has_consflux<RP, std::void_t<decltype(&RP::template consflux<1>)>> : std::true_type {};

// A step instantiation fits the 160 KiB of LDS a workgroup may hold.
template <class RP, typename R, int T, bool FLUXFORM, bool REGS>
constexpr bool step_fits() {
    return sizeof(TileSmem<T, RP::MEQN, RP::MAUX, R, FLUXFORM, REGS>) + 64 <= 160 * 1024;
}

// One tile shape of one precision.  R = double: the FP64 parity form;
// R = float: the FP32-bulk form (flux form for a conservative solver).
// WITH_REGS = false leaves out the time-sync instantiations.
template <class RP, typename R, int T, int NW, bool WITH_REGS>
inline int launch_step_shape(const StepArgs& a, const StepLaunch& st) {
    // kernels that keep time-sync registers are separate instantiations, so the
    // plain update carries none of their code or register pressure; the MC
    // limiter on every wave family has its own compile-time instantiation
    constexpr bool FF = sizeof(R) == 4 && RP::CONSERVATIVE;
    static std::atomic<int> resident[2][2];   // zero-initialised (static storage)
    if constexpr (!step_fits<RP, R, T, FF, false>()) {
        return (int) hipErrorInvalidValue;
    } else {
        const bool mc = all_mc_limiter<RP>(a);
        if (a.reg) {
            if constexpr (WITH_REGS && step_fits<RP, R, T, FF, true>()) {
                if (mc)
                    return launch_persistent(step_tiles<RP, R, T, NW, FF, true, 4>, NW * 64, a, st, resident[1][1]);
                return launch_persistent(step_tiles<RP, R, T, NW, FF, true>, NW * 64, a, st, resident[0][1]);
            }
            return (int) hipErrorInvalidValue;
        }
        if (mc)
            return launch_persistent(step_tiles<RP, R, T, NW, FF, false, 4>, NW * 64, a, st, resident[1][0]);
        return launch_persistent(step_tiles<RP, R, T, NW, FF, false>, NW * 64, a, st, resident[0][0]);
    }
}

// Whether a launch of a solver that uses strips goes to the tile kernel all the same
// (tiles_pay).  Larger launches are faster in strips (tiles and strips, us: shallow
// water FP64 16 x 16, 2800 patches 82 / 63; 32 x 32, 6000 patches FP64 569 / 346,
// FP32-bulk 206 / 145; Euler FP64 856 / 502; advection FP64 140 / 69).
inline bool launches_tiles(const StepArgs& a, int tile, int wave_bytes, int simds) {
    const bool inplace = a.qsrc == a.qdst;
    if (inplace && a.ntx * a.nty != 1) return false;
    return tiles_pay(wave_bytes, tile, a.mx, a.my, a.nwork, a.ntx * a.nty, simds,
                     !a.reg ? TILES_PLAIN : a.reg_accumulate ? TILES_ACCUMULATE : TILES_REGISTERS, inplace);
}

inline int device_simds() {
    static std::atomic<int> simds{0};
    int n = simds.load(std::memory_order_relaxed);
    if (n <= 0) {
        int dev = 0, cus = 0;
        if (hipGetDevice(&dev) == hipSuccess &&
            hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) == hipSuccess)
            n = 4 * cus;
        simds.store(n, std::memory_order_relaxed);
    }
    return n;
}

// pairs: two waves of the kernel fit a SIMD.  lds: its bytes per wave.  nw: waves per
// workgroup.
template <typename K>
inline int launch_strips(K kernel, bool pairs, int lds, int nw, const StepArgs& a, const StepLaunch& L) {
    if (a.nwork <= 0) return 0;
    const bool inplace = a.qsrc == a.qdst;
    const int simds = device_simds();
    StripShape sh;
    if (simds <= 0 || !strip_pattern(a.mx, inplace, sh)) return (int) hipErrorInvalidValue;
    strip_rows(a.my, a.nwork, simds, pairs, inplace, sh);
    const long long waves = ((long long) a.nwork + sh.patches - 1) / sh.patches * sh.waves * sh.nsy;
    const long long blocks = ((waves + nw - 1) / nw + 7) / 8 * 8;   // a multiple of the 8 XCDs
    if (waves * 64 > 0x7fffffffLL) return (int) hipErrorInvalidConfiguration;
    if (L.start || L.stop)
        hipExtLaunchKernelGGL(kernel, dim3((unsigned) blocks), dim3(64 * nw), lds * nw, L.st, L.start, L.stop, 0, a, sh);
    else
        hipLaunchKernelGGL(kernel, dim3((unsigned) blocks), dim3(64 * nw), lds * nw, L.st, a, sh);
    return (int) hipGetLastError();
}

// The strip kernel of one precision: with and without time-sync registers
// (overwritten, or added to when subcycling), and with order (2, 2) and the MC
// limiter on every wave family fixed at compile time.
template <class RP, typename R, bool WITH_REGS>
inline int launch_step_strips(int nw, const StepArgs& a, const StepLaunch& st) {
    constexpr bool FF = sizeof(R) == 4 && RP::CONSERVATIVE, pairs = strip_waves_per_eu<RP, R>() > 1;
    constexpr int lds = strip_lds<RP, R>();
    const bool std = all_mc_limiter<RP>(a) && a.order2 && a.transverse == 2;
    if (a.reg) {
        if constexpr (WITH_REGS) {
            if (a.reg_accumulate)
                return std ? launch_strips(step_strips<RP, R, FF, 2, true>, pairs, lds, nw, a, st)
                           : launch_strips(step_strips<RP, R, FF, 2, false>, pairs, lds, nw, a, st);
            return std ? launch_strips(step_strips<RP, R, FF, 1, true>, pairs, lds, nw, a, st)
                       : launch_strips(step_strips<RP, R, FF, 1, false>, pairs, lds, nw, a, st);
        }
        return (int) hipErrorInvalidValue;
    }
    return std ? launch_strips(step_strips<RP, R, FF, 0, true>, pairs, lds, nw, a, st)
               : launch_strips(step_strips<RP, R, FF, 0, false>, pairs, lds, nw, a, st);
}

// Waves per workgroup by default.  Strips: four, which share nothing but lie on the
// four SIMDs of one CU, beside each other in its cache (one and four, subcycled dam
// break FP64 9.80 and 9.62 ms, dam break FP64 22.53 and 22.46, shock-bubble FP32
// 5.20 and 5.16, advection 567 and 565 us; three leave a SIMD of every CU idle).  Single
// waves may also come two to a SIMD beside an idle one when a launch meets an idle
// device: Euler FP64 on 134 patches of 61 x 61, 960 waves, 97 us alone and 71 among
// other steps with one wave, 68 and 71 with four.
// 16 x 16 tiles: four for FP64, two for the FP32-bulk form (a sweep's 18 rows, three
// per wave, are three groups for each of two waves, where four take two, two, one
// and one and wait at the barrier; FP64 tiles need the latency hiding of four).
// hipclaw_set_waves and the autotuner choose 2, 3 or 4.
constexpr int STRIP_WAVES = 4;
constexpr int default_tile_waves(bool fp64, int tile) { return tile != 16 ? 0 : fp64 ? 4 : 2; }   // (0: one choice)

// Whether the tile kernel is instantiated for a tile (T = 32 only WITH32).
template <class RP, typename R, bool WITH_REGS, bool WITH32>
constexpr bool has_tile(int tile, bool regs) {
    constexpr bool FF = sizeof(R) == 4 && RP::CONSERVATIVE;
    if (regs && !WITH_REGS) return false;
    return tile == 8    ? (regs ? step_fits<RP, R, 8, FF, true>() : step_fits<RP, R, 8, FF, false>())
           : tile == 16 ? (regs ? step_fits<RP, R, 16, FF, true>() : step_fits<RP, R, 16, FF, false>())
                        : WITH32 && tile == 32 &&
                              (regs ? step_fits<RP, R, 32, FF, true>() : step_fits<RP, R, 32, FF, false>());
}

// The small launches of a solver that uses strips have one shape per tile and
// precision: the choice of 2, 3 or 4 waves is the strips' (and each further kernel
// makes the code larger that every launch is fetched from: with all of them a call of
// two small kernels took 0.5 to 1 us more).
template <class RP, typename R, bool WITH_REGS, bool WITH32>
inline int launch_step_tiles(int tile, int waves, const StepArgs& a, const StepLaunch& st) {
    if (waves == 0) waves = default_tile_waves(sizeof(R) == 8, tile);
    switch (tile) {
    case 8: return launch_step_shape<RP, R, 8, 2, WITH_REGS>(a, st);
    case 16:
        if constexpr (uses_strips<RP>())
            return launch_step_shape<RP, R, 16, default_tile_waves(sizeof(R) == 8, 16), WITH_REGS>(a, st);
        else
            return waves == 2 ? launch_step_shape<RP, R, 16, 2, WITH_REGS>(a, st)
                 : waves == 3 ? launch_step_shape<RP, R, 16, 3, WITH_REGS>(a, st)
                              : launch_step_shape<RP, R, 16, 4, WITH_REGS>(a, st);
    case 32:
        if constexpr (WITH32) return launch_step_shape<RP, R, 32, 16, WITH_REGS>(a, st);
        return (int) hipErrorInvalidValue;
    default: return (int) hipErrorInvalidValue;
    }
}

// waves = 0: the default; 2, 3 or 4 select the variant (of the strips, which then take
// small launches too, unless in place).
template <class RP, typename R, bool WITH_REGS, bool WITH32 = false>
inline int launch_step_tile(int tile, int waves, const StepArgs& a, const StepLaunch& st) {
    if constexpr (uses_strips<RP>()) {
        if ((waves > 0 && a.qsrc != a.qdst) || !has_tile<RP, R, WITH_REGS, WITH32>(tile, a.reg != nullptr) ||
            !launches_tiles(a, tile, RP::MEQN * RP::MWAVES * (int) sizeof(R), device_simds()))
            return launch_step_strips<RP, R, WITH_REGS>(waves > 0 ? waves : STRIP_WAVES, a, st);
    }
    return launch_step_tiles<RP, R, WITH_REGS, WITH32>(tile, waves, a, st);
}

}  // namespace hipclaw
