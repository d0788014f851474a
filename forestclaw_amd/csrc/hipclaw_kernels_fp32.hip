// FP32-bulk patch step: Riemann solves, limiter and transverse splitting in
// FP32, conservative FP64 interface fluxes and FP64 q storage.  Compiled with
// FMA contraction allowed (this form is measured against the FP64 oracle with
// a stated error tolerance, not bit for bit).
#include "hipclaw_internal.h"

namespace hipclaw {

int launch_step_fp32(int solver, int tile, int waves, const StepArgs& a, const StepLaunch& st) {
    switch (solver) {
    case 0: return launch_step_tile<RPAdvection<float>, float, true, true>(tile, waves, a, st);
    case 1: return launch_step_tile<RPShallow<float>, float, true, true>(tile, waves, a, st);
    case 2: return launch_step_tile<RPEuler<float>, float, true>(tile, waves, a, st);
    default: return (int) hipErrorInvalidValue;
    }
}

bool step_supported(int solver, int precision, int tile) {
    if (tile != 8 && tile != 16 && tile != 32) return false;
    // 32 x 32: the shallow-water solver, and advection in the FP32-bulk form
    if (tile == 32) return precision == 0 ? solver == 1 : solver != 2;
    return solver >= 0 && solver <= 2;
}

}  // namespace hipclaw
