// Device Riemann solvers for the batched patch update.
//
// Each solver works on ONE interface held in registers: qL is the cell to the
// left of the interface (the reference's qr(i-1,:)), qR the cell to the right
// (ql(i,:)).  IXY = 1 for an x-interface, 2 for a y-interface.  The arithmetic
// is written in the same order as the reference Fortran so that, compiled
// with FMA contraction off, the FP64 instantiation reproduces it bit for bit:
//
//   shallow water : applications/clawpack/shallow/2d/rp/clawpack46_rpn2.f:91-242,
//                   clawpack46_rpt2.f:287-319 (Roe, entropy fix on)
//   Euler         : applications/clawpack/euler/2d/rp/clawpack46_rpn2_euler4.f:83-285,
//                   clawpack46_rpt2_euler4.f:345-383 (Roe, entropy fix on)
//   advection     : applications/clawpack/advection/2d/all/clawpack46_rpn2adv.f:28-58,
//                   clawpack46_rpt2adv.f:79-86
//
// Solvers are compile-time functors (no device function pointers) so the
// compiler can keep waves, speeds and fluctuations in VGPRs.
#pragma once

#include <type_traits>

#include <hip/hip_runtime.h>

namespace hipclaw {

struct PhysParams {
    double grav;   // shallow water gravity
    double gamma;  // Euler ratio of specific heats
    // A registered solver's own constants (what the reference keeps in a
    // solver's common block or __constant__ memory, e.g. rho, bulk, cc, zz of
    // the acoustics solver's common /cparam/).
    double p[8];
};

// c ? a : b.  A 64-bit select is two 32-bit ones, and the short encoding of
// v_cndmask, whose mask is VCC, takes 9.6 ns when another one comes right before
// it (2.2 ns otherwise; two waves per SIMD): a compare and two of them 16 to 20
// ns, with the long encoding, whose mask is any scalar pair, 6.5 ns.  The wait
// states are those a vector instruction needs before it reads a mask that one
// wrote.
__device__ __forceinline__ double pick(bool c, double a, double b) {
    const unsigned long long m = __builtin_amdgcn_ballot_w64(c);
    int lo, hi;
    asm("s_nop 1\n\tv_cndmask_b32_e64 %0, %2, %3, %6\n\tv_cndmask_b32_e64 %1, %4, %5, %6"
        : "=&v"(lo), "=v"(hi)
        : "v"(__double2loint(b)), "v"(__double2loint(a)), "v"(__double2hiint(b)), "v"(__double2hiint(a)), "s"(m));
    return __hiloint2double(hi, lo);
}
// c ? 0 : b
__device__ __forceinline__ double pick_zero(bool c, double b) {
    const unsigned long long m = __builtin_amdgcn_ballot_w64(c);
    int lo, hi;
    asm("s_nop 1\n\tv_cndmask_b32_e64 %0, %2, 0, %4\n\tv_cndmask_b32_e64 %1, %3, 0, %4"
        : "=&v"(lo), "=v"(hi)
        : "v"(__double2loint(b)), "v"(__double2hiint(b)), "s"(m));
    return __hiloint2double(hi, lo);
}
__device__ __forceinline__ float pick(bool c, float a, float b) { return c ? a : b; }

// min / max.  FP64 selects as the reference's MIN / MAX (a compare and a
// select); FP32 uses the hardware v_min_f32 / v_max_f32, which differ only
// for NaN operands.
template <typename R>
__device__ __forceinline__ R rmin(R a, R b) { return a < b ? a : b; }
template <typename R>
__device__ __forceinline__ R rmax(R a, R b) { return a > b ? a : b; }
template <>
__device__ __forceinline__ float rmin<float>(float a, float b) { return __builtin_fminf(a, b); }
template <>
__device__ __forceinline__ float rmax<float>(float a, float b) { return __builtin_fmaxf(a, b); }
// min(x, c) with c a number: of a NaN, c, as the select's.
__device__ __forceinline__ double rcap(double x, double c) { return __builtin_fmin(x, c); }
__device__ __forceinline__ float rcap(float x, float c) { return __builtin_fminf(x, c); }
// max(0, x), a NaN staying one
__device__ __forceinline__ double rpos0(double x) { return pick_zero(0.0 > x, x); }
__device__ __forceinline__ float rpos0(float x) { return __builtin_fmaxf(0.0f, x); }
// The parts of a speed below and above zero: of a NaN, 0, as the selects
// min(x, 0) and max(x, 0); they differ from those in the sign of a zero, which
// no sum they enter keeps.
__device__ __forceinline__ double rneg(double x) { return __builtin_fmin(x, 0.0); }
__device__ __forceinline__ double rplus(double x) { return __builtin_fmax(x, 0.0); }
__device__ __forceinline__ float rneg(float x) { return __builtin_fminf(x, 0.0f); }
__device__ __forceinline__ float rplus(float x) { return __builtin_fmaxf(x, 0.0f); }

// Sums that start at zero: 0 + x and 0 - x.  FP64 keeps the reference's
// accumulations from zero, whose only effect is the sign of a zero result;
// FP32 drops them.
template <typename R>
__device__ __forceinline__ R zadd(R x) { return sizeof(R) == 4 ? x : R(0) + x; }
template <typename R>
__device__ __forceinline__ R zsub(R x) { return sizeof(R) == 4 ? -x : R(0) - x; }

// a b + c.  FP64 rounds twice, as the reference does; FP32 is one fused
// operation, written out instead of left to the compiler's contraction, so that
// every copy of the code gives the same bits.
__device__ __forceinline__ double mad(double a, double b, double c) {
#pragma clang fp contract(off)
    return a * b + c;
}
__device__ __forceinline__ float mad(float a, float b, float c) { return __builtin_fmaf(a, b, c); }

// The next term a b of an unrolled sum, which its first term starts.
template <typename R>
__device__ __forceinline__ void sum_term(R& sum, R a, R b, bool& first) {
#pragma clang fp contract(off)
    sum = first ? R(a * b) : mad(a, b, sum);
    first = false;
}

// Division and square root.  FP64 keeps IEEE-correct operations (the parity
// form); the FP32-bulk form uses the hardware reciprocal and square root
// (v_rcp_f32, v_sqrt_f32, 1 ulp), whose error is far below the form's
// stated tolerance.
template <typename R>
__device__ __forceinline__ R dv(R a, R b) { return a / b; }

// FP64 reciprocal of the flux form's FP64 fluxes: the hardware estimate
// (v_rcp_f64) refined by two Newton-Raphson steps r <- r + r (1 - x r), which
// square the relative error each.  Not correctly rounded (within a few ulp),
// which the flux form does not need: both cells beside an interface evaluate
// its flux with this same code on the same values, so they get the same bits.
__device__ __forceinline__ double flux_rcp(double x) {
    double r = __builtin_amdgcn_rcp(x);
    r = __builtin_fma(r, __builtin_fma(-x, r, 1.0), r);
    r = __builtin_fma(r, __builtin_fma(-x, r, 1.0), r);
    return r;
}
template <>
__device__ __forceinline__ float dv<float>(float a, float b) { return a * __builtin_amdgcn_rcpf(b); }
template <typename R>
__device__ __forceinline__ R sq(R a) { return sqrt(a); }
template <>
__device__ __forceinline__ float sq<float>(float a) { return __builtin_amdgcn_sqrtf(a); }

// FP64 quotients q = n / b of one b, as IEEE rounds them.  With `fast` (the same
// in every lane) b's reciprocal is refined once and each quotient corrected by
// its exact residual (Markstein, "Computation of elementary functions on the IBM
// RISC System/6000 processor", 1990), without the scaling that a general division
// needs: b and 1 / b have to be normal numbers and every n zero, infinite, not a
// number, or within FAST_EXP powers of two of 1.  A general division takes 27 ns,
// the reciprocal 18 and each quotient 10 (per SIMD, two waves on it).
constexpr int FAST_EXP = 900;
template <int N>
__device__ __forceinline__ void quotients(const double (&n)[N], double b, bool fast, double (&q)[N]) {
    if (fast) {
        const double y = flux_rcp(b);
#pragma unroll
        for (int k = 0; k < N; k++) {
            const double t = n[k] * y;
            q[k] = __builtin_amdgcn_div_fixup(__builtin_fma(__builtin_fma(-b, t, n[k]), y, t), b, n[k]);
        }
    } else {
#pragma unroll
        for (int k = 0; k < N; k++) q[k] = n[k] / b;
    }
}
// The correctly rounded square root of a number between 2^-900 and 2^900
// (Goldschmidt's iteration from the hardware estimate, then two corrections by
// the exact residual; P. Markstein, "Software division and square root using
// Goldschmidt's algorithms", RNC6, 2004): 26 ns where the general one takes 39.
__device__ __forceinline__ double fast_root(double x) {
    const double y = __builtin_amdgcn_rsq(x);
    double g = x * y, h = 0.5 * y;
    const double r = __builtin_fma(-h, g, 0.5);
    g = __builtin_fma(g, r, g);
    h = __builtin_fma(h, r, h);
    g = __builtin_fma(__builtin_fma(-g, g, x), h, g);
    return __builtin_fma(__builtin_fma(-g, g, x), h, g);
}
__device__ __forceinline__ bool all_lanes(bool x) { return __builtin_amdgcn_ballot_w64(!x) == 0; }
// x > 0 and within 2^+-100; |x| zero, infinite, not a number or between 2^lo and
// 2^hi.
__device__ __forceinline__ bool moderate(double x) {
    return (unsigned) (__double2hiint(x) - ((1023 - 100) << 20)) < 200u << 20;
}
__device__ __forceinline__ bool exponent_within(double x, int lo, int hi) {
    return (unsigned) (__builtin_amdgcn_frexp_exp(x) - lo) <= (unsigned) (hi - lo);
}

// A solver that divides by one value several times (RP::RANGED; with the tests
// that spare the entropy fix its divisions, 100 dam break steps 24.2 -> 23.3 ms,
// 100 shock-bubble steps 12.5 -> 11.7 ms, batched 24 x 20 shallow water 134 -> 125
// us): RP::in_range(q,
// pp) says whether a cell's values allow the fast forms above, RP::cells gives
// `cell` in both directions, rpn2c takes whether both cells are in range, rpt2_pair
// splits both fluctuations of an interface, and right_going gives apdq once more
// from the waves, their speeds and amdq, so that it need not be kept beside them.
template <class RP, class = void>
struct ranged : std::false_type {};
template <class RP>
struct ranged<RP, std::enable_if_t<RP::RANGED>> : std::true_type {};

// A solver whose rpt2 is linear in asdq (RP::RPT2_LINEAR): the FP32 form then
// scales asdq by dt / (2 dx) before the transverse solve instead of scaling
// both results after it.  Solvers without the flag keep the reference's order.
template <class RP, class = void>
struct rpt2_linear : std::false_type {};
template <class RP>
struct rpt2_linear<RP, std::enable_if_t<RP::RPT2_LINEAR>> : std::true_type {};

// A solver whose wave speeds follow from what rpn2 hands to rpt2
// (RP::speeds(roe, s), the same operations): they need not be kept beside it.
template <class RP, class = void>
struct roe_speeds : std::false_type {};
template <class RP>
struct roe_speeds<RP, std::void_t<decltype(&RP::speeds)>> : std::true_type {};

// A solver whose FP32 arithmetic names its fused operations (RP::EXPLICIT_FMA):
// every inlined copy of it gives the same bits.
template <class RP, class = void>
struct explicit_fma : std::false_type {};
template <class RP>
struct explicit_fma<RP, std::enable_if_t<RP::EXPLICIT_FMA>> : std::true_type {};

// ----------------------------------------------------------------- shallow water
// Wave components that are zero by construction.  A sum over the waves that
// starts at +0 may skip those terms without changing its bits (in
// round-to-nearest such a sum is never -0, so adding x * 0 = ±0 leaves it
// as it is), so the step kernel and the solvers skip them.
template <class RP, int IXY, class = void>
struct wave_zeros {
    __host__ __device__ static constexpr bool at(int, int) { return false; }
};
template <class RP, int IXY>
struct wave_zeros<RP, IXY, decltype((void) RP::template wave_zero<IXY>(0, 0))> {
    __host__ __device__ static constexpr bool at(int mw, int m) { return RP::template wave_zero<IXY>(mw, m); }
};

template <typename R>
struct RPShallow {
    static constexpr int MEQN = 3, MWAVES = 3, MAUX = 0;
    static constexpr bool CONSERVATIVE = true;  // amdq + apdq = f(qR) - f(qL)
    static constexpr bool RPT2_LINEAR = true;   // bm, bp linear in asdq
    static constexpr bool EXPLICIT_FMA = true;  // no contraction left to the compiler (mad)
    static constexpr bool RANGED = sizeof(R) == 8;
    // u, v, a (and in FP32 1 / (2 a), which rpt2 then takes from the normal solve)
    static constexpr int NROE = sizeof(R) == 4 ? 4 : 3;

    __device__ __forceinline__ static void speeds(const R roe[NROE], R s[MWAVES]) {
        s[0] = roe[0] - roe[2]; s[1] = roe[0]; s[2] = roe[0] + roe[2];
    }

    // the shear wave carries no depth and no normal momentum
    template <int IXY>
    __host__ __device__ static constexpr bool wave_zero(int mw, int m) {
        return mw == 1 && (m == 0 || m == (IXY == 1 ? 1 : 2));
    }

    // What rpn2 computes from one cell alone: sqrt(h), hu_n / sqrt(h),
    // hu_t / sqrt(h), u_n = hu_n / h and sqrt(g h) (n: the sweep's normal
    // direction).  The step kernel evaluates them once per cell and hands each
    // interface its two cells' values (the same operations, so the same bits).
    static constexpr int NCELL = 5;
    //
    // FP32 takes all five from one hardware reciprocal square root (v_rsq_f32,
    // 1 ulp): sqrt(h) = h / sqrt(h), 1 / h = (1 / sqrt(h))^2, sqrt(g h) =
    // sqrt(g) sqrt(h); FP64 keeps the reference's divisions and square roots.
    template <int IXY>
    __device__ __forceinline__ static void cell(const R* q, const PhysParams& pp, R c[NCELL]) {
        constexpr int mu = IXY == 1 ? 1 : 2, mv = IXY == 1 ? 2 : 1;
        if constexpr (sizeof(R) == 4) {
            const float rs = __builtin_amdgcn_rsqf(q[0]);
            const float hs = q[0] * rs;
            c[0] = hs;
            c[1] = q[mu] * rs;
            c[2] = q[mv] * rs;
            c[3] = c[1] * rs;
            c[4] = sqrt_grav(pp) * hs;
        } else {
            const R hs = sq(q[0]);
            c[0] = hs;
            c[1] = dv(q[mu], hs);
            c[2] = dv(q[mv], hs);
            c[3] = dv(q[mu], q[0]);
            c[4] = sq((R) pp.grav * q[0]);
        }
    }

    // Depth and gravity within 2^+-100, momenta zero or between 2^-600 and
    // 2^200: u is then zero or above 2^-760, u + a and a difference of depths or
    // momenta zero or above a sum's last place, 2^-155, 2^-152 and 2^-652, so the
    // numerators of rpn2 are zero or above 2^-760 and all below 2^410.
    __device__ __forceinline__ static bool in_range(const double* q, const PhysParams& pp) {
        return moderate(q[0]) && moderate(pp.grav) && exponent_within(q[1], -600, 200) && exponent_within(q[2], -600, 200);
    }

    __device__ __forceinline__ static void cells(const double* q, const PhysParams& pp, bool fast, double cx[NCELL],
                                                 double cy[NCELL]) {
        const double n[2] = {q[1], q[2]};
        double hs, c, r[2], u[2];
        if (fast) {
            hs = fast_root(q[0]);
            c = fast_root(pp.grav * q[0]);
            quotients(n, hs, true, r);
            quotients(n, q[0], true, u);
        } else {
            hs = sqrt(q[0]);
            c = sqrt(pp.grav * q[0]);
            quotients(n, hs, false, r);
            quotients(n, q[0], false, u);
        }
        cx[0] = cy[0] = hs;
        cx[1] = cy[2] = r[0];
        cx[2] = cy[1] = r[1];
        cx[3] = u[0];
        cy[3] = u[1];
        cx[4] = cy[4] = c;
    }

    // sqrt(g) in FP32 (uniform; the compiler keeps it out of the sweeps' loops)
    __device__ __forceinline__ static float sqrt_grav(const PhysParams& pp) {
        return __builtin_amdgcn_sqrtf((float) pp.grav);
    }

    // u_n - sqrt(g h) (SIGN = -1) or u_n + sqrt(g h) (SIGN = +1) of the
    // intermediate state h, hu_n of the entropy fix
    template <int SIGN>
    __device__ __forceinline__ static R char_speed(R hu, R h, const PhysParams& pp) {
        return SIGN < 0 ? dv(hu, h) - sq((R) pp.grav * h) : dv(hu, h) + sq((R) pp.grav * h);
    }

    template <int IXY>
    __device__ __forceinline__ static void rpn2(const R* qL, const R* qR, const R* auxL,
                                                const R* auxR, const PhysParams& pp,
                                                R wave[MWAVES][MEQN], R s[MWAVES], R amdq[MEQN],
                                                R apdq[MEQN], R roe[NROE]) {
        R cL[NCELL], cR[NCELL];
        cell<IXY>(qL, pp, cL);
        cell<IXY>(qR, pp, cR);
        rpn2c<IXY>(qL, qR, cL, cR, auxL, auxR, pp, wave, s, amdq, apdq, roe);
    }

    // rpn2 from the two cells' values of `cell`
    template <int IXY>
    __device__ __forceinline__ static void rpn2c(const R* qL, const R* qR, const R* cL,
                                                 const R* cR, const R* /*auxL*/,
                                                 const R* /*auxR*/, const PhysParams& pp,
                                                 R wave[MWAVES][MEQN], R s[MWAVES], R amdq[MEQN],
                                                 R apdq[MEQN], R roe[NROE], bool fast = false) {
        if constexpr (sizeof(R) == 4) rpn2c_fp32<IXY>(qL, qR, cL, cR, pp, wave, s, amdq, apdq, roe);
        else rpn2c_fp64<IXY>(qL, qR, cL, cR, pp, wave, s, amdq, apdq, roe, fast);
    }

    // FP32: one reciprocal and one reciprocal square root for the Roe averages
    // (1 / (2 a) = rsq(g h) / 2), and the entropy fix without branches: the
    // states left and right of the shear wave have the same depth and normal
    // momentum, so one intermediate state serves both, and at most one of the
    // two outer waves is transonic there.
    template <int IXY>
    __device__ __forceinline__ static void rpn2c_fp32(const R* qL, const R* qR, const R* cL, const R* cR,
                                                      const PhysParams& pp, R wave[MWAVES][MEQN],
                                                      R s[MWAVES], R amdq[MEQN], R apdq[MEQN], R roe[NROE]) {
#pragma clang fp contract(off)
        constexpr int mu = IXY == 1 ? 1 : 2, mv = IXY == 1 ? 2 : 1;
        const float gh = (0.5f * (float) pp.grav) * (qL[0] + qR[0]);
        const float ra = __builtin_amdgcn_rsqf(gh), rh = __builtin_amdgcn_rcpf(cL[0] + cR[0]);
        const float u = (cL[1] + cR[1]) * rh, v = (cL[2] + cR[2]) * rh;
        const float a = gh * ra, inv2a = 0.5f * ra;
        roe[0] = u; roe[1] = v; roe[2] = a; roe[NROE - 1] = inv2a;
        const float d0 = qR[0] - qL[0], d1 = qR[mu] - qL[mu], d2 = qR[mv] - qL[mv];
        const float s0 = u - a, s2 = u + a;
        const float a1 = mad(s2, d0, -d1) * inv2a, a3 = mad(-s0, d0, d1) * inv2a, a2 = mad(-v, d0, d2);
        wave[0][0] = a1;   wave[0][mu] = a1 * s0; wave[0][mv] = a1 * v; s[0] = s0;
        wave[1][0] = 0.0f; wave[1][mu] = 0.0f;    wave[1][mv] = a2;     s[1] = u;
        wave[2][0] = a3;   wave[2][mu] = a3 * s2; wave[2][mv] = a3 * v; s[2] = s2;
        // characteristic speeds of the left, intermediate and right states
        const float hm = qL[0] + a1, hum = qL[mu] + wave[0][mu];
        const float rm = __builtin_amdgcn_rsqf(hm), um = hum * rm * rm, cm = sqrt_grav(pp) * (hm * rm);
        const float lL = cL[3] - cL[4], lR = cR[3] + cR[4], l1 = um - cm, l3 = um + cm;
        const bool t1 = lL < 0.0f && l1 > 0.0f, t3 = l3 < 0.0f && lR > 0.0f;
        const float r = __builtin_amdgcn_rcpf(t3 ? lR - l3 : l1 - lL);
        const float f1 = t1 ? lL * ((l1 - s0) * r) : rneg(s0);
        float f3 = t3 ? l3 * ((lR - s2) * r) : rneg(s2);
        f3 = u > 0.0f ? 0.0f : f3;
        const float f2 = rneg(u), g1 = s0 - f1, g2 = rplus(u), g3 = s2 - f3;
        amdq[0] = mad(f3, a3, f1 * a1);
        amdq[mu] = mad(f3, wave[2][mu], f1 * wave[0][mu]);
        amdq[mv] = mad(f2, a2, mad(f3, wave[2][mv], f1 * wave[0][mv]));
        apdq[0] = mad(g3, a3, g1 * a1);
        apdq[mu] = mad(g3, wave[2][mu], g1 * wave[0][mu]);
        apdq[mv] = mad(g2, a2, mad(g3, wave[2][mv], g1 * wave[0][mv]));
    }

    // Whether the entropy fix has to look at the speed of an intermediate state:
    // not if that is subcritical by a margin above all rounding,
    // (hu)^2 < 0.998 g h^3, since hu / h -+ sqrt(g h) then has the sign of -+1.
    __device__ __forceinline__ static bool near_critical(R hu, R h, const PhysParams& pp) {
        const R t = (R) pp.grav * h * h * h;
        return !(hu * hu < R(0.998) * t && t > R(1e-200) && t < R(1e300));
    }

    template <int IXY>
    __device__ __forceinline__ static void rpn2c_fp64(const R* qL, const R* qR, const R* cL, const R* cR,
                                                      const PhysParams& pp, R wave[MWAVES][MEQN],
                                                      R s[MWAVES], R amdq[MEQN], R apdq[MEQN], R roe[NROE],
                                                      bool fast) {
        constexpr int mu = IXY == 1 ? 1 : 2, mv = IXY == 1 ? 2 : 1;
        const R grav = (R) pp.grav;
        const R h = dv(qL[0] + qR[0], R(2));
        const R hsqrtl = cL[0];
        const R hsqrtr = cR[0];
        const R hsq2 = hsqrtl + hsqrtr;
        const R d0 = qR[0] - qL[0], d1 = qR[mu] - qL[mu], d2 = qR[mv] - qL[mv];
        const R nu[2] = {cL[1] + cR[1], cL[2] + cR[2]};
        R uv[2], a13[2], a;
        auto averages = [&](bool f) __attribute__((always_inline)) {
            quotients(nu, hsq2, f, uv);
            a = f ? fast_root(grav * h) : sqrt(grav * h);
            const R na[2] = {(uv[0] + a) * d0 - d1, -((uv[0] - a) * d0) + d1};
            quotients(na, R(2) * a, f, a13);
        };
        if (fast) averages(true);
        else averages(false);
        const R u = uv[0], v = uv[1], a1 = a13[0], a3 = a13[1];
        roe[0] = u; roe[1] = v; roe[2] = a;
        const R a2 = -(v * d0) + d2;

        wave[0][0] = a1;   wave[0][mu] = a1 * (u - a); wave[0][mv] = a1 * v; s[0] = u - a;
        wave[1][0] = R(0); wave[1][mu] = R(0);         wave[1][mv] = a2;     s[1] = u;
        wave[2][0] = a3;   wave[2][mu] = a3 * (u + a); wave[2][mv] = a3 * v; s[2] = u + a;

        // entropy fix
        const R s0 = cL[3] - cL[4];   // dv(qL[mu], qL[0]) - sq(grav * qL[0])
        if (s0 > R(0) && s[0] > R(0)) {
#pragma unroll
            for (int m = 0; m < 3; m++) amdq[m] = R(0);
        } else {
            const R h1 = qL[0] + wave[0][0];
            const R hu1 = qL[mu] + wave[0][mu];
            R sfract = rneg(s[0]);
            if (near_critical(hu1, h1, pp)) {
                const R s1 = char_speed<-1>(hu1, h1, pp);
                if (s0 < R(0) && s1 > R(0)) sfract = s0 * dv(s1 - s[0], s1 - s0);
            }
#pragma unroll
            for (int m = 0; m < 3; m++) amdq[m] = sfract * wave[0][m];
            if (!(s[1] > R(0))) {
#pragma unroll
                for (int m = 0; m < 3; m++) amdq[m] = amdq[m] + s[1] * wave[1][m];
                const R s03 = cR[3] + cR[4];   // dv(qR[mu], qR[0]) + sq(grav * qR[0])
                const R h3 = qR[0] - wave[2][0];
                const R hu3 = qR[mu] - wave[2][mu];
                bool add = s[2] < R(0);
                sfract = s[2];
                if (near_critical(hu3, h3, pp)) {
                    const R s3 = char_speed<1>(hu3, h3, pp);
                    if (s3 < R(0) && s03 > R(0)) {
                        sfract = s3 * dv(s03 - s[2], s03 - s3);
                        add = true;
                    }
                }
                if (add) {
#pragma unroll
                    for (int m = 0; m < 3; m++) amdq[m] = amdq[m] + sfract * wave[2][m];
                }
            }
        }
        right_going<IXY>(wave, s, amdq, apdq);
    }

    // apdq: what amdq leaves of the waves' sum (FP64)
    template <int IXY>
    __device__ __forceinline__ static void right_going(const R wave[MWAVES][MEQN], const R s[MWAVES], const R amdq[MEQN],
                                                       R apdq[MEQN]) {
#pragma clang fp contract(off)
#pragma unroll
        for (int m = 0; m < MEQN; m++) {
            R df = R(0);
            bool first = true;
#pragma unroll
            for (int mw = 0; mw < MWAVES; mw++)
                if (!wave_zero<IXY>(mw, m)) sum_term(df, s[mw], wave[mw][m], first);
            apdq[m] = df - amdq[m];
        }
    }

    template <int IXY>
    __device__ __forceinline__ static void rpt2(const R roe[NROE], const R asdq[MEQN],
                                                const R* /*aux1*/, const R* /*aux2*/,
                                                const R* /*aux3*/, const PhysParams&, R bm[MEQN],
                                                R bp[MEQN]) {
        constexpr int mu = IXY == 1 ? 1 : 2, mv = IXY == 1 ? 2 : 1;
        const R u = roe[0], v = roe[1], a = roe[2];
        if constexpr (sizeof(R) == 4) {
#pragma clang fp contract(off)
            // waves a1 (1, u, v - a), a2 (0, 1, 0), a3 (1, u, v + a), summed by
            // their common factors
            const float r2 = roe[NROE - 1];
            const float a1 = mad(v + a, asdq[0], -asdq[mv]) * r2, a3 = mad(a - v, asdq[0], asdq[mv]) * r2;
            const float a2 = mad(-u, asdq[0], asdq[mu]);
            const float m1 = rneg(v - a) * a1, m3 = rneg(v + a) * a3;
            const float p1 = rplus(v - a) * a1, p3 = rplus(v + a) * a3;
            bm[0] = m1 + m3;
            bm[mu] = mad(u, bm[0], rneg(v) * a2);
            bm[mv] = mad(v, bm[0], a * (m3 - m1));
            bp[0] = p1 + p3;
            bp[mu] = mad(u, bp[0], rplus(v) * a2);
            bp[mv] = mad(v, bp[0], a * (p3 - p1));
        } else {
            const R a1 = dv((v + a) * asdq[0] - asdq[mv], R(2) * a);
            const R a3 = dv(-((v - a) * asdq[0]) + asdq[mv], R(2) * a);
            split<IXY>(roe, asdq, a1, a3, bm, bp);
        }
    }

    // both fluctuations of an interface; fast: its cells are in range
    template <int IXY>
    __device__ __forceinline__ static void rpt2_pair(const double roe[NROE], const double amdq[MEQN],
                                                     const double apdq[MEQN], bool fast, double bmA[MEQN],
                                                     double bpA[MEQN], double bmP[MEQN], double bpP[MEQN]) {
        constexpr int mv = IXY == 1 ? 2 : 1;
        const double v = roe[1], a = roe[2];
        const double n[4] = {(v + a) * amdq[0] - amdq[mv], -((v - a) * amdq[0]) + amdq[mv],
                             (v + a) * apdq[0] - apdq[mv], -((v - a) * apdq[0]) + apdq[mv]};
        bool ok = true;
#pragma unroll
        for (int k = 0; k < 4; k++) ok = ok && exponent_within(n[k], -FAST_EXP, FAST_EXP);
        double w[4];
        if (fast && all_lanes(ok)) quotients(n, 2.0 * a, true, w);
        else quotients(n, 2.0 * a, false, w);
        split<IXY>(roe, amdq, w[0], w[1], bmA, bpA);
        split<IXY>(roe, apdq, w[2], w[3], bmP, bpP);
    }

    template <int IXY>
    __device__ __forceinline__ static void split(const R roe[NROE], const R asdq[MEQN], R a1, R a3, R bm[MEQN],
                                                 R bp[MEQN]) {
        constexpr int mu = IXY == 1 ? 1 : 2, mv = IXY == 1 ? 2 : 1;
        const R u = roe[0], v = roe[1], a = roe[2];
        const R a2 = asdq[mu] - u * asdq[0];
        R wb[3][3], sb[3];
        wb[0][0] = a1;   wb[0][mu] = a1 * u; wb[0][mv] = a1 * (v - a); sb[0] = v - a;
        wb[1][0] = R(0); wb[1][mu] = a2;     wb[1][mv] = R(0);         sb[1] = v;
        wb[2][0] = a3;   wb[2][mu] = a3 * u; wb[2][mv] = a3 * (v + a); sb[2] = v + a;
#pragma unroll
        for (int m = 0; m < 3; m++) {
            R m_ = rneg(sb[0]) * wb[0][m], p_ = rplus(sb[0]) * wb[0][m];
#pragma unroll
            for (int mw = 1; mw < 3; mw++) {
                if (mw == 1 && m != mu) continue;   // wb[1][0], wb[1][mv] are zero
                m_ = m_ + rneg(sb[mw]) * wb[mw][m];
                p_ = p_ + rplus(sb[mw]) * wb[mw][m];
            }
            bm[m] = m_;
            bp[m] = p_;
        }
    }

    // physical flux f(q) (IXY = 1) or g(q) (IXY = 2), used by the flux form
    template <int IXY>
    __device__ __forceinline__ static void flux(const double* q, const double* /*aux*/,
                                                const PhysParams& pp, double* f) {
        constexpr int mu = IXY == 1 ? 1 : 2, mv = IXY == 1 ? 2 : 1;
        const double h = q[0], un = q[mu] / h;
        f[0] = q[mu];
        f[mu] = q[mu] * un + 0.5 * pp.grav * h * h;
        f[mv] = q[mv] * un;
    }

    // f(q) and g(q) of one cell with one division (the flux form's update).
    // Never contracted into FMAs: both cells beside an interface evaluate it
    // and must get the same bits.
    __device__ __forceinline__ static void fluxes(const double* q, const double* /*aux*/,
                                                  const PhysParams& pp, double* f, double* g) {
#pragma clang fp contract(off)
        const double h = q[0], rh = flux_rcp(h), u = q[1] * rh, v = q[2] * rh;
        const double p = 0.5 * pp.grav * h * h;
        f[0] = q[1]; f[1] = q[1] * u + p; f[2] = q[2] * u;
        g[0] = q[2]; g[1] = q[1] * v;     g[2] = q[2] * v + p;
    }

    // conservative flux stored in the time-sync registers, operation for
    // operation as applications/clawpack/shallow/2d/radialdam/rpn2cons_update.f:27-46
    template <int IXY>
    __device__ __forceinline__ static void consflux(const double* q, const double* /*aux*/,
                                                    const PhysParams& pp, double* f) {
        consflux_of<IXY>(q, q[IXY == 1 ? 1 : 2] / q[0], pp, f);
    }
    template <int IXY>
    __device__ __forceinline__ static void consflux_of(const double* q, double un, const PhysParams& pp, double* f) {
        constexpr int mu = IXY == 1 ? 1 : 2, mv = IXY == 1 ? 2 : 1;
        const double hun = q[mu], hut = q[mv], h = q[0];
        f[0] = hun;
        f[mu] = (hun * hun) / h + (0.5 * pp.grav) * (h * h);
        f[mv] = un * hut;
    }
    // the same from the cell's values in both directions (`cells`)
    template <int IXY>
    __device__ __forceinline__ static void consflux_cells(const double* q, const double cx[NCELL], const double cy[NCELL],
                                                          const PhysParams& pp, double* f) {
        consflux_of<IXY>(q, IXY == 1 ? cx[3] : cy[3], pp, f);
    }
};

// ----------------------------------------------------------------- Euler
template <typename R>
struct RPEuler {
    static constexpr int MEQN = 4, MWAVES = 4, MAUX = 0;
    static constexpr bool CONSERVATIVE = true;
    static constexpr bool RPT2_LINEAR = true;   // bm, bp linear in asdq
    static constexpr bool EXPLICIT_FMA = true;  // no contraction left to the compiler (mad)
    static constexpr bool RANGED = sizeof(R) == 8;
    // u, v, a, enth, g1a2, and in FP32 u2v2, euv and 1 / (2 a) of the normal solve
    // (FP64 has no registers for the first two of them, which rpt2 computes again)
    static constexpr int NROE = sizeof(R) == 4 ? 8 : 5;

    __device__ __forceinline__ static void speeds(const R roe[NROE], R s[MWAVES]) {
        s[0] = roe[0] - roe[2]; s[1] = s[2] = roe[0]; s[3] = roe[0] + roe[2];
    }

    // the shear wave carries no density and no normal momentum
    template <int IXY>
    __host__ __device__ static constexpr bool wave_zero(int mw, int m) {
        return mw == 1 && (m == 0 || m == (IXY == 1 ? 1 : 2));
    }

    // What rpn2 computes from one cell alone (n: the sweep's normal
    // direction): sqrt(rho), rho u_n / sqrt(rho), rho u_t / sqrt(rho),
    // (E + p) / sqrt(rho) with p from (rho u)^2 + (rho v)^2, u_n and the sound
    // speed of the entropy fix, whose p sums the momenta in the sweep's order.
    // The step kernel evaluates them once per cell (the same operations, so
    // the same bits).  FP32 takes sqrt(rho), 1 / sqrt(rho) and 1 / rho from one
    // hardware reciprocal square root; FP64 keeps the reference's divisions.
    static constexpr int NCELL = 6;
    template <int IXY>
    __device__ __forceinline__ static void cell(const R* q, const PhysParams& pp, R c[NCELL]) {
        constexpr int mu = IXY == 1 ? 1 : 2, mv = IXY == 1 ? 2 : 1;
        const R gamma = (R) pp.gamma;
        const R gamma1 = (R) (pp.gamma - 1.0);
        if constexpr (sizeof(R) == 4) {
#pragma clang fp contract(off)
            const float r = __builtin_amdgcn_rsqf(q[0]);
            // one pressure (the two summation orders differ only in rounding)
            const float u = q[1] * r, v = q[2] * r, p = gamma1 * mad(-0.5f, mad(u, u, v * v), q[3]);
            c[0] = q[0] * r;
            c[1] = q[mu] * r;
            c[2] = q[mv] * r;
            c[3] = (q[3] + p) * r;
            c[4] = c[1] * r;
            c[5] = __builtin_amdgcn_sqrtf(gamma * p) * r;
            return;
        }
        const R rs = sq(q[0]);
        const R p = gamma1 * (q[3] - dv(R(0.5) * (q[1] * q[1] + q[2] * q[2]), q[0]));
        const R pn = gamma1 * (q[3] - dv(R(0.5) * (q[mu] * q[mu] + q[mv] * q[mv]), q[0]));
        c[0] = rs;
        c[1] = dv(q[mu], rs);
        c[2] = dv(q[mv], rs);
        c[3] = dv(q[3] + p, rs);
        c[4] = dv(q[mu], q[0]);
        c[5] = sq(dv(gamma * pn, q[0]));
    }

    // (the momenta's squares are summed in one order for both directions: a sum
    // of two rounds the same either way)
    __device__ __forceinline__ static void cells(const double* q, const PhysParams& pp, bool fast, double cx[NCELL],
                                                 double cy[NCELL]) {
#pragma clang fp contract(off)
        const double gamma1 = pp.gamma - 1.0;
        const double k[1] = {0.5 * (q[1] * q[1] + q[2] * q[2])};
        double rs, r[3], u[3];
        auto values = [&](bool f) __attribute__((always_inline)) {
            rs = f ? fast_root(q[0]) : sqrt(q[0]);
            double d[1];
            quotients(k, q[0], f, d);
            const double p = gamma1 * (q[3] - d[0]);
            const double nr[3] = {q[1], q[2], q[3] + p}, nu[3] = {q[1], q[2], pp.gamma * p};
            quotients(nr, rs, f, r);
            quotients(nu, q[0], f, u);
        };
        if (fast) values(true);
        else values(false);
        cx[0] = cy[0] = rs;
        cx[1] = cy[2] = r[0];
        cx[2] = cy[1] = r[1];
        cx[3] = cy[3] = r[2];
        cx[4] = u[0];
        cy[4] = u[1];
        cx[5] = cy[5] = sqrt(u[2]);
    }

    // Density, energy and gamma - 1 within 2^+-100, momenta zero or between
    // 2^-300 and 2^200: their squares over the density are zero or above 2^-701,
    // the pressures and enthalpies zero or above a sum's last place, 2^-860, and
    // all below 2^520.
    __device__ __forceinline__ static bool in_range(const double* q, const PhysParams& pp) {
        return moderate(q[0]) && moderate(q[3]) && moderate(pp.gamma - 1.0) && exponent_within(q[1], -300, 200) &&
               exponent_within(q[2], -300, 200);
    }

    // Whether the entropy fix has to look at the speed of an intermediate state:
    // not if that is subsonic by a margin above all rounding,
    // (rho u)^2 < 0.99 gamma p rho, with a pressure that is no small difference.
    __device__ __forceinline__ static bool near_sonic(R rho, R rhou, R rhov, R en, R gamma, R gamma1) {
#pragma clang fp contract(off)
        const R e = en * rho, t = gamma * gamma1 * (e - R(0.5) * (rhou * rhou + rhov * rhov));
        return !(rhou * rhou < R(0.99) * t && t > R(1e-6) * e && e > R(1e-200) && e < R(1e300) && rho > R(0));
    }

    template <int IXY>
    __device__ __forceinline__ static void rpn2(const R* qL, const R* qR, const R* auxL,
                                                const R* auxR, const PhysParams& pp,
                                                R wave[MWAVES][MEQN], R s[MWAVES], R amdq[MEQN],
                                                R apdq[MEQN], R roe[NROE]) {
        R cL[NCELL], cR[NCELL];
        cell<IXY>(qL, pp, cL);
        cell<IXY>(qR, pp, cR);
        rpn2c<IXY>(qL, qR, cL, cR, auxL, auxR, pp, wave, s, amdq, apdq, roe);
    }

    // rpn2 from the two cells' values of `cell`
    template <int IXY>
    __device__ __forceinline__ static void rpn2c(const R* qL, const R* qR, const R* cL,
                                                 const R* cR, const R* /*auxL*/,
                                                 const R* /*auxR*/, const PhysParams& pp,
                                                 R wave[MWAVES][MEQN], R s[MWAVES], R amdq[MEQN],
                                                 R apdq[MEQN], R roe[NROE], bool fast = false) {
#pragma clang fp contract(off)
        constexpr int mu = IXY == 1 ? 1 : 2, mv = IXY == 1 ? 2 : 1;
        const R gamma = (R) pp.gamma;
        const R gamma1 = (R) (pp.gamma - 1.0);
        const R rhsqrtl = cL[0];
        const R rhsqrtr = cR[0];
        const R rhsq2 = rhsqrtl + rhsqrtr;
        R u, v, enth, a, g1a2, inv2a = R(0);
        if constexpr (sizeof(R) == 4) {
            // one reciprocal and one reciprocal square root: a = a2s rsq(a2s),
            // gamma1 / a2s = gamma1 rsq(a2s)^2, 1 / (2 a) = rsq(a2s) / 2
            const float rh = __builtin_amdgcn_rcpf(rhsq2);
            u = (cL[1] + cR[1]) * rh;
            v = (cL[2] + cR[2]) * rh;
            enth = (cL[3] + cR[3]) * rh;
        } else {
            const R n[3] = {cL[1] + cR[1], cL[2] + cR[2], cL[3] + cR[3]};
            R r[3];
            quotients(n, rhsq2, fast, r);
            u = r[0]; v = r[1]; enth = r[2];
        }
        const R u2v2 = mad(v, v, u * u);
        const R a2s = gamma1 * mad(R(-.5), u2v2, enth);
        if constexpr (sizeof(R) == 4) {
            const float ra = __builtin_amdgcn_rsqf(a2s);
            a = a2s * ra;
            g1a2 = gamma1 * (ra * ra);
            inv2a = 0.5f * ra;
            roe[7] = inv2a;
        } else {
            a = sq(a2s);
            g1a2 = dv(gamma1, a2s);
        }
        const R euv = enth - u2v2;
        roe[0] = u; roe[1] = v; roe[2] = a; roe[3] = enth; roe[4] = g1a2;
        if constexpr (sizeof(R) == 4) { roe[5] = u2v2; roe[6] = euv; }

        const R d0 = qR[0] - qL[0], d1 = qR[mu] - qL[mu], d2 = qR[mv] - qL[mv], d3 = qR[3] - qL[3];
        const R a3 = g1a2 * (mad(v, d2, mad(u, d1, euv * d0)) - d3);
        const R a2 = mad(-v, d0, d2);
        const R t4 = mad(-a, a3, mad(a - u, d0, d1));
        R a4;
        if constexpr (sizeof(R) == 4) a4 = t4 * inv2a;
        else a4 = dv(t4, R(2) * a);
        const R a1 = d0 - a3 - a4;

        wave[0][0] = a1; wave[0][mu] = a1 * (u - a); wave[0][mv] = a1 * v;
        wave[0][3] = a1 * mad(-u, a, enth); s[0] = u - a;
        wave[1][0] = R(0); wave[1][mu] = R(0); wave[1][mv] = a2;
        wave[1][3] = a2 * v; s[1] = u;
        wave[2][0] = a3; wave[2][mu] = a3 * u; wave[2][mv] = a3 * v;
        wave[2][3] = a3 * R(0.5) * u2v2; s[2] = u;
        wave[3][0] = a4; wave[3][mu] = a4 * (u + a); wave[3][mv] = a4 * v;
        wave[3][3] = a4 * mad(u, a, enth); s[3] = u + a;

        // entropy fix
        const R s0 = cL[4] - cL[5];   // u_n - c of the left cell
        if (s0 >= R(0) && s[0] > R(0)) {
#pragma unroll
            for (int m = 0; m < 4; m++) amdq[m] = R(0);
        } else {
            const R rho1 = qL[0] + wave[0][0];
            const R rhou1 = qL[mu] + wave[0][mu];
            const R rhov1 = qL[mv] + wave[0][mv];
            const R en1 = qL[3] + wave[0][3];
            R sfract = rneg(s[0]);
            if (sizeof(R) == 4 || near_sonic(rho1, rhou1, rhov1, en1, gamma, gamma1)) {
                const R p1 = gamma1 * (en1 - dv(R(0.5) * mad(rhov1, rhov1, rhou1 * rhou1), rho1));
                const R c1 = sq(dv(gamma * p1, rho1));
                const R s1 = dv(rhou1, rho1) - c1;
                if (s0 < R(0) && s1 > R(0)) sfract = dv(s0 * (s1 - s[0]), s1 - s0);
            }
#pragma unroll
            for (int m = 0; m < 4; m++) amdq[m] = sfract * wave[0][m];
            if (!(s[1] >= R(0))) {
#pragma unroll
                for (int m = 0; m < 4; m++) {
                    amdq[m] = mad(s[1], wave[1][m], amdq[m]);
                    amdq[m] = mad(s[2], wave[2][m], amdq[m]);
                }
                const R s3 = cR[4] + cR[5];   // u_n + c of the right cell
                const R rho2 = qR[0] - wave[3][0];
                const R rhou2 = qR[mu] - wave[3][mu];
                const R rhov2 = qR[mv] - wave[3][mv];
                const R en2 = qR[3] - wave[3][3];
                bool add = s[3] < R(0);
                sfract = s[3];
                if (sizeof(R) == 4 || near_sonic(rho2, rhou2, rhov2, en2, gamma, gamma1)) {
                    const R p2 = gamma1 * (en2 - dv(R(0.5) * mad(rhov2, rhov2, rhou2 * rhou2), rho2));
                    const R c2 = sq(dv(gamma * p2, rho2));
                    const R s2 = dv(rhou2, rho2) + c2;
                    if (s2 < R(0) && s3 > R(0)) {
                        sfract = dv(s2 * (s3 - s[3]), s3 - s2);
                        add = true;
                    }
                }
                if (add) {
#pragma unroll
                    for (int m = 0; m < 4; m++) amdq[m] = mad(sfract, wave[3][m], amdq[m]);
                }
            }
        }
        right_going<IXY>(wave, s, amdq, apdq);
    }

    // apdq: what amdq leaves of the waves' sum (FP64)
    template <int IXY>
    __device__ __forceinline__ static void right_going(const R wave[MWAVES][MEQN], const R s[MWAVES], const R amdq[MEQN],
                                                       R apdq[MEQN]) {
#pragma clang fp contract(off)
#pragma unroll
        for (int m = 0; m < MEQN; m++) {
            R df = R(0);
            bool first = true;
#pragma unroll
            for (int mw = 0; mw < MWAVES; mw++)
                if (!wave_zero<IXY>(mw, m)) sum_term(df, s[mw], wave[mw][m], first);
            apdq[m] = df - amdq[m];
        }
    }

    template <int IXY>
    __device__ __forceinline__ static void rpt2(const R roe[NROE], const R asdq[MEQN],
                                                const R* /*aux1*/, const R* /*aux2*/,
                                                const R* /*aux3*/, const PhysParams&, R bm[MEQN],
                                                R bp[MEQN]) {
#pragma clang fp contract(off)
        constexpr int mu = IXY == 1 ? 1 : 2, mv = IXY == 1 ? 2 : 1;
        const R u = roe[0], v = roe[1], a = roe[2], enth = roe[3], g1a2 = roe[4];
        const R u2v2 = sizeof(R) == 4 ? roe[NROE - 3] : mad(v, v, u * u);
        const R euv = sizeof(R) == 4 ? roe[NROE - 2] : enth - u2v2;
        const R a3 = g1a2 * (mad(v, asdq[mv], mad(u, asdq[mu], euv * asdq[0])) - asdq[3]);
        const R a2 = mad(-u, asdq[0], asdq[mu]);
        const R t4 = mad(-a, a3, mad(a - v, asdq[0], asdq[mv]));
        if constexpr (sizeof(R) == 4) {
            // waves a1 (1, u, v - a, H - v a), a3 (1, u, v, (u^2 + v^2) / 2) +
            // a2 (0, 1, 0, u), a4 (1, u, v + a, H + v a), summed by their common
            // factors
            const float a4 = t4 * roe[7], a1 = asdq[0] - a3 - a4;
            auto split = [&](float w1, float w2, float w4, float* b) {
#pragma clang fp contract(off)
                const float x1 = w1 * a1, x4 = w4 * a4, y3 = w2 * a3, y2 = w2 * a2;
                const float t = x1 + x4, d = a * (x4 - x1);
                b[0] = t + y3;
                b[mu] = mad(u, b[0], y2);
                b[mv] = mad(v, b[0], d);
                b[3] = mad(enth, t, mad(v, d, mad(0.5f * u2v2, y3, u * y2)));
            };
            split(rneg(v - a), rneg(v), rneg(v + a), bm);
            split(rplus(v - a), rplus(v), rplus(v + a), bp);
            return;
        }
        const R a4 = dv(t4, R(2) * a);
        const R a1 = asdq[0] - a3 - a4;
        R wb[3][4], sb[3];
        wb[0][0] = a1; wb[0][mu] = a1 * u; wb[0][mv] = a1 * (v - a);
        wb[0][3] = a1 * (enth - v * a); sb[0] = v - a;
        wb[1][0] = a3; wb[1][mu] = a3 * u + a2; wb[1][mv] = a3 * v;
        wb[1][3] = a3 * R(0.5) * u2v2 + a2 * u; sb[1] = v;
        wb[2][0] = a4; wb[2][mu] = a4 * u; wb[2][mv] = a4 * (v + a);
        wb[2][3] = a4 * (enth + v * a); sb[2] = v + a;
#pragma unroll
        for (int m = 0; m < 4; m++) {
            R m_ = rneg(sb[0]) * wb[0][m], p_ = rplus(sb[0]) * wb[0][m];
#pragma unroll
            for (int mw = 1; mw < 3; mw++) {
                m_ = m_ + rneg(sb[mw]) * wb[mw][m];
                p_ = p_ + rplus(sb[mw]) * wb[mw][m];
            }
            bm[m] = m_;
            bp[m] = p_;
        }
    }

    // both fluctuations of an interface (one quotient each)
    template <int IXY>
    __device__ __forceinline__ static void rpt2_pair(const double roe[NROE], const double amdq[MEQN],
                                                     const double apdq[MEQN], bool /*fast*/, double bmA[MEQN],
                                                     double bpA[MEQN], double bmP[MEQN], double bpP[MEQN]) {
        const PhysParams none{};
        rpt2<IXY>(roe, amdq, nullptr, nullptr, nullptr, none, bmA, bpA);
        rpt2<IXY>(roe, apdq, nullptr, nullptr, nullptr, none, bmP, bpP);
    }

    template <int IXY>
    __device__ __forceinline__ static void flux(const double* q, const double* /*aux*/,
                                                const PhysParams& pp, double* f) {
        constexpr int mu = IXY == 1 ? 1 : 2, mv = IXY == 1 ? 2 : 1;
        const double rho = q[0], un = q[mu] / rho;
        const double p = (pp.gamma - 1.0) * (q[3] - 0.5 * (q[1] * q[1] + q[2] * q[2]) / rho);
        f[0] = q[mu];
        f[mu] = q[mu] * un + p;
        f[mv] = q[mv] * un;
        f[3] = (q[3] + p) * un;
    }

    // f(q) and g(q) of one cell with one division (the flux form's update).
    // Never contracted into FMAs: both cells beside an interface evaluate it
    // and must get the same bits.
    __device__ __forceinline__ static void fluxes(const double* q, const double* /*aux*/,
                                                  const PhysParams& pp, double* f, double* g) {
#pragma clang fp contract(off)
        const double rr = flux_rcp(q[0]), u = q[1] * rr, v = q[2] * rr;
        const double p = (pp.gamma - 1.0) * (q[3] - 0.5 * (q[1] * u + q[2] * v));
        f[0] = q[1]; f[1] = q[1] * u + p; f[2] = q[2] * u; f[3] = (q[3] + p) * u;
        g[0] = q[2]; g[1] = q[1] * v;     g[2] = q[2] * v + p; g[3] = (q[3] + p) * v;
    }

    // conservative flux stored in the time-sync registers (the reference has
    // no Euler rpn2_cons; this is the physical flux, evaluated as the oracle does)
    template <int IXY>
    __device__ __forceinline__ static void consflux(const double* q, const double* /*aux*/,
                                                    const PhysParams& pp, double* f) {
        constexpr int mu = IXY == 1 ? 1 : 2, mv = IXY == 1 ? 2 : 1;
        consflux_of<IXY>(q, q[mu] / q[0], q[mv] / q[0], pp, f);
    }
    template <int IXY>
    __device__ __forceinline__ static void consflux_of(const double* q, double un, double ut, const PhysParams& pp,
                                                       double* f) {
        constexpr int mu = IXY == 1 ? 1 : 2, mv = IXY == 1 ? 2 : 1;
        const double rho = q[0], en = q[3];
        const double p = (pp.gamma - 1.0) * (en - 0.5 * rho * (un * un + ut * ut));
        f[0] = q[mu];
        f[mu] = q[mu] * un + p;
        f[mv] = q[mu] * ut;
        f[3] = un * (en + p);
    }
    // the same from the cell's values in both directions (`cells`)
    template <int IXY>
    __device__ __forceinline__ static void consflux_cells(const double* q, const double cx[NCELL], const double cy[NCELL],
                                                          const PhysParams& pp, double* f) {
        if constexpr (IXY == 1) consflux_of<IXY>(q, cx[4], cy[4], pp, f);
        else consflux_of<IXY>(q, cy[4], cx[4], pp, f);
    }
};

// ----------------------------------------------------------------- advection
// aux(:,:,1) = u, aux(:,:,2) = v.  The normal speed is the right cell's aux
// component IXY; rpt2 takes the transverse velocity from aux2 (bmasdq) and
// aux3 (bpasdq) as clawpack46_rpt2adv.f:79-86.
template <typename R>
struct RPAdvection {
    static constexpr int MEQN = 1, MWAVES = 1, MAUX = 2;
    // colour equation q_t + u q_x + v q_y = 0: the fluctuations are not a flux
    // difference unless the velocity is uniform, so no flux form exists
    static constexpr bool CONSERVATIVE = false;
    static constexpr bool RPT2_LINEAR = true;   // bm, bp linear in asdq
    static constexpr bool EXPLICIT_FMA = true;  // no contraction left to the compiler (mad)
    static constexpr int NROE = 1;

    template <int IXY>
    __device__ __forceinline__ static void rpn2(const R* qL, const R* qR, const R* /*auxL*/,
                                                const R* auxR,
                                                const PhysParams&, R wave[MWAVES][MEQN],
                                                R s[MWAVES], R amdq[MEQN], R apdq[MEQN],
                                                R roe[NROE]) {
#pragma clang fp contract(off)
        const R delta = qR[0] - qL[0];
        wave[0][0] = delta;
        s[0] = auxR[IXY - 1];
        amdq[0] = R(0) + rneg(s[0]) * wave[0][0];
        apdq[0] = R(0) + rplus(s[0]) * wave[0][0];
        roe[0] = R(0);
    }

    template <int IXY>
    __device__ __forceinline__ static void rpt2(const R* /*roe*/, const R asdq[MEQN],
                                                const R* /*aux1*/, const R* aux2, const R* aux3,
                                                const PhysParams&, R bm[MEQN], R bp[MEQN]) {
#pragma clang fp contract(off)
        constexpr int kv = IXY == 1 ? 1 : 0;   // the transverse velocity component
        bm[0] = rneg(aux2[kv]) * asdq[0];
        bp[0] = rplus(aux3[kv]) * asdq[0];
    }

    template <int IXY>
    __device__ __forceinline__ static void flux(const double* q, const double* aux,
                                                const PhysParams&, double* f) {
        f[0] = aux[IXY - 1] * q[0];
    }

    __device__ __forceinline__ static void fluxes(const double* q, const double* aux,
                                                  const PhysParams&, double* f, double* g) {
#pragma clang fp contract(off)
        f[0] = aux[0] * q[0];
        g[0] = aux[1] * q[0];
    }

    // conservative flux stored in the time-sync registers: u_n q with the
    // cell's velocity (applications/clawpack/advection/2d/adv_order3/user_4.6/rpn2cons_update.f:14-26)
    template <int IXY>
    __device__ __forceinline__ static void consflux(const double* q, const double* aux,
                                                    const PhysParams&, double* f) {
        f[0] = aux[IXY - 1] * q[0];
    }
};

}  // namespace hipclaw
