// Batched patch update, one wave per group of column strips.
//
// The same step as step_tiles (hipclaw_step.h), organised without barriers: a
// wave holds S strips of W interior columns, one staged column (W + 4 of them,
// with the halo) per lane, and marches up the rows.  Rows and the y-interfaces
// between them live in registers (some in the lane's own LDS words where that
// gains a wave per SIMD); the x-direction goes across lanes with DPP shifts.  With row n loaded the wave
//
//   * sweeps row n - 1 in x (normal and transverse solves);
//   * solves the y-interface between rows n - 1 and n;
//   * limits, corrects and splits the y-interface between rows n - 2 and
//     n - 1, whose limiter needed the one above it;
//   * updates and stores row n - 2.
//
// Every sum is taken in the order step_tiles takes it, so the FP64 form gives
// the same bits.  Sums do not start from a zero, which the reference's do and
// which only turns a sum of -0 into +0: the two flux parts fm and gm whose
// differences enter the update keep theirs (zadd), so that no difference is -0
// where the reference's is +0, and no other use of a sum tells the zeros apart
// (60 fewer FP64 additions per row for shallow water, 80 for Euler: batched
// 24 x 20 shallow water 138 -> 133 us, dam break 255 -> 248 us per step).
#pragma once

#include <type_traits>

#include "hipclaw_step.h"
#include "hipclaw_strip_shape.h"

namespace hipclaw {

// Any value: what a skipped stage leaves behind is not read, and must not keep
// the registers it stands in alive.
template <typename V, int N>
__device__ __forceinline__ void unset(V (&v)[N]) {
#pragma unroll
    for (int k = 0; k < N; k++) v[k] = __builtin_nondeterministic_value(v[k]);
}

// Register update (reg_add of the tile kernel) of a position's fields, el v each.
// Each register has one writer per launch, so that adding to it (ACC, subcycling)
// needs no old value back: an add done in the L2, with the same rounding, that
// nothing waits for.  One that is known to be zero (fresh) is simply written: the
// adds are a tenth of a subcycled step (71 us for 1,480 patches of 16 x 16, 62
// with stores in their place).
template <int ACC, int N, typename V>
__device__ __forceinline__ void reg_put(double* r, int stride, double el, const V (&v)[N], bool fresh) {
    if (ACC && !fresh) {
#pragma unroll
        for (int m = 0; m < N; m++) unsafeAtomicAdd(r + m * stride, el * (double) v[m]);
    } else {
#pragma unroll
        for (int m = 0; m < N; m++) r[m * stride] = 0.0 + el * (double) v[m];
    }
}

// x, computed where it stands: an address used in a rare branch of the row loop
// must not be hoisted out of it into registers that live through every row.
__device__ __forceinline__ int opaque(int x) {
    asm volatile("" : "+v"(x));
    return x;
}

// What a step leaves to the next stands in LDS, each lane its own column, where
// that gains a wave per SIMD: sets of MEQN values, of which the last three are kept
// for the two latest rows, then MWAVES products.
//   * Euler FP64, 324 registers: two waves instead of one (100 shock-bubble steps on
//     2,740 patches of 16 x 16 11.1 -> 9.8 ms).  Its 40 values are 20 KiB per wave,
//     eight waves all of a CU's 160.
//   * Shallow water FP32, 186 registers: three instead of two (200 dam break steps
//     on 11,296 patches of 32 x 32 64.1 -> 63.0 ms, 100 ensemble steps 26.4 -> 26.1).
template <class RP, typename R>
constexpr bool strip_carry() {
    return sizeof(R) == 8 ? RP::MEQN * RP::MWAVES > 9 && ranged<RP>::value
                          : RP::MEQN * RP::MWAVES == 9 && explicit_fma<RP>::value;
}
enum { CARRY_TU = 0, CARRY_PD, CARRY_PU, CARRY_FXM, CARRY_FXP = CARRY_FXM + 2, CARRY_GPL = CARRY_FXP + 2,
       CARRY_DL = CARRY_GPL + 2 };
template <class RP, typename R>
constexpr int strip_lds() { return strip_carry<RP, R>() ? (CARRY_DL * RP::MEQN + RP::MWAVES) * 64 * (int) sizeof(R) : 0; }

// Waves per SIMD the register allocation aims for, with nothing in scratch: a
// reload waits for the stores in flight (shallow water FP32 with three waves and 6
// spills, before the values above stood in LDS, 0.412 ms on 11,296 patches of
// 32 x 32, with two waves and none 0.331).  A registered FP64 solver of more wave
// components than shallow water gets all 512 registers.
template <class RP, typename R>
constexpr int strip_waves_per_eu() {
    return RP::MEQN * RP::MWAVES == 1 || (sizeof(R) == 4 && strip_carry<RP, R>()) ? 3
           : sizeof(R) == 8 && RP::MEQN * RP::MWAVES > 9 && !strip_carry<RP, R>() ? 1 : 2;
}

template <class RP, typename R, bool FLUXFORM, int KEEP, bool STD>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(strip_waves_per_eu<RP, R>())))
step_strips(StepArgs a, StripShape sh) {
#pragma clang fp contract(off)
    constexpr int MEQN = RP::MEQN, MW = RP::MWAVES, MAUX = RP::MAUX, NROE = RP::NROE;
    constexpr int NC = cell_values<RP>::N, NCD = NC > 0 ? NC : 1;
    constexpr int MAD = MAUX > 0 ? MAUX : 1;
    constexpr bool REGS = KEEP > 0;
    constexpr int ACC = KEEP == 2;        // registers add up over substeps
    // Steps per round of the row loop: two copies of the step change their
    // results over by name instead of by register moves, but only where both
    // give the same bits.
    constexpr int U = sizeof(R) == 4 && explicit_fma<RP>::value ? 2 : 1;
    // FP32 with a linear rpt2: the factor dt / (2 dx) goes on asdq
    constexpr bool PRE = sizeof(R) == 4 && rpt2_linear<RP>::value;
    constexpr bool RANGED = ranged<RP>::value;
    constexpr bool CARRY = strip_carry<RP, R>();
    extern __shared__ double carry_mem[];
    using WZ1 = wave_zeros<RP, 1>;
    using WZ2 = wave_zeros<RP, 2>;

    const int mx = a.mx, my = a.my, mbc = a.mbc;
    const int nxp = mx + 2 * mbc;
    const long long plane = (long long) nxp * (my + 2 * mbc);
    const int H = sh.H;
    const int lane = threadIdx.x & 63;

    // Workgroups are dispatched round-robin over the 8 XCDs: each XCD takes one
    // contiguous run of waves, so that neighbouring strips find the cells they
    // share in the same L2.  (The grid is a multiple of 8.)
    const int blk = (int) (blockIdx.x & 7) * (int) (gridDim.x >> 3) + (int) (blockIdx.x >> 3);
    const int wid = blk * (int) (blockDim.x >> 6) + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    if (wid == 0 && lane == 0) a.cfl[2] = __builtin_amdgcn_s_memrealtime();   // (of the first workgroup)
    const int pw = wid / sh.nsy, ty = wid - pw * sh.nsy;
    const int round = pw / sh.waves, wk = pw - round * sh.waves;
    const int patch0 = round * sh.patches;
    if (patch0 >= a.nwork) return;        // (the whole wave)
    // the lane's segment, staged column kp in it and patch; lanes without a
    // column repeat another one and write nothing
    unsigned sg = 0;
    if (sh.waves > StripShape::WAVES) {
        const int most = StripShape::LANES - StripShape::HALO;
        sg = strip_segment(0, min(most, mx - wk * most), 0, wk * most);
    } else {
#pragma unroll
        for (int k = 0; k < StripShape::SEGS; k++) {
            unsigned w = 0;
#pragma unroll
            for (int v = 0; v < StripShape::WAVES; v++) w = wk == v ? sh.seg[v][k] : w;
            if (k == 0 || (w && lane >= (int) (w & 63))) sg = w;
        }
    }
    const int W = (sg >> 6) & 63;
    int kp = lane - (int) (sg & 63);
    int pi = patch0 + (int) ((sg >> 12) & 15);
    const bool act = kp < W + 4 && pi < a.nwork;
    kp = min(kp, W + 3);
    pi = min(pi, a.nwork - 1);
    const int slot = a.work[pi];
    const int i0 = 1 + (int) (sg >> 16), j0 = 1 + min(ty * H, my - H);
    const int i = i0 - 2 + kp;                       // the lane's patch column (1-based)
    const bool incol = act && kp >= 2 && kp <= W + 1;   // an interior column of the strip
    const bool ifx = act && kp >= 2 && kp <= W + 2;     // x-interfaces (left of the lane's cell) of the strip
    const bool ify = act && kp >= 1 && kp <= W + 2;     // columns whose y-interfaces count for the Courant number

    const double dt = a.dtscale ? a.dt * a.dtscale[slot] : a.dt;
    const double dxs = a.dxs[slot], dys = a.dys[slot];
    const double dtdx64 = dt / dxs, dtdy64 = dt / dys;
    const R dtdx = (R) dtdx64, dtdy = (R) dtdy64;

    // offsets of the lane's column to a same-size neighbour's cells, for rows
    // below, in and above the patch (StepArgs::pull)
    int dlo = 0, dmid = 0, dhi = 0;
    if (a.pull) {
        const int* __restrict__ pt = a.pull + 8 * (long long) slot;
        const bool gx = i < 1 || i > mx;
        const int hx = i > mx ? 1 : 0;
        dmid = gx ? pt[hx] : 0;
        dlo = gx ? pt[4 + hx] : pt[2];
        dhi = gx ? pt[6 + hx] : pt[3];
    }
    // deferred fix-up: whether the lane's column lies on a corrected x-face, and
    // that face's increments (of row j at qx[m my + j])
    bool fix = false;
    const double* qx = nullptr;
    if (a.qcorr && (i == 1 || i == mx)) {
        const int face = i == 1 ? 0 : 1;
        fix = (a.cmask[slot] >> face) & 1;
        qx = a.qcorr + (long long) slot * a.cstride + face * MEQN * my - 1;
    }
    const double* qp = a.qsrc + (long long) slot * a.pstride + (long long) (j0 + mbc - 3) * nxp + (i + mbc - 1);
    const double* ap = MAUX > 0 ? a.aux + (long long) slot * a.astride + (long long) (j0 + mbc - 3) * nxp + (i + mbc - 1)
                                : nullptr;
    double* qo = a.qdst + (long long) slot * a.pstride + (long long) (j0 + mbc - 1) * nxp + (i + mbc - 1);

    // time-sync registers: whether the lane's x-interface lies on a patch face,
    // whether its cell is the first interior or first ghost cell of one, and that
    // face's registers from the strip's first row on; rows of an overlapping last
    // strip that the strip before it owns are left to it.  What only the patch's
    // first and last rows need is looked up there.
    const int own_y = ty * H + 1 - j0;
    const bool bottom = j0 == 1, top = j0 + H - 1 == my;
    const bool onface = act && ((kp == 2 && i == 1) || (kp == W + 2 && i == mx + 1));
    const bool byface = onface || (act && ((kp == 1 && i == 0) || (kp == W + 1 && i == mx)));
    const double dtdy_el = dt * dys;
    double* rx = nullptr;
    if constexpr (REGS) rx = a.reg + (long long) slot * a.rstride + (i <= 1 ? 0 : 4 * MEQN * mx) + j0 - 1;
    const bool freshx = ACC && a.cmask && ((a.cmask[slot] >> (i <= 1 ? 0 : 1)) & 1);
    // the registers of y-face `face`, kind 0, at the lane's column; length of the face
    // times dt; whether they are zero
    auto yreg = [&](int face, double* el, bool* fresh) __attribute__((always_inline)) {
        const int sl = opaque(slot);
        *fresh = ACC && a.cmask && ((a.cmask[sl] >> face) & 1);
        *el = (a.dtscale ? a.dt * a.dtscale[sl] : a.dt) * a.dxs[sl];
        return a.reg + (long long) sl * a.rstride + face * 4 * MEQN * mx + i - 1;
    };

    double pq[MEQN], pv[MEQN];            // the row in flight, and the pending fix-up of its x-face cells
    R pa[MAD];
    double qr[4][MEQN];                   // rows A (n - 2), B (n - 1), C (n) and N (n + 1), in turn
    R ar[4][MAD];
    int j = j0 - 2;                       // patch row of the row in flight

    // What one step leaves to the next, in two copies that steps of even and
    // odd n write in turn: per-cell values of the Riemann solver for row C
    // (x and y); the y-interface between rows B and C as solved, with its waves'
    // products with those of the interface below; the transverse parts of row B
    // at its upper face and its normal x-flux parts; of the y-interface between
    // rows A and B the transverse parts it sends up and its flux.
    R cx[2][NCD], cy[2][NCD];
    R wv[2][MW][MEQN], sv[2][MW], am[2][MEQN], apq[2][MEQN], ro[2][NROE], dl[2][MW];
    R tu[2][MEQN], fxm[2][MEQN], fxp[2][MEQN];
    R gPd[2][MEQN], gPu[2][MEQN], gpl[2][MEQN];
    double G[2][MEQN];
    bool inA = false, inB = false, inC = false;   // every lane's cell of the row is in range (RP::RANGED)
    R smaxx = R(0), smaxy = R(0);         // largest |s| of every interface the lane solves
    const R halfx = R(0.5) * dtdx, halfy = R(0.5) * dtdy;
    R* const carry = (R*) carry_mem + (threadIdx.x >> 6) * ((CARRY_DL * MEQN + MW) * 64) + lane;


    // Step n: row C is row n.  Every stage is entered as the rows it needs are
    // there, from the same code in every row, so that a flux at the seam of two
    // strips has the same bits in both.  Two steps per round: what they leave to
    // each other changes places by name instead of by moves.
#pragma unroll 1
    for (int n0 = -1; n0 <= H + 3; n0 += U) {
#pragma unroll
        for (int e = 0; e < U; e++) {
            const int n = n0 + e;
            const int P = e, O = 1 - e, A = e, B = e + 1, C = e + 2, N = (e + 3) & 3;
            if (U > 1 && n > H + 3) break;
            R* const kept = carry + (n & 1) * (MEQN * 64);          // this row's and
            R* const last = carry + (1 - (n & 1)) * (MEQN * 64);    // the last row's sets of the two latest rows
            // ---- row n + 1 under way ----
            if (n < H + 3) {
                const double* p = qp + (j < 1 ? dlo : j > my ? dhi : dmid);
#pragma unroll
                for (int m = 0; m < MEQN; m++) pq[m] = p[m * plane];
                if (fix && j >= 1 && j <= my) {
#pragma unroll
                    for (int m = 0; m < MEQN; m++) pv[m] = qx[m * my + j];
                }
                if constexpr (MAUX > 0) {
#pragma unroll
                    for (int m = 0; m < MAUX; m++) pa[m] = (R) ap[m * plane];
                    ap += nxp;
                }
                qp += nxp;
            }
            if constexpr (NC > 0) {
                R q[MEQN];
#pragma unroll
                for (int m = 0; m < MEQN; m++) q[m] = (R) qr[C][m];
                if constexpr (RANGED) {
                    inC = all_lanes(RP::in_range(q, a.pp));
                    RP::cells(q, a.pp, inC, cx[P], cy[P]);
                } else {
                    RP::template cell<1>(q, a.pp, cx[P]);
                    RP::template cell<2>(q, a.pp, cy[P]);
                }
            }
            if constexpr (REGS && !FLUXFORM) {
                // FP64 form: conservative flux of the pre-step state at the first
                // interior and first ghost cell of every patch edge
                // (clawpack46_time_sync.f:58-147)
                double ac[MAD], fl[MEQN];
#pragma unroll
                for (int m = 0; m < MAD; m++) ac[m] = MAUX > 0 ? (double) ar[C][m] : 0.0;
                const int b = n - 2;          // interior row of the strip
                if (byface && b >= own_y && b >= 0 && b < H) {
                    if constexpr (RANGED) RP::template consflux_cells<1>(qr[C], cx[P], cy[P], a.pp, fl);
                    else RP::template consflux<1>(qr[C], ac, a.pp, fl);
                    double* r = rx + b + (i == 0 || i == mx + 1 ? REG_EFOUT : REG_EFIN) * MEQN * mx;
                    reg_put<ACC>(r, mx, dtdy_el, fl, freshx);
                }
                const bool below = bottom && (b == -1 || b == 0), above = top && (b == H - 1 || b == H);
                if ((below || above) && incol) {
                    if constexpr (RANGED) RP::template consflux_cells<2>(qr[C], cx[P], cy[P], a.pp, fl);
                    else RP::template consflux<2>(qr[C], ac, a.pp, fl);
                    double el;
                    bool fr;
                    // (a strip of one row has both faces, one after the other)
                    if (below) {
                        double* r = yreg(2, &el, &fr) + (b < 0 ? REG_EFOUT : REG_EFIN) * MEQN * mx;
                        reg_put<ACC>(r, mx, el, fl, fr);
                    }
                    if (above) {
                        double* r = yreg(3, &el, &fr) + (b == H ? REG_EFOUT : REG_EFIN) * MEQN * mx;
                        reg_put<ACC>(r, mx, el, fl, fr);
                    }
                }
            }

            // ---- x sweep of row B (n - 1) ----
            R gt[MEQN], gm[MEQN];             // of the y-face between rows A and B: transverse part, flux part
            if (n >= 2) {
                R qL[MEQN], qR[MEQN], auxL[MAD];
#pragma unroll
                for (int m = 0; m < MEQN; m++) { qR[m] = (R) qr[B][m]; qL[m] = prev_lane(qR[m]); }
#pragma unroll
                for (int m = 0; m < MAD; m++) auxL[m] = MAUX > 0 ? prev_lane(ar[B][m]) : R(0);
                R w[MW][MEQN], s[MW], amdq[MEQN], apdq[MEQN], roe[NROE];
                if constexpr (NC > 0) {
                    R cL[NCD];
#pragma unroll
                    for (int c = 0; c < NC; c++) cL[c] = prev_lane(cx[O][c]);
                    if constexpr (RANGED)
                        RP::template rpn2c<1>(qL, qR, cL, cx[O], auxL, ar[B], a.pp, w, s, amdq, apdq, roe, inB);
                    else
                        RP::template rpn2c<1>(qL, qR, cL, cx[O], auxL, ar[B], a.pp, w, s, amdq, apdq, roe);
                } else {
                    RP::template rpn2<1>(qL, qR, auxL, ar[B], a.pp, w, s, amdq, apdq, roe);
                }
#pragma unroll
                for (int mw = 0; mw < MW; mw++) smaxx = fmax(smaxx, fabs(s[mw]));
                R cq[MEQN];
#pragma unroll
                for (int m = 0; m < MEQN; m++) cq[m] = R(0);
                if (STD || a.order2) {
                    R dotl[MW], dotr[MW];
#pragma unroll
                    for (int mw = 0; mw < MW; mw++) {
                        R d = R(0);
                        bool first = true;
#pragma unroll
                        for (int m = 0; m < MEQN; m++) {
                            if (WZ1::at(mw, m)) continue;
                            const R wl = prev_lane(w[mw][m]);
                            sum_term(d, wl, w[mw][m], first);
                        }
                        dotl[mw] = d;
                        dotr[mw] = next_lane(d);
                    }
                    limited_correction<RP, R, 1, STD, true>(a, w, s, dotl, dotr, dtdx, cq);
                }
#pragma unroll
                for (int m = 0; m < MEQN; m++) {
                    fxm[P][m] = mad(R(0.5), cq[m], zadd(amdq[m]));
                    if constexpr (!FLUXFORM) fxp[P][m] = mad(R(0.5), cq[m], -apdq[m]);
                    if constexpr (CARRY) {
                        kept[(CARRY_FXM * MEQN + m) * 64] = fxm[P][m];
                        if constexpr (!FLUXFORM) kept[(CARRY_FXP * MEQN + m) * 64] = fxp[P][m];
                    }
                }
                if (STD || a.transverse) {
                    if (STD || (a.order2 && a.transverse == 2)) {
#pragma unroll
                        for (int m = 0; m < MEQN; m++) { amdq[m] = amdq[m] + cq[m]; apdq[m] = apdq[m] - cq[m]; }
                    }
                    if constexpr (PRE) {
#pragma unroll
                        for (int m = 0; m < MEQN; m++) { amdq[m] = halfx * amdq[m]; apdq[m] = halfx * apdq[m]; }
                    }
                    R bmA[MEQN], bpA[MEQN], bmP[MEQN], bpP[MEQN];
                    R a1[MAD], a3[MAD];
#pragma unroll
                    for (int m = 0; m < MAD; m++) {
                        a1[m] = MAUX > 0 ? prev_lane(ar[A][m]) : R(0);
                        a3[m] = MAUX > 0 ? prev_lane(ar[C][m]) : R(0);
                    }
                    if constexpr (RANGED) {
                        RP::template rpt2_pair<1>(roe, amdq, apdq, inB, bmA, bpA, bmP, bpP);
                    } else {
                        RP::template rpt2<1>(roe, amdq, a1, auxL, a3, a.pp, bmA, bpA);
                        RP::template rpt2<1>(roe, apdq, ar[A], ar[B], ar[C], a.pp, bmP, bpP);
                    }
#pragma unroll
                    for (int m = 0; m < MEQN; m++) {
                        const R gAd = PRE ? bmA[m] : halfx * bmA[m], gAu = PRE ? bpA[m] : halfx * bpA[m];
                        const R gBd = PRE ? bmP[m] : halfx * bmP[m], gBu = PRE ? bpP[m] : halfx * bpP[m];
                        const R below = CARRY ? carry[(CARRY_TU * MEQN + m) * 64] : tu[O][m];
                        gt[m] = below + (-next_lane(gAd) - gBd);
                        tu[P][m] = -next_lane(gAu) - gBu;
                        if constexpr (CARRY) carry[(CARRY_TU * MEQN + m) * 64] = tu[P][m];
                    }
                } else {
#pragma unroll
                    for (int m = 0; m < MEQN; m++) {
                        gt[m] = R(0);
                        tu[P][m] = R(0);
                        if constexpr (CARRY) carry[(CARRY_TU * MEQN + m) * 64] = R(0);
                    }
                }
            } else {
                unset(gt); unset(tu[P]); unset(fxm[P]); unset(fxp[P]);
            }

            // ---- the y-interface between rows B and C, as solved ----
            R dlo[MW];                        // the products of the interface below
            if (n >= 1) {
                R qL[MEQN], qR[MEQN];
#pragma unroll
                for (int m = 0; m < MEQN; m++) { qL[m] = (R) qr[B][m]; qR[m] = (R) qr[C][m]; }
                if constexpr (RANGED)
                    RP::template rpn2c<2>(qL, qR, cy[O], cy[P], ar[B], ar[C], a.pp, wv[P], sv[P], am[P], apq[P], ro[P], inB && inC);
                else if constexpr (NC > 0)
                    RP::template rpn2c<2>(qL, qR, cy[O], cy[P], ar[B], ar[C], a.pp, wv[P], sv[P], am[P], apq[P], ro[P]);
                else
                    RP::template rpn2<2>(qL, qR, ar[B], ar[C], a.pp, wv[P], sv[P], am[P], apq[P], ro[P]);
#pragma unroll
                for (int mw = 0; mw < MW; mw++) {
                    R d = R(0);
                    bool first = true;
#pragma unroll
                    for (int m = 0; m < MEQN; m++)
                        if (!WZ2::at(mw, m)) sum_term(d, wv[O][mw][m], wv[P][mw][m], first);
                    if constexpr (CARRY) {
                        dlo[mw] = carry[(CARRY_DL * MEQN + mw) * 64];
                        carry[(CARRY_DL * MEQN + mw) * 64] = d;
                    } else {
                        dlo[mw] = dl[O][mw];
                    }
                    dl[P][mw] = d;
                }
            } else {
#pragma unroll
                for (int mw = 0; mw < MW; mw++) unset(wv[P][mw]);
                unset(sv[P]); unset(am[P]); unset(apq[P]); unset(ro[P]); unset(dl[P]); unset(dlo);
            }

            double out[MEQN], Fx[MEQN];       // row A's new values; x-flux left of the cell
            R fm[MEQN], fp[MEQN];
            if (n >= 3) {
                // ---- the y-interface between rows A and B: limiter, flux, transverse ----
                R so[MW];
                if constexpr (roe_speeds<RP>::value) {
                    RP::speeds(ro[O], so);
                } else {
#pragma unroll
                    for (int mw = 0; mw < MW; mw++) so[mw] = sv[O][mw];
                }
                R ap[MEQN];
                if constexpr (RANGED) {
                    RP::template right_going<2>(wv[O], so, am[O], ap);
                } else {
#pragma unroll
                    for (int m = 0; m < MEQN; m++) ap[m] = apq[O][m];
                }
#pragma unroll
                for (int mw = 0; mw < MW; mw++) smaxy = fmax(smaxy, fabs(so[mw]));
                R cq[MEQN];
#pragma unroll
                for (int m = 0; m < MEQN; m++) cq[m] = R(0);
                if (STD || a.order2) limited_correction<RP, R, 2, STD, true>(a, wv[O], so, dlo, dl[P], dtdy, cq);
#pragma unroll
                for (int m = 0; m < MEQN; m++) {
                    gm[m] = gt[m] + mad(R(0.5), cq[m], zadd(am[O][m]));
                    if constexpr (!FLUXFORM) gpl[P][m] = gt[m] + mad(R(0.5), cq[m], -ap[m]);
                    if constexpr (CARRY && !FLUXFORM) kept[(CARRY_GPL * MEQN + m) * 64] = gpl[P][m];
                }
                R nAd[MEQN], nAu[MEQN];
                if (STD || a.transverse) {
                    R amdq[MEQN], apdq[MEQN];
#pragma unroll
                    for (int m = 0; m < MEQN; m++) { amdq[m] = am[O][m]; apdq[m] = ap[m]; }
                    if (STD || (a.order2 && a.transverse == 2)) {
#pragma unroll
                        for (int m = 0; m < MEQN; m++) { amdq[m] = amdq[m] + cq[m]; apdq[m] = apdq[m] - cq[m]; }
                    }
                    if constexpr (PRE) {
#pragma unroll
                        for (int m = 0; m < MEQN; m++) { amdq[m] = halfy * amdq[m]; apdq[m] = halfy * apdq[m]; }
                    }
                    // the rows below and above the interface, left and right of the cell
                    R lA[MAD], rA[MAD], lB[MAD], rB[MAD];
#pragma unroll
                    for (int m = 0; m < MAD; m++) {
                        lA[m] = MAUX > 0 ? prev_lane(ar[A][m]) : R(0);
                        rA[m] = MAUX > 0 ? next_lane(ar[A][m]) : R(0);
                        lB[m] = MAUX > 0 ? prev_lane(ar[B][m]) : R(0);
                        rB[m] = MAUX > 0 ? next_lane(ar[B][m]) : R(0);
                    }
                    if constexpr (RANGED) {
                        RP::template rpt2_pair<2>(ro[O], amdq, apdq, inA && inB, nAd, nAu, gPd[P], gPu[P]);
                    } else {
                        RP::template rpt2<2>(ro[O], amdq, lA, ar[A], rA, a.pp, nAd, nAu);
                        RP::template rpt2<2>(ro[O], apdq, lB, ar[B], rB, a.pp, gPd[P], gPu[P]);
                    }
                    if constexpr (!PRE) {
#pragma unroll
                        for (int m = 0; m < MEQN; m++) {
                            nAd[m] = halfy * nAd[m]; nAu[m] = halfy * nAu[m];
                            gPd[P][m] = halfy * gPd[P][m]; gPu[P][m] = halfy * gPu[P][m];
                        }
                    }
                } else {
#pragma unroll
                    for (int m = 0; m < MEQN; m++) nAd[m] = nAu[m] = gPd[P][m] = gPu[P][m] = R(0);
                }
                // ---- row A: x-fluxes with the transverse parts of its two y-interfaces, update ----
#pragma unroll
                for (int m = 0; m < MEQN; m++) {
                    R pd = gPd[O][m], pu = gPu[O][m], xm = fxm[O][m], xp = fxp[O][m];
                    if constexpr (CARRY) {
                        pd = carry[(CARRY_PD * MEQN + m) * 64];
                        pu = carry[(CARRY_PU * MEQN + m) * 64];
                        xm = last[(CARRY_FXM * MEQN + m) * 64];
                        if constexpr (!FLUXFORM) xp = last[(CARRY_FXP * MEQN + m) * 64];
                        carry[(CARRY_PD * MEQN + m) * 64] = gPd[P][m];
                        carry[(CARRY_PU * MEQN + m) * 64] = gPu[P][m];
                    }
                    const R t1 = -nAd[m] - pd;             // into the x-face left of the cell
                    const R t2 = -nAu[m] - pu;             // into the one right of it
                    const R t2l = prev_lane(t2);
                    fm[m] = (xm + t2l) + t1;
                    if constexpr (!FLUXFORM) fp[m] = (xp + t2l) + t1;
                }
                if constexpr (FLUXFORM) {
                    // FP64 fluxes f and g of the row's cells, each evaluated once: the
                    // flux right of a cell is its f plus the next interface's fm, the
                    // one above it its g plus gm, and each is the next cell's too
                    double f[MEQN], g[MEQN], ac[MAD];
#pragma unroll
                    for (int m = 0; m < MAD; m++) ac[m] = MAUX > 0 ? (double) ar[A][m] : 0.0;
                    RP::fluxes(qr[A], ac, a.pp, f, g);
#pragma unroll
                    for (int m = 0; m < MEQN; m++) {
                        G[P][m] = g[m] + (double) gm[m];
                        const double Fr = f[m] + (double) next_lane(fm[m]);
                        Fx[m] = prev_lane(Fr);
                        out[m] = fmad64(-dtdy64, G[P][m] - G[O][m], fmad64(-dtdx64, Fr - Fx[m], qr[A][m]));
                    }
                } else {
#pragma unroll
                    for (int m = 0; m < MEQN; m++) {
                        const R Dx = next_lane(fm[m]) - fp[m];
                        const R Dy = gm[m] - (CARRY ? last[(CARRY_GPL * MEQN + m) * 64] : gpl[O][m]);
                        if constexpr (sizeof(R) == sizeof(double)) out[m] = (qr[A][m] - dtdx * Dx) - dtdy * Dy;
                        else out[m] = fmad64(-dtdy64, (double) Dy, fmad64(-dtdx64, (double) Dx, qr[A][m]));
                    }
                }
            } else {
                unset(gPd[P]); unset(gPu[P]); unset(gpl[P]); unset(G[P]);
                unset(out); unset(Fx); unset(gm); unset(fm); unset(fp);
            }

            // ---- the row in flight into N, with the pending fix-up of its edge
            // cells in the reference's order (same-size faces before coarse/fine
            // ones).  The wait for the row is here and not where it is first used:
            // the stores of the row just updated come in between, and a wait after
            // them would be for them too ----
#pragma unroll
            for (int m = 0; m < MEQN; m++) {
                asm volatile("" : "+v"(pq[m]));
                qr[N][m] = pq[m];
            }
#pragma unroll
            for (int m = 0; m < MAUX; m++) {
                asm volatile("" : "+v"(pa[m]));
                ar[N][m] = pa[m];
            }
            if (a.qcorr) {
                const bool onx = fix && j >= 1 && j <= my;
                bool done = false;
                if ((j == 1 || j == my) && i >= 1 && i <= mx) {
                    const int sl = opaque(slot), fy = j == 1 ? 2 : 3, mask = a.cmask[sl];
                    if ((mask >> fy) & 1) {
                        const double* qy = a.qcorr + (long long) sl * a.cstride + fy * MEQN * mx + i - 1;
                        const bool yfirst = !onx || sync_y_first(mask, i == 1 ? 0 : 1, fy);
                        done = true;
#pragma unroll
                        for (int m = 0; m < MEQN; m++) {
                            const double w = qy[m * mx], v = onx ? pv[m] : 0.0;
                            double q = qr[N][m];
                            if (yfirst) q = q + w;
                            if (onx) q = q + v;
                            if (!yfirst) q = q + w;
                            qr[N][m] = q;
                        }
                    }
                }
                if (onx && !done) {
#pragma unroll
                    for (int m = 0; m < MEQN; m++) qr[N][m] = qr[N][m] + pv[m];
                }
            }

            if (n >= 3) {
                if constexpr (REGS) {
                    // the y-flux (FP64: both flux parts) through the patch's bottom and top edges
                    const int face = bottom && n == 3 ? 2 : top && n == H + 3 ? 3 : -1;
                    if (face >= 0 && incol) {
                        bool fr;
                        double el, *r = yreg(face, &el, &fr);
                        if constexpr (FLUXFORM) {
                            reg_put<ACC>(r + REG_EFIN * MEQN * mx, mx, el, G[P], fr);
                        } else {
                            reg_put<ACC>(r + REG_FM * MEQN * mx, mx, el, gm, fr);
                            reg_put<ACC>(r + REG_FP * MEQN * mx, mx, -el, gpl[P], fr);
                        }
                    }
                }
            }
            if (n >= 4) {
                // ---- the strip's interior row n - 4 out ----
                if (incol) {
#pragma unroll
                    for (int m = 0; m < MEQN; m++) qo[m * plane] = out[m];
                }
                if constexpr (REGS) {
                    const int b = n - 4;
                    if (onface && b >= own_y) {
                        double* r = rx + b;
                        if constexpr (FLUXFORM) {
                            reg_put<ACC>(r + REG_EFIN * MEQN * mx, mx, dtdy_el, Fx, freshx);
                        } else {
                            reg_put<ACC>(r + REG_FM * MEQN * mx, mx, dtdy_el, fm, freshx);
                            reg_put<ACC>(r + REG_FP * MEQN * mx, mx, -dtdy_el, fp, freshx);
                        }
                    }
                }
                qo += nxp;
            }
            inA = inB;
            inB = inC;
            j++;
        }
        if constexpr (U == 2) {
#pragma unroll
            for (int m = 0; m < MEQN; m++) {
                const double t = qr[0][m];
                qr[0][m] = qr[2][m];
                qr[1][m] = qr[3][m];
                qr[2][m] = t;
            }
#pragma unroll
            for (int m = 0; m < MAUX; m++) {
                const R t = ar[0][m];
                ar[0][m] = ar[2][m];
                ar[1][m] = ar[3][m];
                ar[2][m] = t;
            }
        } else {
#pragma unroll
            for (int m = 0; m < MEQN; m++) {
                qr[0][m] = qr[1][m]; qr[1][m] = qr[2][m]; qr[2][m] = qr[3][m];
                am[1][m] = am[0][m]; apq[1][m] = apq[0][m];
                tu[1][m] = tu[0][m]; fxm[1][m] = fxm[0][m]; fxp[1][m] = fxp[0][m];
                gPd[1][m] = gPd[0][m]; gPu[1][m] = gPu[0][m]; gpl[1][m] = gpl[0][m];
                G[1][m] = G[0][m];
            }
#pragma unroll
            for (int m = 0; m < MAUX; m++) { ar[0][m] = ar[1][m]; ar[1][m] = ar[2][m]; ar[2][m] = ar[3][m]; }
#pragma unroll
            for (int m = 0; m < NCD; m++) { cx[1][m] = cx[0][m]; cy[1][m] = cy[0][m]; }
#pragma unroll
            for (int mw = 0; mw < MW; mw++) {
                sv[1][mw] = sv[0][mw]; dl[1][mw] = dl[0][mw];
#pragma unroll
                for (int m = 0; m < MEQN; m++) wv[1][mw][m] = wv[0][mw][m];
            }
#pragma unroll
            for (int m = 0; m < NROE; m++) ro[1][m] = ro[0][m];
        }
    }

    // ---- CFL: wave64 max over the lanes' interfaces; the wave's end ----
    double cfl = fmax(ifx ? dtdx64 * (double) smaxx : 0.0, ify ? dtdy64 * (double) smaxy : 0.0);
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1) cfl = fmax(cfl, __shfl_xor(cfl, off, 64));
    if (lane == 0) {
        unsigned long long* w = a.cfl + (wid & (CFL_WORDS - 1)) * CFL_STRIDE;
        if (cfl > 0.0) atomicMax(w, (unsigned long long) __double_as_longlong(cfl));
        atomicMax(w + 1, (unsigned long long) __builtin_amdgcn_s_memrealtime());
    }
}

}  // namespace hipclaw
