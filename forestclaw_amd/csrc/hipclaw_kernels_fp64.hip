// FP64 kernels: the oracle-parity patch step, the ghost fill, and the
// compensated mass sums.  This translation unit is compiled with
// -ffp-contract=off so that every FP64 operation rounds exactly as the
// reference's CPU Fortran does.
#include "hipclaw_internal.h"

#include <algorithm>

namespace hipclaw {

#define QIX(i, j, m) (((long long) (m) * nyp + ((j) + mbc - 1)) * nxp + ((i) + mbc - 1))

// fclaw2d_clawpatch_compute_slopes with mth = 5
// (src/patches/clawpatch/fclaw2d_clawpatch_utils.f:45-55)
__device__ __forceinline__ double amr_slope(double sl, double sr) {
    const double sc = (sl + sr) / 2.0;
    const double mn = fmin(fmin(2 * fabs(sl), 2 * fabs(sr)), fabs(sc));
    return mn * fmax(0.0, copysign(1.0, sl * sr)) * copysign(1.0, sc);
}

__device__ __forceinline__ void corner_cell(int mx, int my, int icorner, int ibc, int jbc,
                                            int& i1, int& j1) {
    i1 = (icorner & 1) ? mx + ibc : 1 - ibc;
    j1 = (icorner & 2) ? my + jbc : 1 - jbc;
}

// Interpolate one coarse cell (ic,jc) of `qc` into the 2x2 fine cells whose first
// child is (fi,fj) in `qf` (fclaw2d_clawpatch46_interpolate.f:120-137).
__device__ __forceinline__ void interp_cell(const double* qc, double* qf, int m, int ic, int jc,
                                            int fi, int fj, int nxp, int nyp, int mbc) {
    const double c = qc[QIX(ic, jc, m)];
    const double gx = amr_slope(c - qc[QIX(ic - 1, jc, m)], qc[QIX(ic + 1, jc, m)] - c);
    const double gy = amr_slope(c - qc[QIX(ic, jc - 1, m)], qc[QIX(ic, jc + 1, m)] - c);
    qf[QIX(fi, fj, m)] = c + gx * -0.25 + gy * -0.25;
    qf[QIX(fi + 1, fj, m)] = c + gx * 0.25 + gy * -0.25;
    qf[QIX(fi, fj + 1, m)] = c + gx * -0.25 + gy * 0.25;
    qf[QIX(fi + 1, fj + 1, m)] = c + gx * 0.25 + gy * 0.25;
}

// e / d for e >= 0 and a quotient below 2^22: the product with the reciprocal is
// off by one at most (a general 32-bit division is some 20 instructions).
struct SmallDiv {
    int d;
    float r;
    __device__ __forceinline__ explicit SmallDiv(int n) : d(n), r(__builtin_amdgcn_rcpf((float) n)) {}
    __device__ __forceinline__ int operator()(int e) const {
        const int k = (int) ((float) e * r), rem = e - k * d;
        return rem < 0 ? k - 1 : rem >= d ? k + 1 : k;
    }
};

// One wave per ghost op, OPW ops (waves) per workgroup.  Ops of one phase
// write disjoint ghost cells and read only cells no op of the phase writes,
// so each lane issues the loads of up to U elements before their stores: the
// source and destination slabs are the same allocation, and without this the
// compiler must wait for every store before the next load.
// W lanes (t = 0..W-1) work on the op: a wave, several, or a quarter of one for
// the corner ops of the fused launch.
__device__ __forceinline__ void ghost_exchange_op(const GhostArgs& g, const GhostOp& op, int t, int W = 64) {
    const int mx = g.mx, my = g.my, mbc = g.mbc, meqn = g.meqn;
    const int nxp = mx + 2 * mbc, nyp = my + 2 * mbc;
    const int TI = HIPCLAW_TIME_INTERP_SLOT;
    double* qd = ((op.dst & TI) ? g.qti : g.q) + (long long) (op.dst & ~TI) * g.pstride;
    const double* qs = ((op.src & TI) ? g.qti : g.q) + (long long) (op.src & ~TI) * g.pstride;
    constexpr int U = 4;

    switch (op.type) {
    case GHOST_COPY_FACE:      // fclaw2d_clawpatch46_copy.f:40-84
    case GHOST_COPY_CORNER: {  // fclaw2d_clawpatch46_copy.f:95-133
        const bool face = op.type == GHOST_COPY_FACE;
        const int len = (op.which < 2) ? my : mx;
        const int n = face ? meqn * mbc * len : meqn * mbc * mbc;
        const SmallDiv by_field(face ? mbc * len : mbc * mbc), by_mbc(mbc);
        for (int base = t; base < n; base += W * U) {
            double v[U];
            long long di[U];
#pragma unroll
            for (int u = 0; u < U; u++) {
                const int e = base + W * u;
                di[u] = -1;
                if (e >= n) continue;
                int m, i1, j1;
                if (face) {
                    m = by_field(e);
                    const int r = e - m * mbc * len, l = by_mbc(r), bb = r - l * mbc;  // ghost layer 0..mbc-1
                    if (op.which == 0) { i1 = 1 - mbc + bb; j1 = 1 + l; }
                    else if (op.which == 1) { i1 = mx + 1 + bb; j1 = 1 + l; }
                    else if (op.which == 2) { i1 = 1 + l; j1 = 1 - mbc + bb; }
                    else { i1 = 1 + l; j1 = my + 1 + bb; }
                } else {
                    m = by_field(e);
                    const int r = e - m * mbc * mbc, l = by_mbc(r);
                    corner_cell(mx, my, op.which, l + 1, r - l * mbc + 1, i1, j1);
                }
                v[u] = qs[QIX(i1 + op.ti, j1 + op.tj, m)];
                di[u] = QIX(i1, j1, m);
            }
#pragma unroll
            for (int u = 0; u < U; u++)
                if (di[u] >= 0) qd[di[u]] = v[u];
        }
        break;
    }
    case GHOST_AVERAGE_FACE:      // fclaw2d_clawpatch46_average.f:61-174 (manifold = 0)
    case GHOST_AVERAGE_CORNER: {  // fclaw2d_clawpatch46_average.f:225-270
        const bool face = op.type == GHOST_AVERAGE_FACE;
        const int len = (op.which < 2) ? my : mx;
        const int n = face ? meqn * mbc * len : meqn * mbc * mbc;
        const SmallDiv by_field(face ? mbc * len : mbc * mbc), by_mbc(mbc);
        for (int base = t; base < n; base += W * U) {
            double v[U];
            long long di[U];
#pragma unroll
            for (int u = 0; u < U; u++) {
                const int e = base + W * u;
                di[u] = -1;
                if (e >= n) continue;
                int m, ic, jc;
                if (face) {
                    m = by_field(e);
                    const int r = e - m * mbc * len, l = by_mbc(r), bb = r - l * mbc + 1;  // ibc/jbc 1..mbc
                    if (op.which < 2) { ic = (op.which == 0) ? 1 - bb : mx + bb; jc = 1 + l; }
                    else { ic = 1 + l; jc = (op.which == 2) ? 1 - bb : my + bb; }
                } else {
                    m = by_field(e);
                    const int r = e - m * mbc * mbc, l = by_mbc(r);
                    corner_cell(mx, my, op.which, l + 1, r - l * mbc + 1, ic, jc);
                }
                const int fi = 2 * ic - 1 + op.ti, fj = 2 * jc - 1 + op.tj;
                // faces: only cells whose four children are interior to this fine grid
                if (face && (fi < 1 || fi + 1 > mx || fj < 1 || fj + 1 > my)) continue;
                double sum = 0;
                sum = sum + qs[QIX(fi, fj, m)];
                sum = sum + qs[QIX(fi + 1, fj, m)];
                sum = sum + qs[QIX(fi, fj + 1, m)];
                sum = sum + qs[QIX(fi + 1, fj + 1, m)];
                v[u] = sum / 4.0;
                di[u] = QIX(ic, jc, m);
            }
#pragma unroll
            for (int u = 0; u < U; u++)
                if (di[u] >= 0) qd[di[u]] = v[u];
        }
        break;
    }
    case GHOST_INTERP_FACE:      // fclaw2d_clawpatch46_interpolate.f:91-197; dst = fine, src = coarse
    case GHOST_INTERP_CORNER: {  // fclaw2d_clawpatch46_interpolate.f:263-311
        const bool face = op.type == GHOST_INTERP_FACE;
        const int hb = mbc / 2;
        const int n = face ? meqn * hb * mx : meqn * hb * hb;  // the reference bounds the face loop by mx
        const SmallDiv by_field(face ? hb * mx : hb * hb), by_hb(hb);
        constexpr int UI = 2;
        for (int base = t; base < n; base += W * UI) {
            double c[UI], gx[UI], gy[UI];
            long long d0[UI];
#pragma unroll
            for (int u = 0; u < UI; u++) {
                const int e = base + W * u;
                d0[u] = -1;
                if (e >= n) continue;
                int m, ic, jc;
                if (face) {
                    m = by_field(e);
                    const int r = e - m * hb * mx, l = by_hb(r), bb = r - l * hb + 1;
                    if (op.which < 2) { ic = (op.which == 0) ? bb : mx - bb + 1; jc = 1 + l; }
                    else { ic = 1 + l; jc = (op.which == 2) ? bb : my - bb + 1; }
                } else {
                    m = by_field(e);
                    const int r = e - m * hb * hb, l = by_hb(r), ibc = l + 1, jbc = r - l * hb + 1;
                    ic = (op.which & 1) ? mx - ibc + 1 : ibc;
                    jc = (op.which & 2) ? my - jbc + 1 : jbc;
                }
                const int fi = 2 * ic - 1 + op.ti, fj = 2 * jc - 1 + op.tj;
                if (face && (fi < 1 - mbc || fi + 1 > mx + mbc || fj < 1 - mbc || fj + 1 > my + mbc)) continue;
                const double cc = qs[QIX(ic, jc, m)];
                gx[u] = amr_slope(cc - qs[QIX(ic - 1, jc, m)], qs[QIX(ic + 1, jc, m)] - cc);
                gy[u] = amr_slope(cc - qs[QIX(ic, jc - 1, m)], qs[QIX(ic, jc + 1, m)] - cc);
                c[u] = cc;
                d0[u] = QIX(fi, fj, m);
            }
            // fine cells (fi..fi+1, fj..fj+1), fclaw2d_clawpatch46_interpolate.f:120-137
#pragma unroll
            for (int u = 0; u < UI; u++) {
                if (d0[u] < 0) continue;
                qd[d0[u]] = c[u] + gx[u] * -0.25 + gy[u] * -0.25;
                qd[d0[u] + 1] = c[u] + gx[u] * 0.25 + gy[u] * -0.25;
                qd[d0[u] + nxp] = c[u] + gx[u] * -0.25 + gy[u] * 0.25;
                qd[d0[u] + nxp + 1] = c[u] + gx[u] * 0.25 + gy[u] * 0.25;
            }
        }
        break;
    }
    default:
        break;
    }
}

template <int OPW>
__global__ void __launch_bounds__(64 * OPW) ghost_phase(GhostArgs g) {
    const int o = blockIdx.x * OPW + (OPW > 1 ? __builtin_amdgcn_readfirstlane(threadIdx.x >> 6) : 0);
    if (o >= g.nops) return;
    ghost_exchange_op(g, g.ops[o], threadIdx.x & 63);
}

// Physical BC of one patch per workgroup (clawpack46_bc2_default.f): faces 0
// and 1 together, then faces 2 and 3, whose strips include the corner cells
// the first two wrote.  Within a pair no element reads a cell the pair
// writes (mx, my >= 2 mbc), so all loads of a lane precede its stores.  The
// BC reads and writes cells of its own patch only, so applying it op.reps
// times in a row equals that many phases of it.
constexpr int PHYSBC_THREADS = 256;
// Every thread of the workgroup (PHYSBC_THREADS) calls this: it synchronises.
__device__ __forceinline__ void physbc_op(const GhostArgs& g, const GhostOp& op) {
    const int mx = g.mx, my = g.my, mbc = g.mbc, meqn = g.meqn;
    const int nxp = mx + 2 * mbc, nyp = my + 2 * mbc;
    const int TI = HIPCLAW_TIME_INTERP_SLOT;
    double* qd = ((op.dst & TI) ? g.qti : g.q) + (long long) (op.dst & ~TI) * g.pstride;
    constexpr int U = 4;
    const int npass = 2 * (op.reps > 1 ? op.reps : 1);
    for (int pass = 0; pass < npass; pass++) {
        const int pair = pass & 1;
        const int len = pair == 0 ? my + 2 * mbc : mx + 2 * mbc;
        const int per = meqn * mbc * len, n = 2 * per;
        const SmallDiv by_field(mbc * len), by_mbc(mbc);
        for (int base = threadIdx.x; base < n; base += PHYSBC_THREADS * U) {
            double v[U];
            long long di[U];
#pragma unroll
            for (int u = 0; u < U; u++) {
                const int e = base + PHYSBC_THREADS * u;
                di[u] = -1;
                if (e >= n) continue;
                const int face = 2 * pair + (e >= per);
                const int mth = (signed char) ((op.bc >> (8 * face)) & 0xff);
                if (mth != 1 && mth != 3) continue;
                const int f = e - (e >= per ? per : 0);
                const int m = by_field(f), r = f - m * mbc * len;
                const int l = by_mbc(r), b = r - l * mbc + 1;
                int id, jd, is, js;
                if (face < 2) {
                    jd = js = 1 - mbc + l;
                    if (face == 0) { id = 1 - b; is = (mth == 1) ? 1 : b; }
                    else { id = mx + b; is = (mth == 1) ? mx : mx + 1 - b; }
                } else {
                    id = is = 1 - mbc + l;
                    if (face == 2) { jd = 1 - b; js = (mth == 1) ? 1 : b; }
                    else { jd = my + b; js = (mth == 1) ? my : my + 1 - b; }
                }
                const int mn = (face < 2) ? 1 : 2;  // normal momentum negated on walls
                const double x = qd[QIX(is, js, m)];
                v[u] = (mth == 3 && m == mn) ? -x : x;
                di[u] = QIX(id, jd, m);
            }
#pragma unroll
            for (int u = 0; u < U; u++)
                if (di[u] >= 0) qd[di[u]] = v[u];
        }
        __syncthreads();
    }
}

__global__ void __launch_bounds__(PHYSBC_THREADS) physbc_phase(GhostArgs g) {
    const int o = blockIdx.x;
    if (o >= g.nops) return;
    physbc_op(g, g.ops[o]);
}

// One workgroup per destination patch of a phase group: the patch's
// exchange ops (one wave each, the four waves taking them in turn), then,
// once they are all written, its physical BC.  groups[b] = (first exchange
// op, end of its exchange ops, physical-BC op or -1, unused), indices into
// g.ops.  A group
// writes ghost cells of its own patch only; exchange ops read interior cells
// of other patches, or (interpolation) cells of a coarser patch that its own
// physical BC may write again with the same values (the BC is a function of
// the patch's interior and its non-physical ghost cells).
__global__ void __launch_bounds__(PHYSBC_THREADS) ghost_groups(GhostArgs g, const int4* __restrict__ groups,
                                                              int ngroups) {
    const int b = blockIdx.x;
    if (b >= ngroups) return;
    const int4 gr = groups[b];
    const int w = threadIdx.x >> 6;
    for (int o = gr.x + w; o < gr.y; o += PHYSBC_THREADS / 64) ghost_exchange_op(g, g.ops[o], threadIdx.x & 63);
    if (gr.z >= 0) {
        __syncthreads();
        physbc_op(g, g.ops[gr.z]);
    }
}

// ---------------------------------------------------------------- fused ghost fill + sync
// The fused launch lasts as long as its longest chain of dependent loads, so
// what an op reads is resolved in stages (the faces' relations, then all the
// values), and an op's elements are spread over several waves instead of being
// taken in turn (flat_waves): shock-bubble FP64 on 2,740 patches of 16 x 16 16.4
// -> 11.9 us per launch, dam break FP64 on 3,400 of 32 x 32 17.4 -> 13.8.

// A face's relation; k: the face whose ghost strip holds (i, j), -1 for an
// interior cell.
__device__ __forceinline__ int strip_of(int mx, int my, int i, int j) {
    return i < 1 ? 0 : i > mx ? 1 : j < 1 ? 2 : j > my ? 3 : -1;
}
__device__ __forceinline__ FaceRel load_rel(const FaceRel* __restrict__ frel, int slot, int k) {
    const int4* p = (const int4*) (frel + 4 * (long long) slot + (k < 0 ? 0 : k));
    const int4 a = p[0], b = p[1];
    return FaceRel{a.x, a.y, a.z, a.w, b.x, b.y, b.z, b.w};
}

// Where cell (i, j) of patch `slot` comes from as the ghost fill of this step
// leaves it, for an interior cell or a face ghost cell that is not a corner and
// not filled by interpolation (r: the relation of its strip, k): the neighbour's
// interior cell (same size), the average of the fine child's four cells
// (fclaw2d_clawpatch46_average.f:61-174, the child whose cells lie in its
// interior), or the physical BC of the patch's own interior
// (clawpack46_bc2_default.f).  All of it reads interior cells only, which no wave
// of the fused launch writes.
struct CellRef {
    const double* p;
    enum Mode { value, negated, average, zero } mode;
};
__device__ __forceinline__ CellRef cell_ref(const GhostArgs& g, const FaceRel& r, int k, int slot, int i, int j, int m) {
    const int mx = g.mx, my = g.my, mbc = g.mbc;
    const int nxp = mx + 2 * mbc, nyp = my + 2 * mbc;
    CellRef c{nullptr, CellRef::value};
    int from = slot, is = i, js = j;
    if (k >= 0) {
        if (r.rel == FREL_SAME) {
            from = r.nb0;
            is = i + r.ti0;
            js = j + r.tj0;
        } else if (r.rel == FREL_HALF) {
            c.mode = CellRef::average;
            from = r.nb0;
            is = 2 * i - 1 + r.ti0;
            js = 2 * j - 1 + r.tj0;
            if (is < 1 || is + 1 > mx || js < 1 || js + 1 > my) {
                from = r.nb1;
                is = 2 * i - 1 + r.ti1;
                js = 2 * j - 1 + r.tj1;
                // one of the two children covers every cell of the face strip
                if (is < 1 || is + 1 > mx || js < 1 || js + 1 > my) c.mode = CellRef::zero;
            }
        } else {
            // FREL_PHYS (the host admits nothing else where this is called):
            // extrapolation copies the first interior cell, a wall mirrors the strip
            // and negates the normal momentum
            const int mth = r.bc;
            if (k == 0) is = mth == 1 ? 1 : 1 - i;
            else if (k == 1) is = mth == 1 ? mx : 2 * mx + 1 - i;
            else if (k == 2) js = mth == 1 ? 1 : 1 - j;
            else js = mth == 1 ? my : 2 * my + 1 - j;
            if (mth == 3 && m == (k < 2 ? 1 : 2)) c.mode = CellRef::negated;
        }
    }
    c.p = g.q + (long long) from * g.pstride + QIX(is, js, m);
    return c;
}
__device__ __forceinline__ void cell_loads(const CellRef& c, int nxp, double v[4]) {
    v[0] = v[1] = v[2] = v[3] = 0.0;
    if (c.mode != CellRef::zero) v[0] = c.p[0];
    if (c.mode == CellRef::average) { v[1] = c.p[1]; v[2] = c.p[nxp]; v[3] = c.p[nxp + 1]; }
}
__device__ __forceinline__ double cell_value(const CellRef& c, const double v[4]) {
    if (c.mode == CellRef::average) return ((((0.0 + v[0]) + v[1]) + v[2]) + v[3]) / 4.0;
    return c.mode == CellRef::negated ? -v[0] : v[0];
}

// Interior coarse cell (ic, jc) of patch c and its slopes
// (fclaw2d_clawpatch46_interpolate.f:120-137).
__device__ __forceinline__ void coarse_cell(const GhostArgs& g, const FaceRel* __restrict__ frel, int c, int ic, int jc,
                                            int m, double& cc, double& gx, double& gy) {
    constexpr int DI[4] = {-1, 1, 0, 0}, DJ[4] = {0, 0, -1, 1};
    const int nxp = g.mx + 2 * g.mbc, nyp = g.my + 2 * g.mbc, mbc = g.mbc;
    FaceRel r[4];
    int k[4];
#pragma unroll
    for (int d = 0; d < 4; d++) {
        k[d] = strip_of(g.mx, g.my, ic + DI[d], jc + DJ[d]);
        r[d] = FaceRel{};
        if (k[d] >= 0) r[d] = load_rel(frel, c, k[d]);
    }
    cc = g.q[(long long) c * g.pstride + QIX(ic, jc, m)];
    CellRef n[4];
    double v[4][4], x[4];
#pragma unroll
    for (int d = 0; d < 4; d++) {
        n[d] = cell_ref(g, r[d], k[d], c, ic + DI[d], jc + DJ[d], m);
        cell_loads(n[d], nxp, v[d]);
    }
#pragma unroll
    for (int d = 0; d < 4; d++) x[d] = cell_value(n[d], v[d]);
    gx = amr_slope(cc - x[0], x[1] - cc);
    gy = amr_slope(cc - x[2], x[3] - cc);
}

// A cell as cell_ref's, or of a face strip that is filled by interpolation from a
// coarser patch (recomputed from the coarse patch's cells).
__device__ __forceinline__ double fused_cell(const GhostArgs& g, const FaceRel* __restrict__ frel, int slot, int i,
                                             int j, int m) {
    const int k = strip_of(g.mx, g.my, i, j);
    FaceRel r{};
    if (k >= 0) r = load_rel(frel, slot, k);
    if (k >= 0 && r.rel == FREL_DOUBLE) {
        // fine cell (i, j) = child (a, b) of coarse cell (ic, jc):
        // i = 2 ic - 1 + ti + a
        const int u = i - r.ti0 + 1, v = j - r.tj0 + 1;
        double cc, gx, gy;
        coarse_cell(g, frel, r.nb0, u >> 1, v >> 1, m, cc, gx, gy);
        return cc + gx * (u & 1 ? 0.25 : -0.25) + gy * (v & 1 ? 0.25 : -0.25);
    }
    const CellRef c = cell_ref(g, r, k, slot, i, j, m);
    double v[4];
    cell_loads(c, g.mx + 2 * g.mbc, v);
    return cell_value(c, v);
}

// Interpolation op (dst = fine, src = coarse) as in ghost_exchange_op, its
// coarse-side reads resolved by cell_ref.
__device__ __forceinline__ void fused_interp_op(const GhostArgs& g, const FaceRel* __restrict__ frel, const GhostOp& op,
                                                int t, int W) {
    const int mx = g.mx, my = g.my, mbc = g.mbc, meqn = g.meqn;
    const int nxp = mx + 2 * mbc, nyp = my + 2 * mbc;
    double* qd = g.q + (long long) op.dst * g.pstride;
    const bool face = op.type == GHOST_INTERP_FACE;
    const int hb = mbc / 2;
    const int n = face ? meqn * hb * mx : meqn * hb * hb;
    const SmallDiv by_field(face ? hb * mx : hb * hb), by_hb(hb);
    for (int e = t; e < n; e += W) {
        int m, ic, jc;
        if (face) {
            m = by_field(e);
            const int r = e - m * hb * mx, l = by_hb(r), bb = r - l * hb + 1;
            if (op.which < 2) { ic = (op.which == 0) ? bb : mx - bb + 1; jc = 1 + l; }
            else { ic = 1 + l; jc = (op.which == 2) ? bb : my - bb + 1; }
        } else {
            m = by_field(e);
            const int r = e - m * hb * hb, l = by_hb(r), ibc = l + 1, jbc = r - l * hb + 1;
            ic = (op.which & 1) ? mx - ibc + 1 : ibc;
            jc = (op.which & 2) ? my - jbc + 1 : jbc;
        }
        const int fi = 2 * ic - 1 + op.ti, fj = 2 * jc - 1 + op.tj;
        if (face && (fi < 1 - mbc || fi + 1 > mx + mbc || fj < 1 - mbc || fj + 1 > my + mbc)) continue;
        double cc, gx, gy;
        coarse_cell(g, frel, op.src, ic, jc, m, cc, gx, gy);
        const long long d0 = QIX(fi, fj, m);
        qd[d0] = cc + gx * -0.25 + gy * -0.25;
        qd[d0 + 1] = cc + gx * 0.25 + gy * -0.25;
        qd[d0 + nxp] = cc + gx * -0.25 + gy * 0.25;
        qd[d0 + nxp + 1] = cc + gx * 0.25 + gy * 0.25;
    }
}

// Physical BC of one patch (clawpack46_bc2_default.f), each ghost
// cell written once with its final value: the sources are interior cells or
// ghost cells of a neighbouring face strip, recomputed through fused_cell, and
// a corner both of whose faces are physical takes the y-face's value (the
// reference applies faces 2 and 3 after faces 0 and 1).
__device__ __forceinline__ void fused_physbc_op(const GhostArgs& g, const FaceRel* __restrict__ frel, const GhostOp& op, int t,
                                                int W) {
    const int mx = g.mx, my = g.my, mbc = g.mbc, meqn = g.meqn;
    const int nxp = mx + 2 * mbc, nyp = my + 2 * mbc;
    double* qd = g.q + (long long) op.dst * g.pstride;
    auto code = [&](int f) { return (int) (signed char) ((op.bc >> (8 * f)) & 0xff); };
    const bool phys[4] = {code(0) == 1 || code(0) == 3, code(1) == 1 || code(1) == 3,
                          code(2) == 1 || code(2) == 3, code(3) == 1 || code(3) == 3};
    for (int face = 0; face < 4; face++) {
        if (!phys[face]) continue;
        const int mth = code(face);
        const int len = face < 2 ? my + 2 * mbc : mx + 2 * mbc;
        const int n = meqn * mbc * len;
        const SmallDiv by_field(mbc * len), by_mbc(mbc);
        for (int e = t; e < n; e += W) {
            const int m = by_field(e), r = e - m * mbc * len;
            const int l = by_mbc(r), b = r - l * mbc + 1;
            int id, jd, is, js;
            if (face < 2) {
                jd = js = 1 - mbc + l;
                // the corners of two physical faces are the y-face's
                if ((jd < 1 && phys[2]) || (jd > my && phys[3])) continue;
                if (face == 0) { id = 1 - b; is = (mth == 1) ? 1 : b; }
                else { id = mx + b; is = (mth == 1) ? mx : mx + 1 - b; }
            } else {
                id = is = 1 - mbc + l;
                if (face == 2) { jd = 1 - b; js = (mth == 1) ? 1 : b; }
                else { jd = my + b; js = (mth == 1) ? my : my + 1 - b; }
            }
            const int mn = (face < 2) ? 1 : 2;  // normal momentum negated on walls
            const double x = fused_cell(g, frel, op.dst, is, js, m);
            qd[QIX(id, jd, m)] = (mth == 3 && m == mn) ? -x : x;
        }
    }
}

// Time-sync increments (as time_sync_cells): a same-size op writes every
// position of its face, a coarse/fine op the positions its fine patch covers
// (the other child's op writes the rest; the reference adds zero for the
// positions a child does not cover).  A wave takes the positions of `ops`
// consecutive ops, up to SYNC_ITEMS per lane, in two stages of loads: the ops,
// then sizes and registers.  An op at a time is a chain of memory latencies for
// little more than one load per lane (whole launch, dam break FP32 on 11,296
// patches of 32 x 32, items 1, 2, 3, 4: 37, 35, 32, 35 us, of which the
// registers' and increments' 70 MB need 14; ensemble of 64 runs 61, 62, 58, 66).
constexpr int SYNC_ITEMS = 3;
__device__ void fused_sync_ops(const FlatArgs& f, int op0, int ops, int t) {
    const int mx = f.g.mx, meqn = f.g.meqn, per = meqn * mx;
    const int n = min(ops, f.nsync - op0) * per;
    const int kout = f.fluxreg ? REG_EFIN : REG_EFOUT;
    const SmallDiv by_per(per), by_mx(mx);
    for (int base = t; base < n; base += 64 * SYNC_ITEMS) {
        int type[SYNC_ITEMS], dst[SYNC_ITEMS], src[SYNC_ITEMS], face[SYNC_ITEMS], m[SYNC_ITEMS], c[SYNC_ITEMS], f0[SYNC_ITEMS];
        bool on[SYNC_ITEMS];
        int4 lo[SYNC_ITEMS];
        int2 hi[SYNC_ITEMS];
#pragma unroll
        for (int u = 0; u < SYNC_ITEMS; u++) {
            const int e = min(base + 64 * u, n - 1);
            const int o = by_per(e), r = e - o * per;
            m[u] = by_mx(r);
            c[u] = r - m[u] * mx;
            const int* op = f.sops + 8 * (long long) (op0 + o);
            lo[u] = *(const int4*) op;
            hi[u] = *(const int2*) (op + 4);
        }
        double ein[SYNC_ITEMS], ft[SYNC_ITEMS], ef[SYNC_ITEMS], ef2[SYNC_ITEMS], fn[SYNC_ITEMS], fn2[SYNC_ITEMS];
        double area[SYNC_ITEMS], area_src[SYNC_ITEMS];
#pragma unroll
        for (int u = 0; u < SYNC_ITEMS; u++) {
            type[u] = lo[u].x; dst[u] = lo[u].y; src[u] = lo[u].z; face[u] = lo[u].w;
            const bool f2c = type[u] == SYNC_F2C;
            f0[u] = f2c ? 2 * c[u] + (face[u] < 2 ? hi[u].y : hi[u].x) : c[u];   // 0-based position on src
            on[u] = base + 64 * u < n && (!f2c || (f0[u] >= 0 && f0[u] + 1 < mx));
            ein[u] = ft[u] = ef[u] = ef2[u] = fn[u] = fn2[u] = 0.0;
            area[u] = area_src[u] = 1.0;
            if (on[u]) {
                const int kfl = (face[u] == 0 || face[u] == 2) ? REG_FP : REG_FM;
                const double* __restrict__ rt = f.reg + (long long) dst[u] * f.rstride + (face[u] * 4 * meqn + m[u]) * mx + c[u];
                const double* __restrict__ rn = f.reg + (long long) src[u] * f.rstride + ((face[u] ^ 1) * 4 * meqn + m[u]) * mx + f0[u];
                area[u] = f.dxs[dst[u]] * f.dys[dst[u]];
                ein[u] = rt[REG_EFIN * per];
                ef[u] = rn[kout * per];
                if (f2c) ef2[u] = rn[kout * per + 1];
                if (!f.fluxreg) {
                    ft[u] = rt[kfl * per];
                    fn[u] = rn[kfl * per];
                    if (f2c) fn2[u] = rn[kfl * per + 1];
                }
                if (type[u] == SYNC_SAMESIZE_PAIR) area_src[u] = f.dxs[src[u]] * f.dys[src[u]];
            }
        }
#pragma unroll
        for (int u = 0; u < SYNC_ITEMS; u++) {
            if (!on[u]) continue;
            const bool f2c = type[u] == SYNC_F2C;
            if (f2c) { ef[u] = ef[u] + ef2[u]; fn[u] = fn[u] + fn2[u]; }
            const double delta = (face[u] == 0 || face[u] == 2) ? (ef[u] - ein[u]) - (fn[u] - ft[u])
                                                                : (ein[u] - ef[u]) - (fn[u] - ft[u]);
            const double v = (f2c ? delta : 0.5 * delta) / area[u];
            const int pos = m[u] * mx + c[u];
            f.qinc[(long long) dst[u] * f.cstride + face[u] * per + pos] = 0.0 + v;
            // the partner's op (dst and src swapped, face ^ 1) would compute the
            // same delta: it reads these two registers and takes their
            // difference in the same order (the FP32 flux form stores no
            // fluctuations, fn = ft = 0)
            if (type[u] == SYNC_SAMESIZE_PAIR)
                f.qinc[(long long) src[u] * f.cstride + (face[u] ^ 1) * per + pos] = 0.0 + 0.5 * delta / area_src[u];
        }
    }
}

// The fused launch, no op depending on another: ghost ops (copies and
// averages read interior cells; interpolations and physical BCs recompute the
// ghost cells they read), then time-sync increments.  A face or physical-BC op
// takes a wave or several; the corner ops, a few cells each, take a quarter of
// one.  The interior cells keep their values before the time sync, which
// every ghost op reads (the reference fills ghost cells before it
// synchronises, src/fclaw2d_advance.c:330-341); the next update adds the
// increments to the cells it stages.
constexpr int FLAT_OPW = 4;           // waves per workgroup
constexpr int FLAT_CORNER_LANES = 16; // lanes of one corner op
constexpr int FLAT_CORNERS = 64 / FLAT_CORNER_LANES;

// Waves of one op, so that no lane takes two elements in turn whose chains are
// long: a physical BC's are the ghost cells of a face, an interpolation's its
// coarse cells (copies and averages load several elements at once anyway, and
// waves without work are not free: ensemble of 64 runs, 22,436 patches of 16 x 16,
// 58 us with two waves for every op, 56 with one).
static int flat_waves(int n) { return std::min(4, (n + 63) / 64); }
__host__ __device__ __forceinline__ int flat_corner_waves(int n) { return (n + FLAT_CORNERS - 1) / FLAT_CORNERS; }
// Time-sync ops of one wave, per positions each: as many as its lanes take at once.
__host__ __device__ __forceinline__ int flat_sync_ops(int per) {
    return per < 64 * SYNC_ITEMS ? 64 * SYNC_ITEMS / per : 1;
}

__global__ void __launch_bounds__(64 * FLAT_OPW) ghost_flat(FlatArgs f) {
    int w = blockIdx.x * FLAT_OPW + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int lane = threadIdx.x & 63;
    if (w < f.nphys * f.phys_parts) {
        const int o = w / f.phys_parts, t = (w - o * f.phys_parts) * 64 + lane;
        fused_physbc_op(f.g, f.frel, f.g.ops[f.ncorner0 + f.phys0 + o], t, 64 * f.phys_parts);
        return;
    }
    w -= f.nphys * f.phys_parts;
    if (w < (f.nbig - f.nphys) * f.parts) {
        const int k = w / f.parts, t = (w - k * f.parts) * 64 + lane, W = 64 * f.parts;
        const GhostOp op = f.g.ops[f.ncorner0 + k + (k < f.phys0 ? 0 : f.nphys)];
        if (op.type == GHOST_INTERP_FACE || op.type == GHOST_INTERP_CORNER) fused_interp_op(f.g, f.frel, op, t, W);
        else ghost_exchange_op(f.g, op, t, W);
        return;
    }
    w -= (f.nbig - f.nphys) * f.parts;
    const int nw0 = flat_corner_waves(f.ncorner0), nw1 = flat_corner_waves(f.ncorner1);
    if (w < nw0 + nw1) {
        // corner ops [0, ncorner0) and [ncorner0 + nbig, ... + ncorner1)
        const bool first = w < nw0;
        const int k = (first ? w : w - nw0) * FLAT_CORNERS + lane / FLAT_CORNER_LANES;
        if (k < (first ? f.ncorner0 : f.ncorner1)) {
            const GhostOp op = f.g.ops[(first ? 0 : f.ncorner0 + f.nbig) + k];
            const int t = lane % FLAT_CORNER_LANES;
            if (op.type == GHOST_INTERP_CORNER) fused_interp_op(f.g, f.frel, op, t, FLAT_CORNER_LANES);
            else ghost_exchange_op(f.g, op, t, FLAT_CORNER_LANES);
        }
        return;
    }
    w -= nw0 + nw1;
    const int ops = flat_sync_ops(f.g.meqn * f.g.mx);
    if (w * ops < f.nsync) fused_sync_ops(f, w * ops, ops, lane);
}

// The pending increments added into the slab (after the last step of an
// advance, so the state is the synchronised one), one workgroup per patch listed
// in slots (those with a corrected face), in the update's
// order: a corner cell belongs to its x-face when that face is
// corrected, and takes both faces' increments in the reference's order.
__global__ void apply_qcorr(double* __restrict__ q, const double* __restrict__ qcorr,
                            const int* __restrict__ cmask, const int* __restrict__ slots,
                            long long pstride, long long cstride, int mx, int my, int mbc, int meqn) {
    const int slot = slots[blockIdx.x], mask = cmask[slot];
    const SmallDiv by_face(meqn * mx), by_mx(mx);
    const int nxp = mx + 2 * mbc, nyp = my + 2 * mbc;
    const double* qc = qcorr + (long long) slot * cstride;
    for (int r = threadIdx.x; r < 4 * meqn * mx; r += blockDim.x) {
        const int fc = by_face(r), r2 = r - fc * meqn * mx, m = by_mx(r2), c = r2 - m * mx + 1;
        if (!((mask >> fc) & 1)) continue;
        const int len = fc < 2 ? my : mx;
        const int other = (c == 1 || c == len) ? (fc < 2 ? (c == 1 ? 2 : 3) : (c == 1 ? 0 : 1)) : -1;
        const bool other_on = other >= 0 && ((mask >> other) & 1);
        if (fc >= 2 && other_on) continue;
        const int i = fc == 0 ? 1 : fc == 1 ? mx : c, j = fc == 2 ? 1 : fc == 3 ? my : c;
        const double v = qc[(fc * meqn + m) * len + c - 1];
        double* cell = q + (long long) slot * pstride + QIX(i, j, m);
        double x = *cell;
        if (other_on) {
            const double w = qc[(other * meqn + m) * mx + (fc == 0 ? 0 : mx - 1)];
            if (sync_y_first(mask, fc, other)) { x = x + w; x = x + v; }
            else { x = x + v; x = x + w; }
        } else {
            x = x + v;
        }
        *cell = x;
    }
}

int launch_ghost_flat(const FlatArgs& args, hipStream_t st) {
    FlatArgs f = args;
    const int side = std::max(f.g.mx, f.g.my);
    f.parts = flat_waves(f.g.meqn * (f.g.mbc / 2) * side);
    f.phys_parts = flat_waves(f.g.meqn * f.g.mbc * (side + 2 * f.g.mbc));
    const int ops = flat_sync_ops(f.g.meqn * f.g.mx);
    const int n = f.nphys * f.phys_parts + (f.nbig - f.nphys) * f.parts + flat_corner_waves(f.ncorner0) + flat_corner_waves(f.ncorner1) + (f.nsync + ops - 1) / ops;
    if (n <= 0) return 0;
    hipLaunchKernelGGL(ghost_flat, dim3((n + FLAT_OPW - 1) / FLAT_OPW), dim3(64 * FLAT_OPW), 0, st, f);
    return (int) hipGetLastError();
}

int launch_apply_qcorr(double* q, const double* qcorr, const int* cmask, const int* slots, int n,
                       long long pstride, long long cstride, int mx, int my, int mbc, int meqn,
                       hipStream_t st) {
    if (n <= 0) return 0;
    hipLaunchKernelGGL(apply_qcorr, dim3(n), dim3(256), 0, st, q, qcorr, cmask,
                       slots, pstride, cstride, mx, my, mbc, meqn);
    return (int) hipGetLastError();
}

__global__ void reset_cfl(unsigned long long* p, unsigned long long* sum) {
    unsigned long long* w = p + (long long) blockIdx.x * CFL_BLOCK + threadIdx.x * CFL_STRIDE;
    w[0] = w[1] = w[2] = 0ull;
    if (sum && blockIdx.x == 0 && threadIdx.x < STEP_SUMS) sum[threadIdx.x] = 0ull;
}

// The end of an advance, in one launch: its Courant number and the steps'
// execution times straight into host memory, and the words cleared for the next
// one.  16 threads per step.  (A loop that takes one step per call and looks at
// the Courant number, 256 patches of 16 x 16: 61 us per call with a reset
// before, events around the step and a copy after, 27 us this way.)
__global__ void __launch_bounds__(CFL_WORDS * STEP_BLOCKS)
collect_steps(unsigned long long* __restrict__ c, int blocks, unsigned long long* __restrict__ sum,
              unsigned long long* __restrict__ out) {
    __shared__ unsigned long long s_cfl[STEP_BLOCKS], s_ticks[STEP_BLOCKS];
    const int n = threadIdx.x / CFL_WORDS, k = threadIdx.x % CFL_WORDS;
    unsigned long long v = 0, e = 0, begin = 0;
    if (n < blocks) {
        unsigned long long* w = c + n * CFL_BLOCK + k * CFL_STRIDE;
        v = w[0];
        e = w[1];
        begin = w[2];
        w[0] = w[1] = w[2] = 0ull;
    }
#pragma unroll
    for (int off = CFL_WORDS / 2; off >= 1; off >>= 1) {
        const unsigned long long v2 = __shfl_xor(v, off, 64), e2 = __shfl_xor(e, off, 64);
        v = v2 > v ? v2 : v;
        e = e2 > e ? e2 : e;
    }
    if (k == 0) {
        s_cfl[n] = v;
        s_ticks[n] = begin && e > begin ? e - begin : 0ull;
    }
    __syncthreads();
    if (threadIdx.x != 0) return;
    unsigned long long most = sum[0], ticks = sum[1], steps = sum[2];
    const unsigned long long first = sum[3] ? sum[3] : begin;
    for (int i = 0; i < blocks; i++) {
        most = s_cfl[i] > most ? s_cfl[i] : most;
        ticks += s_ticks[i];
        steps += s_ticks[i] != 0;
    }
    if (out) {
        out[0] = most; out[1] = ticks; out[2] = steps; out[3] = first;
        out[4] = __builtin_amdgcn_s_memrealtime();
        most = ticks = steps = 0;
    }
    sum[0] = most; sum[1] = ticks; sum[2] = steps; sum[3] = out ? 0ull : first;
}

// ---------------------------------------------------------------- regrid
// Gradient criterion of the reference's tag4refinement / tag4coarsening
// (src/patches/clawpatch/fort_4.6/fclaw2d_clawpatch46_tag4refinement.f,
// src/patches/clawpatch/fort_user/fclaw2d_clawpatch_gradient_exceeds_th.f90,
// unmapped): does some interior cell have |(dq/dx, dq/dy, 0)| above the
// threshold?  out[2w] for the refine threshold, out[2w+1] for the coarsen
// threshold (a negative refine threshold or a coarsen threshold <= 0 always
// counts as exceeded: always refine, never coarsen, as
// src/patches/clawpatch/fclaw2d_clawpatch.cpp:813-817, 890-911 decide).
//
// The square of the gradient from two reciprocals decides every cell that is not
// within 1e-13 (relative) of a threshold's square; only where some lane's is does
// the wave take the reference's divisions and square root, which cost more than
// reading the patch (11,296 patches of 32 x 32: 51 us with them in every cell, 34
// us without; one field is 117 MB, 23 us).
struct TagThreshold {
    double thr, lo, hi;   // the square of a gradient above hi exceeds thr, below lo does not
};
static TagThreshold tag_threshold(double thr, bool always) {
    if (always) return {thr, -1.0, -1.0};
    if (thr > 1e-140 && thr < 1e140) return {thr, thr * thr * (1.0 - 1e-13), thr * thr * (1.0 + 1e-13)};
    return {thr, -1.0, __builtin_inf()};
}
__global__ void __launch_bounds__(256)
tag_patches(const double* __restrict__ q, const int* __restrict__ slots, int n,
            const double* __restrict__ dxs, const double* __restrict__ dys, long long pstride,
            int mx, int my, int mbc, int ivar, TagThreshold refine, TagThreshold coarsen, int2* __restrict__ out) {
    const int w = blockIdx.x;
    if (w >= n) return;
    const int slot = slots[w];
    const int nxp = mx + 2 * mbc, nyp = my + 2 * mbc;
    const double* qp = q + (long long) slot * pstride + QIX(1, 1, ivar);
    const double dx2 = 2 * dxs[slot], dy2 = 2 * dys[slot];
    const double rx = 1.0 / dx2, ry = 1.0 / dy2;
    const SmallDiv by_mx(mx);
    int er = 0, ec = 0;
    constexpr int U = 4;
    for (int base = threadIdx.x; base < mx * my; base += 256 * U) {
        double x[U], y[U];
#pragma unroll
        for (int u = 0; u < U; u++) {
            const int e = min(base + 256 * u, mx * my - 1);
            const int j = by_mx(e);
            const double* c = qp + (long long) j * nxp + (e - j * mx);
            x[u] = c[1] - c[-1];
            y[u] = c[nxp] - c[-nxp];
        }
#pragma unroll
        for (int u = 0; u < U; u++) {
            const double ax = x[u] * rx, ay = y[u] * ry, s = ax * ax + ay * ay;
            if ((s > refine.hi || s < refine.lo) && (s > coarsen.hi || s < coarsen.lo)) {
                er |= s > refine.hi;
                ec |= s > coarsen.hi;
            } else {
                const double dqx = x[u] / dx2, dqy = y[u] / dy2, g3 = 0.0;
                const double ds = sqrt(dqx * dqx + dqy * dqy + g3 * g3);
                er |= ds > refine.thr;
                ec |= ds > coarsen.thr;
            }
        }
    }
    er = __syncthreads_or(er);
    ec = __syncthreads_or(ec);
    if (threadIdx.x == 0) out[w] = make_int2(refine.thr < 0 ? 1 : er, coarsen.thr <= 0 ? 1 : ec);
}

// Repopulate one new patch (cb_fclaw2d_regrid_repopulate,
// src/fclaw2d_regrid.c:95-230): copy of the same old patch, interpolation from
// the old parent (fclaw2d_clawpatch46_fort_interpolate2fine, over the
// reference's loop ranges), or average of the four old children
// (fclaw2d_clawpatch46_fort_average2coarse).  op = (kind, dst, src0..src3, -, -).
__global__ void __launch_bounds__(256)
regrid_remap(const double* __restrict__ qold, double* __restrict__ qnew,
             const int* __restrict__ ops, int nops, long long pstride, int mx, int my, int mbc,
             int meqn) {
    const int o = blockIdx.x;
    if (o >= nops) return;
    const int* op = ops + 8 * o;
    const int kind = op[0];
    const int nxp = mx + 2 * mbc, nyp = my + 2 * mbc;
    double* qd = qnew + (long long) op[1] * pstride;
    if (kind == REGRID_SAME) {
        const double* qs = qold + (long long) op[2] * pstride;
        for (long long e = threadIdx.x; e < pstride; e += blockDim.x) qd[e] = qs[e];
    } else {
        // the cells the transfer does not write (ghost cells of new children
        // and parents) start at zero until the ghost fill
        for (long long e = threadIdx.x; e < pstride; e += blockDim.x) qd[e] = 0.0;
        __syncthreads();
    }
    if (kind == REGRID_CHILD) {
        const double* qc = qold + (long long) op[2] * pstride;
        const int igrid = op[3], ig = igrid % 2, jg = (igrid - ig) / 2;
        const int i1 = 1 - ig, ni = mx / 2 + 1, ic_add = ig * mx / 2;
        const int j1 = 1 - jg, nj = my / 2 + 1, jc_add = jg * my / 2;
        for (int e = threadIdx.x; e < meqn * ni * nj; e += blockDim.x) {
            const int m = e / (ni * nj), r = e - m * ni * nj;
            const int j = j1 + r / ni, i = i1 + r % ni;
            const int ic = i + ic_add, jc = j + jc_add;
            const double c = qc[QIX(ic, jc, m)];
            const double gradx = amr_slope(c - qc[QIX(ic - 1, jc, m)], qc[QIX(ic + 1, jc, m)] - c);
            const double grady = amr_slope(c - qc[QIX(ic, jc - 1, m)], qc[QIX(ic, jc + 1, m)] - c);
            for (int ii = 1; ii <= 2; ii++)
                for (int jj = 1; jj <= 2; jj++) {
                    const double shiftx = (ii - 2 / 2.0 - 0.5) / 2;
                    const double shifty = (jj - 2 / 2.0 - 0.5) / 2;
                    qd[QIX((i - 1) * 2 + ii, (j - 1) * 2 + jj, m)] = c + shiftx * gradx + shifty * grady;
                }
        }
    } else if (kind != REGRID_SAME) {
        for (int e = threadIdx.x; e < meqn * mx * my; e += blockDim.x) {
            const int m = e / (mx * my), r = e - m * mx * my;
            const int jc = r / mx + 1, ic = r - (jc - 1) * mx + 1;
            const int ig = ic > mx / 2, jg = jc > my / 2, g = ig + 2 * jg;
            const double* qf = qold + (long long) op[2 + g] * pstride;
            const int i = ic - ig * mx / 2, j = jc - jg * mx / 2;  // mx, as the reference writes it
            double sum = 0;
            sum = sum + qf[QIX(2 * i - 1, 2 * j - 1, m)];
            sum = sum + qf[QIX(2 * i, 2 * j - 1, m)];
            sum = sum + qf[QIX(2 * i - 1, 2 * j, m)];
            sum = sum + qf[QIX(2 * i, 2 * j, m)];
            qd[QIX(ic, jc, m)] = sum / 4;
        }
    }
}

// A workgroup per COPY_CHUNK values of a patch, then four zeroed registers (slot, face)
// per workgroup: both only move memory, and a launch of its own for either lasts 5 us
// at least (a subcycled dam break's 1,480 fine patches of 16 x 16: copy 9.6 and reset
// 8.0 us apart, 10.8 us together).  Not one workgroup per patch, which copies a large
// one alone (hipclaw_step_batch of a subcycling state, one patch of 256 x 256: 143 us,
// 37 in chunks; 64 x 64 42 and 36, 16 x 16, which is one chunk, 31).
constexpr int COPY_CHUNK = 1024;
template <typename V>
__global__ void __launch_bounds__(256)
copy_patches(const V* __restrict__ src, V* __restrict__ dst, const int* __restrict__ slots, int n, int chunks, int pstride,
             double* __restrict__ reg, const int* __restrict__ resets, int nresets, long long rstride, int per_face) {
    const int b = blockIdx.x;
    if (b < n * chunks) {
        const int w = b / chunks, e0 = (b - w * chunks) * COPY_CHUNK + threadIdx.x;
        const long long base = (long long) slots[w] * pstride;
        V v[COPY_CHUNK / 256];
#pragma unroll
        for (int u = 0; u < COPY_CHUNK / 256; u++) v[u] = src[base + min(e0 + 256 * u, pstride - 1)];
#pragma unroll
        for (int u = 0; u < COPY_CHUNK / 256; u++)
            if (e0 + 256 * u < pstride) dst[base + e0 + 256 * u] = v[u];
        return;
    }
    const int r = (b - n * chunks) * 4 + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    if (r >= nresets) return;
    double* p = reg + (long long) resets[2 * r] * rstride + (long long) resets[2 * r + 1] * per_face;
    for (int e = threadIdx.x & 63; e < per_face; e += 64) p[e] = 0.0;
}

// fclaw2d_clawpatch46_fort_timeinterp
// (src/patches/clawpatch/fort_4.6/fclaw2d_clawpatch46_timeinterp.f:1-58):
// qinterp = qlast + alpha (qcurr - qlast) on the interior cells within mbc of
// the patch edge (the cells fine neighbours interpolate from).
__global__ void timeinterp_band(const double* __restrict__ q, const double* __restrict__ ql,
                                double* __restrict__ qi, const int* __restrict__ slots, int n,
                                long long pstride, int mx, int my, int mbc, int meqn,
                                double alpha) {
    const int w = blockIdx.y;
    if (w >= n) return;
    const long long base = (long long) slots[w] * pstride;
    const int nxp = mx + 2 * mbc, nyp = my + 2 * mbc;
    for (int e = blockIdx.x * blockDim.x + threadIdx.x; e < meqn * mx * my; e += gridDim.x * blockDim.x) {
        const int m = e / (mx * my), r = e - m * mx * my;
        const int j = r / mx + 1, i = r - (j - 1) * mx + 1;
        if (i > mbc && i <= mx - mbc && j > mbc && j <= my - mbc) continue;  // the hole
        const long long o = base + QIX(i, j, m);
        qi[o] = ql[o] + alpha * (q[o] - ql[o]);
    }
}

__global__ void copy_interior(const double* __restrict__ src, double* __restrict__ dst,
                              const int* __restrict__ slots, int n, long long pstride,
                              int mx, int my, int mbc, int meqn) {
    const int w = blockIdx.y;
    if (w >= n) return;
    const long long base = (long long) slots[w] * pstride;
    const int nxp = mx + 2 * mbc, nyp = my + 2 * mbc;
    for (int e = blockIdx.x * blockDim.x + threadIdx.x; e < meqn * mx * my;
         e += gridDim.x * blockDim.x) {
        const int m = e / (mx * my), r = e - m * mx * my;
        const int j = r / mx + 1, i = r - (j - 1) * mx + 1;
        dst[base + QIX(i, j, m)] = src[base + QIX(i, j, m)];
    }
}

// Error-free transformation a + b = s + e (Knuth TwoSum).
__device__ __forceinline__ void two_sum(double a, double b, double& s, double& e) {
    s = a + b;
    const double bb = s - a;
    e = (a - (s - bb)) + (b - bb);
}

// Compensated sums of q*dx*dy over the interior cells of all patches: each thread
// of a fixed number of workgroups keeps a double-double accumulator over the
// patches its workgroup takes, and combines it with the others' by TwoSum at the
// end; a second launch adds the workgroups'.  (Per patch and with the patches
// added on the host: 76 us of kernel and some 80 on the host for 11,296 patches
// of 32 x 32; in two launches 59 us, of which reading the interior's 278 MB is 55.)
constexpr int MASS_GROUPS = 2048;

// The workgroup's sum of its 256 threads' accumulators, in thread 0.
__device__ __forceinline__ void sum_group(double& hi, double& lo, double (*sh)[4]) {
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1) {
        double s, err;
        two_sum(hi, __shfl_xor(hi, off, 64), s, err);
        hi = s;
        lo = lo + __shfl_xor(lo, off, 64) + err;
    }
    if ((threadIdx.x & 63) == 0) { sh[0][threadIdx.x >> 6] = hi; sh[1][threadIdx.x >> 6] = lo; }
    __syncthreads();
    for (int w = 1; w < 4 && threadIdx.x == 0; w++) {
        double s, err;
        two_sum(hi, sh[0][w], s, err);
        hi = s;
        lo = lo + sh[1][w] + err;
    }
    __syncthreads();
}

__global__ void __launch_bounds__(256)
mass_groups(const double* __restrict__ q, const int* __restrict__ slots, int n,
            const double* __restrict__ dxs, const double* __restrict__ dys, long long pstride,
            int mx, int my, int mbc, int meqn, double* __restrict__ out) {
    __shared__ double sh[2][4];
    const int nxp = mx + 2 * mbc, nyp = my + 2 * mbc, cells = mx * my;
    const SmallDiv by_mx(mx);
    constexpr int U = 4;
    for (int m = 0; m < meqn; m++) {
        double hi = 0.0, lo = 0.0;
        for (int w = blockIdx.x; w < n; w += gridDim.x) {
            const int slot = slots[w];
            const double area = dxs[slot] * dys[slot];
            const double* qp = q + (long long) slot * pstride + QIX(1, 1, m);
            for (int base = threadIdx.x; base < cells; base += 256 * U) {
                double v[U];
#pragma unroll
                for (int u = 0; u < U; u++) {
                    const int e = min(base + 256 * u, cells - 1), j = by_mx(e);
                    v[u] = qp[(long long) j * nxp + (e - j * mx)];
                }
#pragma unroll
                for (int u = 0; u < U; u++) {
                    if (base + 256 * u >= cells) continue;
                    double s, err;
                    two_sum(hi, v[u] * area, s, err);
                    hi = s;
                    lo += err;
                }
            }
        }
        sum_group(hi, lo, sh);
        if (threadIdx.x == 0) {
            out[2 * (blockIdx.x * meqn + m)] = hi;
            out[2 * (blockIdx.x * meqn + m) + 1] = lo;
        }
    }
}

// One workgroup per field; out: host memory.
__global__ void __launch_bounds__(256)
mass_total(const double* __restrict__ parts, int groups, int meqn, double* __restrict__ out) {
    __shared__ double sh[2][4];
    const int m = blockIdx.x;
    double hi = 0.0, lo = 0.0;
    for (int b = threadIdx.x; b < groups; b += 256) {
        double s, err;
        two_sum(hi, parts[2 * (b * meqn + m)], s, err);
        hi = s;
        lo += err + parts[2 * (b * meqn + m) + 1];
    }
    sum_group(hi, lo, sh);
    if (threadIdx.x == 0) two_sum(hi, lo, out[2 * m], out[2 * m + 1]);
}

int launch_ghost_exchange(const GhostArgs& g, hipStream_t st) {
    if (g.nops <= 0) return 0;
    hipLaunchKernelGGL(ghost_phase<4>, dim3((g.nops + 3) / 4), dim3(256), 0, st, g);
    return (int) hipGetLastError();
}

int launch_ghost_groups(const GhostArgs& g, const int4* groups, int ngroups, hipStream_t st) {
    if (ngroups <= 0) return 0;
    hipLaunchKernelGGL(ghost_groups, dim3(ngroups), dim3(PHYSBC_THREADS), 0, st, g, groups, ngroups);
    return (int) hipGetLastError();
}

int launch_ghost_physbc(const GhostArgs& g, hipStream_t st) {
    if (g.nops <= 0) return 0;
    hipLaunchKernelGGL(physbc_phase, dim3(g.nops), dim3(PHYSBC_THREADS), 0, st, g);
    return (int) hipGetLastError();
}

int launch_copy_patches(const double* src, double* dst, const int* slots, int n, long long pstride, const Resets& z,
                        hipStream_t st) {
    const bool pairs = pstride % 2 == 0;
    const int values = (int) (pairs ? pstride / 2 : pstride), chunks = (values + COPY_CHUNK - 1) / COPY_CHUNK;
    const long long blocks = (long long) n * chunks + (z.n + 3) / 4;
    if (blocks <= 0) return 0;
    if (blocks > 0x7fffffffLL) return (int) hipErrorInvalidConfiguration;
    if (pairs)
        hipLaunchKernelGGL(copy_patches<double2>, dim3((unsigned) blocks), dim3(256), 0, st, (const double2*) src,
                           (double2*) dst, slots, n, chunks, values, z.reg, z.list, z.n, z.rstride, z.per_face);
    else
        hipLaunchKernelGGL(copy_patches<double>, dim3((unsigned) blocks), dim3(256), 0, st, src, dst, slots, n, chunks,
                           values, z.reg, z.list, z.n, z.rstride, z.per_face);
    return (int) hipGetLastError();
}

// Ghost-patch message of each listed slot (the data a rank sends another for
// a patch bordering it): the q band of mbc ghost and refratio*mbc interior
// layers in the order of fclaw2d_clawpatch46_fort_local_ghost_pack
// (src/patches/clawpatch/fort_4.6/fclaw2d_clawpatch46_local_ghost_pack.f:38-84),
// then, with time sync, the registers in the order of fclaw2d_clawpatch_time_sync_pack_registers
// (src/patches/clawpatch/fclaw2d_clawpatch_conservation.c:112-195): per face
// meqn*len quadruples (fm, fp, edge flux 0, edge flux 1), then len pairs
// (edge length, area).  unpack = 1 writes q and the registers back (edge
// lengths and areas follow from dx, dy and are not read).
//
// A thread takes MESSAGE_ITEMS values, all loaded before they are stored, and
// finds their places by arithmetic: looking them up in a table is one more memory
// latency in a launch that lasts a few of them.
constexpr int MESSAGE_ITEMS = 4;

// slab offset of value e of the band, in the order of the reference's four loops
struct Band {
    int ng, mint, mx, my, nxp, n0, n1, n2;
    SmallDiv narrow, bottom, top;
    __device__ __forceinline__ Band(int mx, int my, int mbc)
        : ng(mbc), mint(2 * mbc), mx(mx), my(my), nxp(mx + 2 * mbc), n0((my - mint + ng) * (mint + ng)),
          n1(n0 + (mint + ng) * (mx + ng - mint)), n2(n1 + (my + ng - mint) * (mint + ng)), narrow(mint + ng),
          bottom(mx + ng - mint), top(mx - mint + ng) {}
    __device__ __forceinline__ int operator()(int e) const {
        int i, j;
        if (e < n0) {                    // left, up to the top strip
            const int r = narrow(e);
            j = 1 - ng + r;
            i = 1 - ng + e - r * narrow.d;
        } else if (e < n1) {             // bottom
            e -= n0;
            const int r = bottom(e);
            j = 1 - ng + r;
            i = mint + 1 + e - r * bottom.d;
        } else if (e < n2) {             // right
            e -= n1;
            const int r = narrow(e);
            j = mint + 1 + r;
            i = mx - mint + 1 + e - r * narrow.d;
        } else {                         // top
            e -= n2;
            const int r = top(e);
            j = my - mint + 1 + r;
            i = 1 - ng + e - r * top.d;
        }
        return (j + ng - 1) * nxp + i + ng - 1;
    }
};

__global__ void __launch_bounds__(256)
ghost_message(double* __restrict__ q, double* __restrict__ reg, const int* __restrict__ slots,
              int nband, long long pstride, long long rstride,
              int mx, int my, int mbc, int meqn, const double* __restrict__ dxs,
              const double* __restrict__ dys, double* __restrict__ buf, int elems, int unpack) {
    const int p = blockIdx.x, slot = slots[p];
    double* qp = q + (long long) slot * pstride;
    double* rp = reg + (long long) slot * rstride;
    double* b = buf + (long long) p * elems;
    const int plane = (mx + 2 * mbc) * (my + 2 * mbc), nq = meqn * nband;
    const double dx = dxs[slot], dy = dys[slot];
    const Band band(mx, my, mbc);
    const SmallDiv by_field(nband), by_my(my), by_mx(mx);
    double v[MESSAGE_ITEMS];
    double* c[MESSAGE_ITEMS];            // the value's place in the patch; a length or an area has none
#pragma unroll
    for (int u = 0; u < MESSAGE_ITEMS; u++) {
        const int k = (blockIdx.y * MESSAGE_ITEMS + u) * 256 + threadIdx.x;
        c[u] = nullptr;
        v[u] = 0.0;
        if (k >= elems) continue;
        if (k < nq) {
            const int m = by_field(k);
            c[u] = qp + (long long) m * plane + band(k - m * nband);
        } else {
            const int per = 4 * meqn + 2, r = k - nq;
            const bool xface = r < 2 * per * my;
            const int len = xface ? my : mx, t2 = xface ? r : r - 2 * per * my, second = t2 >= per * len;
            const int f = (xface ? 0 : 2) + second, t = t2 - second * per * len;
            if (t < 4 * meqn * len) {
                const int j = t >> 2, kind = t & 3;        // kinds FM, FP, EFIN, EFOUT in order
                const int m = xface ? by_my(j) : by_mx(j), pos = j - m * len;
                c[u] = rp + ((f * 4 + kind) * meqn + m) * mx + pos;
            } else {
                v[u] = ((t - 4 * meqn * len) & 1) ? dx * dy : xface ? dy : dx;
            }
        }
        if (unpack) v[u] = b[k];
        else if (c[u]) v[u] = *c[u];
    }
#pragma unroll
    for (int u = 0; u < MESSAGE_ITEMS; u++) {
        const int k = (blockIdx.y * MESSAGE_ITEMS + u) * 256 + threadIdx.x;
        if (k >= elems) continue;
        if (!unpack) b[k] = v[u];
        else if (c[u]) *c[u] = v[u];
    }
}

int launch_ghost_message(double* q, double* reg, const int* slots, int n, int nband, long long pstride,
                         long long rstride, int mx, int my, int mbc, int meqn, const double* dxs, const double* dys,
                         double* buf, int elems, int unpack, hipStream_t st) {
    if (n <= 0) return 0;
    const int chunk = 256 * MESSAGE_ITEMS;
    hipLaunchKernelGGL(ghost_message, dim3(n, (elems + chunk - 1) / chunk), dim3(256), 0, st, q, reg, slots, nband,
                       pstride, rstride, mx, my, mbc, meqn, dxs, dys, buf, elems, unpack);
    return (int) hipGetLastError();
}

// Cell values of the VTK "meqn" array: per patch, cells j = 1..my, i = 1..mx,
// then the meqn fields of the cell, as float (fclaw2d_output_vtk_value_cb,
// src/patches/clawpatch/fclaw2d_clawpatch_output_vtk.c:781-808).
__global__ void __launch_bounds__(256)
vtk_cell_values(const double* __restrict__ q, int first, long long pstride, int mx, int my,
                int mbc, int meqn, float* __restrict__ out) {
    const int p = blockIdx.y;
    const int per = mx * my * meqn;
    const double* qp = q + (long long) (first + p) * pstride;
    const int nxp = mx + 2 * mbc, nyp = my + 2 * mbc;
    for (int e = blockIdx.x * blockDim.x + threadIdx.x; e < per; e += gridDim.x * blockDim.x) {
        const int cell = e / meqn, k = e - cell * meqn;
        const int j = cell / mx, i = cell - j * mx;
        out[(long long) p * per + e] = (float) qp[((long long) k * nyp + j + mbc) * nxp + i + mbc];
    }
}

int launch_vtk_cell_values(const double* q, int first, int count, long long pstride, int mx, int my,
                           int mbc, int meqn, float* out, hipStream_t st) {
    if (count <= 0) return 0;
    const int per = mx * my * meqn;
    dim3 grid((unsigned) std::min(64, (per + 255) / 256), count);
    hipLaunchKernelGGL(vtk_cell_values, grid, dim3(256), 0, st, q, first, pstride, mx, my, mbc,
                       meqn, out);
    return (int) hipGetLastError();
}

int launch_timeinterp(const double* q, const double* qlast, double* qti, const int* slots, int n,
                      long long pstride, int mx, int my, int mbc, int meqn, double alpha,
                      hipStream_t st) {
    if (n <= 0) return 0;
    dim3 grid((meqn * mx * my + 255) / 256, n);
    hipLaunchKernelGGL(timeinterp_band, grid, dim3(256), 0, st, q, qlast, qti, slots, n, pstride,
                       mx, my, mbc, meqn, alpha);
    return (int) hipGetLastError();
}

int launch_tag_patches(const double* q, const int* slots, int n, const double* dxs,
                       const double* dys, long long pstride, int mx, int my, int mbc, int ivar,
                       double thr_refine, double thr_coarsen, int* out, hipStream_t st) {
    if (n <= 0) return 0;
    hipLaunchKernelGGL(tag_patches, dim3(n), dim3(256), 0, st, q, slots, n, dxs, dys, pstride, mx, my, mbc, ivar,
                       tag_threshold(thr_refine, thr_refine < 0), tag_threshold(thr_coarsen, thr_coarsen <= 0),
                       (int2*) out);
    return (int) hipGetLastError();
}

int launch_regrid_remap(const double* qold, double* qnew, const int* ops, int nops,
                        long long pstride, int mx, int my, int mbc, int meqn, hipStream_t st) {
    if (nops <= 0) return 0;
    hipLaunchKernelGGL(regrid_remap, dim3(nops), dim3(256), 0, st, qold, qnew, ops, nops, pstride,
                       mx, my, mbc, meqn);
    return (int) hipGetLastError();
}

int launch_reset_cfl(unsigned long long* p, int blocks, unsigned long long* sum, hipStream_t st) {
    hipLaunchKernelGGL(reset_cfl, dim3(blocks), dim3(CFL_WORDS), 0, st, p, sum);
    return (int) hipGetLastError();
}

int launch_collect_steps(unsigned long long* cfl, int blocks, unsigned long long* sum, unsigned long long* out,
                         hipStream_t st) {
    const int threads = blocks > 0 ? CFL_WORDS * ((blocks + 3) / 4 * 4) : 64;   // (whole waves)
    hipLaunchKernelGGL(collect_steps, dim3(1), dim3(threads), 0, st, cfl, blocks, sum, out);
    return (int) hipGetLastError();
}

int launch_copy_interior(const double* src, double* dst, const int* slots, int n,
                         long long pstride, int mx, int my, int mbc, int meqn,
                         hipStream_t st) {
    if (n <= 0) return 0;
    const int per = meqn * mx * my;
    dim3 grid((per + 255) / 256, n);
    hipLaunchKernelGGL(copy_interior, grid, dim3(256), 0, st, src, dst, slots, n, pstride, mx,
                       my, mbc, meqn);
    return (int) hipGetLastError();
}

int launch_mass(const double* q, const int* slots, int n, const double* dxs, const double* dys,
                long long pstride, int mx, int my, int mbc, int meqn, double* parts, double* out,
                hipStream_t st) {
    const int groups = std::min(n, MASS_GROUPS);
    if (groups > 0)
        hipLaunchKernelGGL(mass_groups, dim3(groups), dim3(256), 0, st, q, slots, n, dxs, dys, pstride,
                           mx, my, mbc, meqn, parts);
    hipLaunchKernelGGL(mass_total, dim3(meqn), dim3(256), 0, st, parts, groups, meqn, out);
    return (int) hipGetLastError();
}

// ---------------------------------------------------------------- time sync
// The reference's fclaw2d_time_sync (src/fclaw2d_time_sync.c:118-202) with its
// Fortran kernels clawpack46_fort_time_sync_samesize / _f2c
// (src/solvers/fc2d_clawpack4.6/fortran_source/clawpack46_time_sync.f:249-700):
// the coarse patch's edge flux is replaced by the sum of the fine fluxes
// across each coarse/fine face, and half the mismatch between same-size
// neighbours goes to each side.  One workgroup per destination patch runs its
// ops in order (same-size faces 0..3, then coarse/fine faces), so a corner
// cell receives its corrections in the reference's order.  Registers are
// read only; every op writes cells of its own destination patch.
__global__ void __launch_bounds__(128) time_sync_groups(SyncArgs a) {
    const int g = blockIdx.x;
    if (g >= a.ngroups) return;
    const int mx = a.mx, mbc = a.mbc, meqn = a.meqn, nx = mx + 2 * mbc;
    const int kout = a.fluxreg ? REG_EFIN : REG_EFOUT;
    for (int o = a.start[g]; o < a.start[g + 1]; o++) {
        const int* op = a.ops + 8 * o;
        const int type = op[0], dst = op[1], src = op[2], face = op[3], ti = op[4], tj = op[5];
        double* __restrict__ q = a.q + (long long) dst * a.pstride;
        const double* __restrict__ rt = a.reg + (long long) dst * a.rstride;
        const double* __restrict__ rn = a.reg + (long long) src * a.rstride;
        const double area = a.dxs[dst] * a.dys[dst];
        const int kn = face ^ 1;              // the neighbour's face on this interface
        const int kfl = (face == 0 || face == 2) ? REG_FP : REG_FM;
        for (int e = threadIdx.x; e < meqn * mx; e += blockDim.x) {
            const int m = e / mx, c = e - m * mx + 1;   // c = 1..mx along the face
            auto R = [&](const double* r, int k, int kind, int pos) -> double {
                return r[((k * 4 + kind) * meqn + m) * mx + pos];
            };
            int i, j;
            if (face == 0) { i = 1; j = c; }
            else if (face == 1) { i = mx; j = c; }
            else if (face == 2) { i = c; j = 1; }
            else { i = c; j = mx; }
            double* qc = q + ((long long) m * nx + (j + mbc - 1)) * nx + (i + mbc - 1);
            const double ein = R(rt, face, REG_EFIN, c - 1);
            const double ft = a.fluxreg ? 0.0 : R(rt, face, kfl, c - 1);
            if (type == SYNC_SAMESIZE) {
                const double ef = R(rn, kn, kout, c - 1);
                const double fn = a.fluxreg ? 0.0 : R(rn, kn, kfl, c - 1);
                const double delta = (face == 0 || face == 2) ? (ef - ein) - (fn - ft)
                                                              : (ein - ef) - (fn - ft);
                *qc = *qc + 0.5 * delta / area;
            } else {
                const int f0 = 2 * c - 1 + (face < 2 ? tj : ti);  // fine rows/columns f0, f0+1
                double deltac = 0.0;
                if (f0 >= 1 && f0 + 1 <= mx) {
                    const double ef = R(rn, kn, kout, f0 - 1) + R(rn, kn, kout, f0);
                    const double flu = a.fluxreg ? 0.0 : R(rn, kn, kfl, f0 - 1) + R(rn, kn, kfl, f0);
                    deltac = (face == 0 || face == 2) ? (ef - ein) - (flu - ft) : (ein - ef) - (flu - ft);
                }
                *qc = *qc + deltac / area;
            }
        }
        __syncthreads();
    }
}

// The same corrections in two passes: every (op, field, position) of the
// group computes its increment into LDS at once, then every edge cell adds
// the increments of the ops on its face(s) in op order and is written once.
// A corner cell belongs to the x-face thread, which also takes the y-face
// ops' increments at the matching position; the sums are the one-op-at-a-time
// sums, operation for operation.
__global__ void __launch_bounds__(256) time_sync_cells(SyncArgs a) {
    extern __shared__ double inc[];   // [maxgroup][meqn][mx], then the ops' faces
    const int g = blockIdx.x;
    if (g >= a.ngroups) return;
    const int mx = a.mx, mbc = a.mbc, meqn = a.meqn, nx = mx + 2 * mbc;
    const int per = meqn * mx;
    const int o0 = a.start[g], nop = a.start[g + 1] - o0;
    int* oface = (int*) (inc + (long long) a.maxgroup * per);
    const int kout = a.fluxreg ? REG_EFIN : REG_EFOUT;
    const int dst = a.ops[8 * o0 + 1];
    const double area = a.dxs[dst] * a.dys[dst];
    const double* __restrict__ rt = a.reg + (long long) dst * a.rstride;
    const SmallDiv by_per(per), by_mx(mx);
    double* __restrict__ q = a.q + (long long) dst * a.pstride;
    // the edge cell of element e = (face, field, position), and the other face of a corner
    auto edge = [&](int e, int& f, int& m, int& c) __attribute__((always_inline)) {
        f = by_per(e);
        const int r = e - f * per;
        m = by_mx(r);
        c = r - m * mx + 1;
        const int i = f == 0 ? 1 : f == 1 ? mx : c, j = f == 2 ? 1 : f == 3 ? mx : c;
        return q + ((long long) m * nx + (j + mbc - 1)) * nx + (i + mbc - 1);
    };
    // a thread's first edge cell is under way while the increments are computed
    double first = 0.0;
    {
        int f, m, c;
        if ((int) threadIdx.x < 4 * per) first = *edge(threadIdx.x, f, m, c);
    }
    for (int k = threadIdx.x; k < nop; k += blockDim.x) oface[k] = a.ops[8 * (o0 + k) + 3];
    for (int e = threadIdx.x; e < nop * per; e += blockDim.x) {
        const int k = by_per(e), r = e - k * per, m = by_mx(r), c = r - m * mx + 1;
        const int* op = a.ops + 8 * (o0 + k);
        const int type = op[0], src = op[2], face = op[3], ti = op[4], tj = op[5];
        const double* __restrict__ rn = a.reg + (long long) src * a.rstride;
        const int kn = face ^ 1;
        const int kfl = (face == 0 || face == 2) ? REG_FP : REG_FM;
        auto R = [&](const double* rr, int kk, int kind, int pos) -> double {
            return rr[((kk * 4 + kind) * meqn + m) * mx + pos];
        };
        const double ein = R(rt, face, REG_EFIN, c - 1);
        const double ft = a.fluxreg ? 0.0 : R(rt, face, kfl, c - 1);
        double v;
        if (type == SYNC_SAMESIZE) {
            const double ef = R(rn, kn, kout, c - 1);
            const double fn = a.fluxreg ? 0.0 : R(rn, kn, kfl, c - 1);
            const double delta = (face == 0 || face == 2) ? (ef - ein) - (fn - ft) : (ein - ef) - (fn - ft);
            v = 0.5 * delta / area;
        } else {
            const int f0 = 2 * c - 1 + (face < 2 ? tj : ti);
            double deltac = 0.0;
            if (f0 >= 1 && f0 + 1 <= mx) {
                const double ef = R(rn, kn, kout, f0 - 1) + R(rn, kn, kout, f0);
                const double flu = a.fluxreg ? 0.0 : R(rn, kn, kfl, f0 - 1) + R(rn, kn, kfl, f0);
                deltac = (face == 0 || face == 2) ? (ef - ein) - (flu - ft) : (ein - ef) - (flu - ft);
            }
            v = deltac / area;
        }
        inc[e] = v;
    }
    __syncthreads();
    for (int e = threadIdx.x; e < 4 * per; e += blockDim.x) {
        int f, m, c;
        double* qc = edge(e, f, m, c);
        if (f >= 2 && (c == 1 || c == mx)) continue;   // corners: the x-face thread
        int f2 = -1, c2 = 0;
        if (f < 2 && (c == 1 || c == mx)) { f2 = c == 1 ? 2 : 3; c2 = f == 0 ? 1 : mx; }
        double v = e == (int) threadIdx.x ? first : *qc;
        bool touched = false;
        for (int k = 0; k < nop; k++) {
            const int fk = oface[k];
            if (fk != f && fk != f2) continue;
            v = v + inc[(k * meqn + m) * mx + (fk == f ? c : c2) - 1];
            touched = true;
        }
        if (touched) *qc = v;
    }
}

int launch_time_sync(const SyncArgs& a, hipStream_t st) {
    if (a.ngroups > 0) {
        const size_t lds = sizeof(double) * (size_t) a.maxgroup * a.meqn * a.mx + sizeof(int) * (size_t) a.maxgroup;
        if (lds <= 32768)
            hipLaunchKernelGGL(time_sync_cells, dim3(a.ngroups), dim3(256), lds, st, a);
        else
            hipLaunchKernelGGL(time_sync_groups, dim3(a.ngroups), dim3(128), 0, st, a);
        if (hipError_t e = hipGetLastError()) return (int) e;
    }
    return (int) hipGetLastError();
}

// ---------------------------------------------------------------- FP64 step
int launch_step_fp64(int solver, int tile, int waves, const StepArgs& a, const StepLaunch& st) {
    switch (solver) {
    case 0: return launch_step_tile<RPAdvection<double>, double, true>(tile, waves, a, st);
    case 1: return launch_step_tile<RPShallow<double>, double, true, true>(tile, waves, a, st);
    case 2: return launch_step_tile<RPEuler<double>, double, true>(tile, waves, a, st);
    default: return (int) hipErrorInvalidValue;
    }
}

}  // namespace hipclaw
