// GAD_IMPLICIT_R on gfx950: the implicit vertical advection (3rd-order upwind) + diffusion solve of a tracer
// (reference core/tracer_implicit.py:34-173; gad_implicit_r.F, gad_u3c4_impl_r.F, solve_pentadiagonal.F).
//
// One thread per water column (every padded column of every member; halo columns carry identity rows, as the
// reference's matrix does). The thread walks k = 1..Nr once: it builds row k of the pentadiagonal matrix from the
// level data of k-1..k+2 (diffusion from kappaRX and the masks; advection from the U3 coefficients of the interface
// below level k, computed here, and of the interface above it, kept from row k-1) and eliminates the row at once
// (the forward sweep of SOLVE_DIAGONAL_KINNER), keeping the normalised super-diagonals d', e' in LDS and y' in the
// output column; the back substitution then walks k = Nr..1. Every expression is the reference's, in its order
// (-ffp-contract=off), so the result is bitwise the reference's. Level data are loaded kPf levels ahead of the row
// being built (a register ring with compile-time slots), so each lane keeps up to 5 x kPf loads in flight; the
// columns of a wave are consecutive points of a row (coalesced). The per-level constants sit in LDS and the rows
// between the first two and the last two run branch-free, so that no wait for a load is forced before its use.
#include <type_traits>

#include "mj_common.h"

namespace mj {
namespace {

#ifndef MJ_IMPR_REG50
#define MJ_IMPR_REG50 1
#endif
constexpr int kImprThreads = 64;  // one wave per workgroup (LDS: 2 * nr * 64 + 3 * nr doubles)
#ifndef MJ_IMPR_PF
#define MJ_IMPR_PF 16
#endif
constexpr int kPf = MJ_IMPR_PF;  // prefetch distance in levels
static_assert(kPf >= 3, "the ring must hold levels m .. m+2");
constexpr double kSixth = 1.0 / 6.0;

struct ImprArgs {
    int T, nx, ny, sNx, sNy, OL, nr, adv;
    int64_t plane, ms3, mms;
    const double *maskC, *rA, *recip_rA, *dt, *rdrF, *rdrC;
    double rkSign;
    const double *kap, *rh, *w, *y;
    double* out;
};

// U3 coefficients of interface K (0-based, between levels K-1 and K; Fortran k = K+1), reference
// tracer_implicit.py:71-86: mCup = maskC(K-1), mCkm2 = maskC(max(0, K-2)), mCkp1 = maskC(min(nr-1, K+1)).
struct Iface {
    double rC, rUp, km, kp;
};
__device__ __forceinline__ Iface iface(const ImprArgs& a, int K, double w, double rA, double rrA, double mCup,
                                       double mCkm2, double mCkp1) {
    Iface f;
    const double rTrans = (w * rA) * mCup;
    f.rC = ((0.5 * rTrans) * rrA) * a.rkSign;
    const double mskM = mCkm2 * (K <= 1 ? 0.0 : 1.0);
    const double mskP = mCkp1 * (K >= a.nr - 1 ? 0.0 : 1.0);
    const double ab = fabs(f.rC);
    f.rUp = (2.0 * kSixth) * ab;
    f.km = (kSixth * (f.rC + ab)) * mskM;
    f.kp = (kSixth * (f.rC - ab)) * mskP;
    return f;
}

// solve_pentadiagonal.F:256-267 (reference tracer_implicit.py:120-124)
__device__ __forceinline__ void norm3(double cp, double& dp, double& ep, double& yp) {
    const bool nz = cp != 0.0;
    const double rec = 1.0 / (nz ? cp : 1.0);
    dp = nz ? dp * rec : 0.0;
    ep = nz ? ep * rec : 0.0;
    yp = nz ? yp * rec : 0.0;
}

// Per-thread state of the sweep down a column.
struct ColState {
    double mC1;            // maskC of level m-1
    Iface up;              // interface m (above level m), built by row m-1
    double dp1, ep1, yp1;  // row m-1 after elimination
    double dp2, ep2, yp2;  // row m-2
};

// Row m of the matrix and its elimination. GEN: any m (the branches of the first and last rows); otherwise
// 2 <= m <= nr-3, branch-free, so that the loads of the ring stay in flight across rows. Level data: mC0, rh0, kap0,
// y0 of level m; mCn, kapn, wn of level m+1; mCk = maskC(min(nr-1, m+2)). Halo columns (in = false) get identity
// rows; their level data are loaded like the others' and ignored.
// STORE: write d', e' to LDS and y' to the output column (else the caller keeps them, from c); NRC: the level count
// when known at compile time (0: a.nr).
template <bool GEN, bool ADV, bool STORE = true, int NRC = 0>
__device__ __forceinline__ void impr_row(const ImprArgs& a, int m, bool in, double rA, double rrA, double mC0,
                                         double rh0, double kap0, double y0, double mCn, double kapn, double wn,
                                         double mCk, ColState& c, double* dpL, double* epL, double* out,
                                         const double* lv) {
    const int nr = NRC ? NRC : a.nr;
    const double dtm = lv[m], rdf = lv[nr + m];
    const double* rdrC = lv + 2 * nr;
    const bool hasU = !GEN || m >= 1, hasL = !GEN || m + 1 < nr;
    // diffusion, reference tracer_implicit.py:54-64
    double rb = 0.0, rd = 0.0, ra = 0.0, re = 0.0;
    if (hasU) rb = -(((((dtm * c.mC1) * rh0) * rdf) * kap0) * rdrC[m]);
    if (hasL) rd = -(((((dtm * mCn) * rh0) * rdf) * kapn) * rdrC[m + 1]);
    double rc = 1.0 - (rb + rd);
    if (ADV) {
        // U3 advection, :95-105: level m takes the updates of interface m+1 (its bottom) first, then those of
        // interface m (its top)
        Iface lo{0.0, 0.0, 0.0, 0.0};
        if (hasL) {
            lo = iface(a, m + 1, wn, rA, rrA, mC0, (!GEN || m >= 1) ? c.mC1 : mC0, mCk);
            rb = rb - ((lo.km * dtm) * rh0) * rdf;
            rc = rc + (((((lo.rC + lo.rUp) + lo.km) * dtm) * rh0) * rdf);
            rd = rd + (((((lo.rC - lo.rUp) + lo.kp) * dtm) * rh0) * rdf);
            re = re - ((lo.kp * dtm) * rh0) * rdf;
        }
        if (hasU) {
            ra = ra + ((c.up.km * dtm) * rh0) * rdf;
            rb = rb - (((((c.up.rC + c.up.rUp) + c.up.km) * dtm) * rh0) * rdf);
            rc = rc - (((((c.up.rC - c.up.rUp) + c.up.kp) * dtm) * rh0) * rdf);
            rd = rd + ((c.up.kp * dtm) * rh0) * rdf;
        }
        c.up = lo;
    }
    if (!in) ra = 0.0, rb = 0.0, rc = 1.0, rd = 0.0, re = 0.0;
    // forward elimination, reference tracer_implicit.py:126-143 (rows 0 and 1 through their own formulas)
    double dq, eq = re, yq;
    if (GEN && m == 0) {
        dq = rd;
        yq = y0;
        norm3(rc, dq, eq, yq);
    } else if (GEN && m == 1) {
        const double c2 = rc - rb * c.dp1;
        dq = rd - rb * c.ep1;
        yq = y0 - rb * c.yp1;
        norm3(c2, dq, eq, yq);
    } else {
        const double bb = rb - ra * c.dp2;
        const double cq = (rc - ra * c.ep2) - bb * c.dp1;
        dq = rd - bb * c.ep1;
        yq = (y0 - ra * c.yp2) - bb * c.yp1;
        norm3(cq, dq, eq, yq);
    }
    if (STORE) {
        dpL[(int64_t)m * kImprThreads] = dq;
        epL[(int64_t)m * kImprThreads] = eq;
        out[(int64_t)m * a.plane] = yq;
    }
    c.dp2 = c.dp1, c.ep2 = c.ep1, c.yp2 = c.yp1;
    c.dp1 = dq, c.ep1 = eq, c.yp1 = yq;
    c.mC1 = mC0;
}

template <bool ADV>
__global__ void __launch_bounds__(kImprThreads) impr_kernel(ImprArgs a) {
    extern __shared__ double lds[];
    const int lane = threadIdx.x;
    const int64_t col = (int64_t)blockIdx.x * kImprThreads + lane;
    const int mem = blockIdx.y;
    // the per-level constants (deltaT, recip_drF, recip_drC) in LDS: read per row without vector-memory waits
    double* lv = lds + (int64_t)2 * a.nr * kImprThreads;
    for (int k = lane; k < a.nr; k += kImprThreads) {
        lv[k] = a.dt[k];
        lv[a.nr + k] = a.rdrF[k];
        lv[2 * a.nr + k] = a.rdrC[k];
    }
    __syncthreads();
    if (col >= (int64_t)a.T * a.plane) return;  // no barriers below
    const int t = (int)(col / a.plane), q = (int)(col - (int64_t)t * a.plane);
    const int j = q / a.nx, i = q - j * a.nx;
    const bool in = j >= a.OL && j < a.OL + a.sNy && i >= a.OL && i < a.OL + a.sNx;
    const int nr = a.nr;
    const int64_t o3 = mem * a.ms3 + (int64_t)t * nr * a.plane + q;
    const int64_t om = mem * a.mms + (int64_t)t * nr * a.plane + q;
    const double* y = a.y + o3;
    double* out = a.out + o3;
    double* dpL = lds + lane;
    double* epL = lds + (int64_t)nr * kImprThreads + lane;
    const int64_t o2 = (int64_t)t * a.plane + q;
    const double rA = ADV ? a.rA[o2] : 0.0;
    const double rrA = ADV ? a.recip_rA[o2] : 0.0;
    // as in impr_reg_kernel: halo columns re-read the tracer's lines
    const double* mCp = in ? a.maskC + om : y;
    const double *rhp = in ? a.rh + o3 : y, *kp = in ? a.kap + o3 : y, *wp = in ? a.w + o3 : y;

    // ring of level data: slot s holds a level m with m % kPf == s; loads are unconditional (levels clamped to
    // nr-1) so that no branch separates a load from its use
    double rmC[kPf], rrh[kPf], rkap[kPf], rw[kPf], ry[kPf];
    auto load = [&](int s, int lev) {
        const int64_t ok = (int64_t)min(lev, nr - 1) * a.plane;
        ry[s] = y[ok];
        rmC[s] = mCp[ok];
        rrh[s] = rhp[ok];
        rkap[s] = kp[ok];
        rw[s] = wp[ok];
    };
#pragma unroll
    for (int s = 0; s < kPf; ++s) load(s, s);
    ColState c{0.0, {0.0, 0.0, 0.0, 0.0}, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0};
    auto mck = [&](int m, int s2, int s1) { return m + 2 < nr ? rmC[s2] : rmC[s1]; };
    // rows 0 and 1
#pragma unroll
    for (int s = 0; s < 2; ++s) {
        if (s < nr) {
            const int s1 = (s + 1) % kPf, s2 = (s + 2) % kPf;
            impr_row<true, ADV>(a, s, in, rA, rrA, rmC[s], rrh[s], rkap[s], ry[s], rmC[s1], rkap[s1], rw[s1],
                           mck(s, s2, s1), c, dpL, epL, out, lv);
            load(s, s + kPf);
        }
    }
    // rows 2 .. nr-3 in laps of kPf (a lap starts at m = 2 mod kPf, so slot (2 + s) % kPf is level m0 + s)
    int m0 = 2;
    for (; m0 + kPf - 1 <= nr - 3; m0 += kPf) {
#pragma unroll
        for (int s = 0; s < kPf; ++s) {
            const int m = m0 + s;
            const int s0 = (2 + s) % kPf, s1 = (3 + s) % kPf, s2 = (4 + s) % kPf;
            impr_row<false, ADV>(a, m, in, rA, rrA, rmC[s0], rrh[s0], rkap[s0], ry[s0], rmC[s1], rkap[s1], rw[s1],
                            rmC[s2], c, dpL, epL, out, lv);
            load(s0, m + kPf);
        }
    }
    // the remaining rows (at most kPf + 1)
#pragma unroll
    for (int s = 0; s < kPf + 2; ++s) {
        const int m = m0 + s;
        if (m < nr) {
            const int s0 = (2 + s) % kPf, s1 = (3 + s) % kPf, s2 = (4 + s) % kPf;
            impr_row<true, ADV>(a, m, in, rA, rrA, rmC[s0], rrh[s0], rkap[s0], ry[s0], rmC[s1], rkap[s1], rw[s1],
                           mck(m, s2, s1), c, dpL, epL, out, lv);
            load(s0, m + kPf);
        }
    }
    // back substitution, reference tracer_implicit.py:150-160: u(nr-1) = y'(nr-1) is in place already
    if (nr < 2) return;
    double u1 = c.yp1;  // u(m+1)
    double u0 = c.yp2 - u1 * dpL[(int64_t)(nr - 2) * kImprThreads];
    out[(int64_t)(nr - 2) * a.plane] = u0;
    double u2 = u1;
    u1 = u0;
    // y'(m) for m = nr-3 .. 0 are re-read from the output column, kPf levels ahead (clamped to level 0)
    double ryp[kPf];
#pragma unroll
    for (int s = 0; s < kPf; ++s) ryp[s] = out[(int64_t)max(nr - 3 - s, 0) * a.plane];
    for (int mb = nr - 3; mb >= 0; mb -= kPf) {
#pragma unroll
        for (int s = 0; s < kPf; ++s) {
            const int m = mb - s;
            if (m >= 0) {
                const double u = (ryp[s] - u1 * dpL[(int64_t)m * kImprThreads]) - u2 * epL[(int64_t)m * kImprThreads];
                out[(int64_t)m * a.plane] = u;
                u2 = u1;
                u1 = u;
                ryp[s] = out[(int64_t)max(m - kPf, 0) * a.plane];
            }
        }
    }
}

// The same sweep for a level count known at compile time: the rows are unrolled, so y' of every level stays in
// registers (d', e' in LDS as before) and makes no round trip through the output column: each column is read once
// and written once. Bitwise the generic kernel's arithmetic.
constexpr int kPfR = 8;
template <bool ADV, int NR>
__global__ void __launch_bounds__(kImprThreads) impr_reg_kernel(ImprArgs a) {
    extern __shared__ double lds[];
    const int lane = threadIdx.x;
    const int64_t col = (int64_t)blockIdx.x * kImprThreads + lane;
    const int mem = blockIdx.y;
    double* lv = lds;
    for (int k = lane; k < NR; k += kImprThreads) {
        lv[k] = a.dt[k];
        lv[NR + k] = a.rdrF[k];
        lv[2 * NR + k] = a.rdrC[k];
    }
    __syncthreads();
    if (col >= (int64_t)a.T * a.plane) return;  // no barriers below
    const int t = (int)(col / a.plane), q = (int)(col - (int64_t)t * a.plane);
    const int j = q / a.nx, i = q - j * a.nx;
    const bool in = j >= a.OL && j < a.OL + a.sNy && i >= a.OL && i < a.OL + a.sNx;
    const int64_t o3 = mem * a.ms3 + (int64_t)t * NR * a.plane + q;
    const int64_t om = mem * a.mms + (int64_t)t * NR * a.plane + q;
    const double* y = a.y + o3;
    double* out = a.out + o3;
    const int64_t o2 = (int64_t)t * a.plane + q;
    const double rA = ADV ? a.rA[o2] : 0.0;
    const double rrA = ADV ? a.recip_rA[o2] : 0.0;
    // a halo column only needs the tracer (identity rows): its other loads read the tracer's lines again, which
    // the wave loads anyway (no HBM traffic)
    const double* mCp = in ? a.maskC + om : y;
    const double *rhp = in ? a.rh + o3 : y, *kp = in ? a.kap + o3 : y, *wp = in ? a.w + o3 : y;
    double rmC[kPfR], rrh[kPfR], rkap[kPfR], rw[kPfR], ry[kPfR];
    auto load = [&](int s, int lev) {
        const int64_t ok = (int64_t)lev * a.plane;
        ry[s] = y[ok];
        rmC[s] = mCp[ok];
        rrh[s] = rhp[ok];
        rkap[s] = kp[ok];
        rw[s] = wp[ok];
    };
#pragma unroll
    for (int s = 0; s < kPfR; ++s) load(s, s < NR ? s : NR - 1);
    ColState c{0.0, {0.0, 0.0, 0.0, 0.0}, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0};
    double* dpL = lds + 3 * NR + lane;
    double* epL = dpL + NR * kImprThreads;
    double ypR[NR];
#pragma unroll
    for (int m = 0; m < NR; ++m) {
        const int s = m % kPfR, s1 = (m + 1) % kPfR, s2 = (m + 2) % kPfR;
        const double mCn = m + 1 < NR ? rmC[s1] : 0.0;
        const double mCk = m + 2 < NR ? rmC[s2] : rmC[s1];
        if (m <= 1 || m >= NR - 2)
            impr_row<true, ADV, false, NR>(a, m, in, rA, rrA, rmC[s], rrh[s], rkap[s], ry[s], mCn, rkap[s1], rw[s1],
                                           mCk, c, nullptr, nullptr, nullptr, lv);
        else
            impr_row<false, ADV, false, NR>(a, m, in, rA, rrA, rmC[s], rrh[s], rkap[s], ry[s], mCn, rkap[s1], rw[s1],
                                            mCk, c, nullptr, nullptr, nullptr, lv);
        dpL[m * kImprThreads] = c.dp1;
        epL[m * kImprThreads] = c.ep1;
        ypR[m] = c.yp1;
        if (m + kPfR < NR) load(s, m + kPfR);
    }
    double u1 = ypR[NR - 1];
    out[(int64_t)(NR - 1) * a.plane] = u1;
    double u0 = ypR[NR - 2] - u1 * dpL[(NR - 2) * kImprThreads];
    out[(int64_t)(NR - 2) * a.plane] = u0;
    double u2 = u1;
    u1 = u0;
#pragma unroll
    for (int m = NR - 3; m >= 0; --m) {
        const double u = (ypR[m] - u1 * dpL[m * kImprThreads]) - u2 * epL[m * kImprThreads];
        out[(int64_t)m * a.plane] = u;
        u2 = u1;
        u1 = u;
    }
}

}  // namespace
}  // namespace mj

using namespace mj;

extern "C" int mj_gad_implicit_r(const mj_impr_grid* g, const mj_impr_config* c, const double* kappaRX,
                                 const double* recip_hFac, const double* wFld, const double* gTracer, double* out,
                                 void* stream) {
    MJ_REQUIRE(g && c, "mj_gad_implicit_r: null grid/config");
    MJ_REQUIRE(c->batch >= 1 && c->batch <= 65535 && c->ntiles >= 1 && c->nr >= 1 && c->nr <= 150,
               "mj_gad_implicit_r: batch in 1..65535, ntiles >= 1, nr in 1..150");
    MJ_REQUIRE(c->sNx >= 1 && c->sNy >= 1 && c->OL >= 0, "mj_gad_implicit_r: bad tile layout");
    MJ_REQUIRE(gTracer && out, "mj_gad_implicit_r: null gTracer/out");
    const int nx = c->sNx + 2 * c->OL, ny = c->sNy + 2 * c->OL;
    const int64_t plane = (int64_t)nx * ny, member = (int64_t)c->ntiles * c->nr * plane;
    MJ_REQUIRE(c->batch == 1 || (c->member_stride3d >= member && (c->mask_member_stride == 0 ||
                                                                  c->mask_member_stride >= member)),
               "mj_gad_implicit_r: member strides smaller than one member's arrays");
    MJ_REQUIRE(c->nr == 1 || (kappaRX && recip_hFac && g->maskC && g->dTtracerLev && g->recip_drF && g->recip_drC),
               "mj_gad_implicit_r: null kappaRX/recip_hFac or grid field");
    MJ_REQUIRE(!c->implicitAdvection || (wFld && g->rA && g->recip_rA),
               "mj_gad_implicit_r: implicit advection needs wFld, rA, recip_rA");
    const double* ins[] = {kappaRX, recip_hFac, wFld};
    for (const double* p : ins) MJ_REQUIRE(p != out, "mj_gad_implicit_r: out aliases an input other than gTracer");
    hipStream_t st = as_stream(stream);
    const int64_t cols = (int64_t)c->ntiles * plane;
    if (c->nr == 1) {  // reference tracer_implicit.py:169-170: returned unchanged
        if (out != gTracer)
            MJ_HIP(hipMemcpy2DAsync(out, (size_t)(c->batch == 1 ? cols : c->member_stride3d) * sizeof(double),
                                    gTracer, (size_t)(c->batch == 1 ? cols : c->member_stride3d) * sizeof(double),
                                    (size_t)cols * sizeof(double), (size_t)c->batch, hipMemcpyDeviceToDevice, st));
        return MJ_OK;
    }
    ImprArgs a;
    a.T = c->ntiles;
    a.nx = nx;
    a.ny = ny;
    a.sNx = c->sNx;
    a.sNy = c->sNy;
    a.OL = c->OL;
    a.nr = c->nr;
    a.adv = c->implicitAdvection ? 1 : 0;
    a.plane = plane;
    a.ms3 = c->member_stride3d;
    a.mms = c->mask_member_stride;
    a.maskC = g->maskC;
    a.rA = g->rA;
    a.recip_rA = g->recip_rA;
    a.dt = g->dTtracerLev;
    a.rdrF = g->recip_drF;
    a.rdrC = g->recip_drC;
    a.rkSign = g->rkSign;
    a.kap = kappaRX;
    a.rh = recip_hFac;
    a.w = c->implicitAdvection ? wFld : gTracer;  // without advection the w loads read a valid dummy
    a.y = gTracer;
    a.out = out;
    const size_t lds = ((size_t)2 * c->nr * kImprThreads + 3 * (size_t)c->nr) * sizeof(double);
    const dim3 grid((unsigned)((cols + kImprThreads - 1) / kImprThreads), (unsigned)c->batch);
#if MJ_IMPR_REG50
    if (c->nr == 50) {  // the LLC90 level count: the register-resident sweep
        const size_t lds50 = (3 * 50 + 2 * 50 * kImprThreads) * sizeof(double);
        if (a.adv)
            hipLaunchKernelGGL((impr_reg_kernel<true, 50>), grid, dim3(kImprThreads), lds50, st, a);
        else
            hipLaunchKernelGGL((impr_reg_kernel<false, 50>), grid, dim3(kImprThreads), lds50, st, a);
        MJ_HIP(hipGetLastError());
        return MJ_OK;
    }
#endif
    const void* kern = a.adv ? (const void*)impr_kernel<true> : (const void*)impr_kernel<false>;
    if (lds > 65536) MJ_HIP(hipFuncSetAttribute(kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
    if (a.adv)
        hipLaunchKernelGGL(impr_kernel<true>, grid, dim3(kImprThreads), lds, st, a);
    else
        hipLaunchKernelGGL(impr_kernel<false>, grid, dim3(kImprThreads), lds, st, a);
    MJ_HIP(hipGetLastError());
    return MJ_OK;
}

// ---------------------------------------------------------------------------------------------------- reverse mode
// u = A(kappaRX, wFld)^-1 y per column. Given ubar: lam = A^-T ubar by the same guarded elimination on the
// transposed diagonals (row m of A^T = (e(m-2), d(m-1), c(m), b(m+1), a(m+2))), ybar = lam, and the cotangents of
// kappaRX and wFld from the derivatives of the rows in those parameters (diffusion: b(k), d(k-1), c in kappaRX(k);
// U3: rows K-1 and K in the rCenter of interface K). One thread per column, in two walks over the levels.
//
// Bound by HBM: five arrays are read on the way down (the matrix and ubar), four on the way up (the parameter
// cotangents), three written. Reading the level data as needed kept one or two loads in flight per lane (772 us for two
// members of 50 levels, 1.7 TB/s of these twelve passes); now both walks run on register rings that load kPfA levels
// ahead, in laps of kPfA rows without branches, and the parameter cotangents of interface m + 1 are formed as soon as
// lam(m) is known, so that lam is not read back: 250 us, 5.0 TB/s, where a copy reaches 4.65 and reads alone 6. Six levels
// ahead: four and eight measured within the spread of the runs, and eight no longer fit the registers. For the LLC90 level
// count, as in the forward solve, the walks are unrolled and y' stays in registers (NR). Other counts send it through the
// output column: 74, 167 and 320 us for 15, 30 and 49 levels, and 323 us for 50.
namespace mj {
namespace {

constexpr int kPfA = 6;
static_assert(kPfA >= 4, "the rings must hold the levels of a row");

struct Row {
    double a, b, c, d, e;
};

// Row m of A from the level data of m - 1 .. m + 2 (mC1, mC0, mCn, mCk: maskC of m-1, m, m+1, min(nr-1, m+2); rh0 of m;
// kap0, kapn of m, m+1; wn of m+1; up: interface m, replaced by interface m + 1). GEN as in impr_row.
template <bool GEN, bool ADV>
__device__ __forceinline__ Row adj_row(const ImprArgs& a, const double* lv, int nr, int m, bool in, double rA, double rrA,
                                       double mC1, double mC0, double mCn, double mCk, double rh0, double kap0,
                                       double kapn, double wn, Iface& up) {
    const double dtm = lv[m], rdf = lv[nr + m];
    const double* rdrC = lv + 2 * nr;
    const bool hasU = !GEN || m >= 1, hasL = !GEN || m + 1 < nr;
    Row r{0.0, 0.0, 0.0, 0.0, 0.0};
    if (hasU) r.b = -(((((dtm * mC1) * rh0) * rdf) * kap0) * rdrC[m]);
    if (hasL) r.d = -(((((dtm * mCn) * rh0) * rdf) * kapn) * rdrC[m + 1]);
    r.c = 1.0 - (r.b + r.d);
    if (ADV) {
        Iface lo{0.0, 0.0, 0.0, 0.0};
        if (hasL) {
            lo = iface(a, m + 1, wn, rA, rrA, mC0, (!GEN || m >= 1) ? mC1 : mC0, mCk);
            r.b = r.b - ((lo.km * dtm) * rh0) * rdf;
            r.c = r.c + (((((lo.rC + lo.rUp) + lo.km) * dtm) * rh0) * rdf);
            r.d = r.d + (((((lo.rC - lo.rUp) + lo.kp) * dtm) * rh0) * rdf);
            r.e = r.e - ((lo.kp * dtm) * rh0) * rdf;
        }
        if (hasU) {
            r.a = r.a + ((up.km * dtm) * rh0) * rdf;
            r.b = r.b - (((((up.rC + up.rUp) + up.km) * dtm) * rh0) * rdf);
            r.c = r.c - (((((up.rC - up.rUp) + up.kp) * dtm) * rh0) * rdf);
            r.d = r.d + ((up.kp * dtm) * rh0) * rdf;
        }
        up = lo;
    }
    if (!in) r = Row{0.0, 0.0, 1.0, 0.0, 0.0};  // halo columns: identity
    return r;
}

// Rows of A around the transposed elimination, and its last two rows.
struct AdjState {
    Row rM2, rM1, r0, rP1, rP2;
    Iface up;
    double mC1;
    double dp1, ep1, yp1, dp2, ep2, yp2;
};

// Row m of A^T = (e(m-2), d(m-1), c(m), b(m+1), a(m+2)), eliminated.
template <bool GEN>
__device__ __forceinline__ void adj_eliminate(AdjState& c, int m, double y0) {
    const double ra = c.rM2.e, rb = c.rM1.d, rc = c.r0.c, rd = c.rP1.b;
    double dq, eq = c.rP2.a, yq;
    if (GEN && m == 0) {
        dq = rd;
        yq = y0;
        norm3(rc, dq, eq, yq);
    } else if (GEN && m == 1) {
        const double c2 = rc - rb * c.dp1;
        dq = rd - rb * c.ep1;
        yq = y0 - rb * c.yp1;
        norm3(c2, dq, eq, yq);
    } else {
        const double bb = rb - ra * c.dp2;
        const double cq = (rc - ra * c.ep2) - bb * c.dp1;
        dq = rd - bb * c.ep1;
        yq = (y0 - ra * c.yp2) - bb * c.yp1;
        norm3(cq, dq, eq, yq);
    }
    c.dp2 = c.dp1, c.ep2 = c.ep1, c.yp2 = c.yp1;
    c.dp1 = dq, c.ep1 = eq, c.yp1 = yq;
}

// Cotangents of kappaRX and wFld at interface k (levels k - 1 and k): lk, lk1 = lam(k), lam(k-1); u, maskC of the levels
// k-2 .. k+1 (uM2, uM1, u0, uP1; likewise m..; clamped where they do not exist); rh0, rh1 of k, k-1; w of k.
template <bool ADV>
__device__ __forceinline__ void adj_params(const ImprArgs& a, const double* lv, int nr, int k, bool in, double rA,
                                           double rrA, double lk, double lk1, double uM2, double uM1, double u0,
                                           double uP1, double mM2, double mM1, double m0, double mP1, double rh0,
                                           double rh1, double w, double& gk, double& gw) {
    const double* rdrC = lv + 2 * nr;
    const double beta = -((((lv[k] * mM1) * rh0) * lv[nr + k]) * rdrC[k]);
    const double delta = -((((lv[k - 1] * m0) * rh1) * lv[nr + k - 1]) * rdrC[k]);
    const double du = u0 - uM1;
    gk = -((lk * beta) * (-du) + (lk1 * delta) * du);
    gw = 0.0;
    if (ADV) {
        const double dw = (((0.5 * rA) * mM1) * rrA) * a.rkSign;
        const double rC = ((0.5 * ((w * rA) * mM1)) * rrA) * a.rkSign;
        const double sg = (double)((rC > 0.0) - (rC < 0.0));
        const double mskM = mM2 * (k <= 1 ? 0.0 : 1.0);
        const double mskP = mP1 * (k >= nr - 1 ? 0.0 : 1.0);
        const double drUp = (2.0 * kSixth) * sg;
        const double dkm = (kSixth * (1.0 + sg)) * mskM;
        const double dkp = (kSixth * (1.0 - sg)) * mskP;
        const double uKm2 = k >= 2 ? uM2 : 0.0, uKp1 = k + 1 < nr ? uP1 : 0.0;
        const double phi = (((-dkm) * uKm2 + ((1.0 + drUp) + dkm) * uM1) + ((1.0 - drUp) + dkp) * u0) - dkp * uKp1;
        const double s1 = (lv[k - 1] * rh1) * lv[nr + k - 1], s0 = (lv[k] * rh0) * lv[nr + k];
        const double rCb = -((lk1 * s1) - (lk * s0)) * phi;
        gw = rCb * dw;
    }
    if (!in) gk = 0.0, gw = 0.0;
}

template <bool ADV, int NR>
__global__ void __launch_bounds__(kImprThreads)
    impr_adjoint_kernel(ImprArgs a, const double* u, const double* ubar, double* ybar, double* kbar, double* wbar) {
    extern __shared__ double lds[];
    const int lane = threadIdx.x;
    const int64_t col = (int64_t)blockIdx.x * kImprThreads + lane;
    const int mem = blockIdx.y;
    const int nr = NR ? NR : a.nr;
    double* lv = lds + (int64_t)2 * nr * kImprThreads;
    for (int k = lane; k < nr; k += kImprThreads) {
        lv[k] = a.dt[k];
        lv[nr + k] = a.rdrF[k];
        lv[2 * nr + k] = a.rdrC[k];
    }
    __syncthreads();
    if (col >= (int64_t)a.T * a.plane) return;  // no barriers below
    const int t = (int)(col / a.plane), q = (int)(col - (int64_t)t * a.plane);
    const int j = q / a.nx, i = q - j * a.nx;
    const bool in = j >= a.OL && j < a.OL + a.sNy && i >= a.OL && i < a.OL + a.sNx;
    const int64_t P = a.plane;
    const int64_t o3 = mem * a.ms3 + (int64_t)t * nr * P + q;
    const int64_t om = mem * a.mms + (int64_t)t * nr * P + q;
    const int64_t o2 = (int64_t)t * P + q;
    const double rA = ADV ? a.rA[o2] : 0.0;
    const double rrA = ADV ? a.recip_rA[o2] : 0.0;
    // a halo column only needs ubar (identity rows): its other loads read those lines again
    const double* const ub = ubar + o3;
    const double* const mCp = in ? a.maskC + om : ub;
    const double *const rhp = in ? a.rh + o3 : ub, *const kp = in ? a.kap + o3 : ub, *const wp = in ? a.w + o3 : ub;
    const double* const uc = in ? u + o3 : ub;
    double* const yb = ybar + o3;
    double* const kb = kbar + o3;
    double* const wbp = ADV ? wbar + o3 : nullptr;
    double* const dpL = lds + lane;
    double* const epL = lds + (int64_t)nr * kImprThreads + lane;
    double ypR[NR ? NR : 1];

    // ---- down: the rows of A, and two rows behind them those of A^T eliminated. Slot s of the rings holds a level r with
    // r % kPfA == s; ubar's are read two levels behind.
    const Row zero{0.0, 0.0, 0.0, 0.0, 0.0};
    AdjState c{zero, zero, zero, zero, zero, {0.0, 0.0, 0.0, 0.0}, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0};
    {
        double rmC[kPfA], rrh[kPfA], rkap[kPfA], rw[kPfA], ry[kPfA];
        auto load = [&](int s, int r) {
            const int64_t ok = (int64_t)(NR ? (r < NR ? r : NR - 1) : min(r, nr - 1)) * P;
            rmC[s] = mCp[ok];
            rrh[s] = rhp[ok];
            rkap[s] = kp[ok];
            rw[s] = ADV ? wp[ok] : 0.0;
            ry[s] = ub[ok];
        };
        double yB1 = 0.0, yB2 = 0.0;  // ubar of levels r - 1, r - 2
        auto step = [&](auto gen, int r, int s) {
            constexpr bool GEN = decltype(gen)::value;
            const int s1 = (s + 1) % kPfA, s2 = (s + 2) % kPfA;
            c.rM2 = c.rM1, c.rM1 = c.r0, c.r0 = c.rP1, c.rP1 = c.rP2;
            c.rP2 = zero;
            if (!GEN || r < nr) {
                const double mCk = !GEN || r + 2 < nr ? rmC[s2] : rmC[s1];
                c.rP2 = adj_row<GEN, ADV>(a, lv, nr, r, in, rA, rrA, c.mC1, rmC[s], rmC[s1], mCk, rrh[s], rkap[s],
                                          rkap[s1], rw[s1], c.up);
                c.mC1 = rmC[s];
            }
            const int m = r - 2;
            if (!GEN || m >= 0) {
                adj_eliminate<GEN>(c, m, yB2);
                dpL[(int64_t)m * kImprThreads] = c.dp1;
                epL[(int64_t)m * kImprThreads] = c.ep1;
                if constexpr (NR != 0)
                    ypR[m >= 0 ? m : 0] = c.yp1;
                else
                    yb[m * P] = c.yp1;
            }
            yB2 = yB1;
            yB1 = ry[s];
            load(s, r + kPfA);
        };
#pragma unroll
        for (int s = 0; s < kPfA; ++s) load(s, s);
        if constexpr (NR != 0) {
#pragma unroll
            for (int r = 0; r < NR + 2; ++r) {
                if (r < 4 || r > NR - 3)
                    step(std::true_type{}, r, r % kPfA);
                else
                    step(std::false_type{}, r, r % kPfA);
            }
        } else {
            // the first lap, laps of interior rows, the rest
#pragma unroll
            for (int s = 0; s < kPfA; ++s)
                if (s < nr + 2) step(std::true_type{}, s, s);
            int r0 = kPfA;
            for (; r0 + kPfA - 1 <= nr - 3; r0 += kPfA) {
#pragma unroll
                for (int s = 0; s < kPfA; ++s) step(std::false_type{}, r0 + s, s);
            }
#pragma unroll
            for (int s = 0; s < kPfA + 4; ++s)
                if (r0 + s < nr + 2) step(std::true_type{}, r0 + s, s % kPfA);
        }
    }
    // ---- up: lam(m), and with it the cotangents at interface k = m + 1. Slot s of the rings holds level l = m - 1 of step
    // m, counted down from nr - 1: l = nr - 1 - n with n % kPfA == s.
    {
        double rmC[kPfA], rrh[kPfA], rw[kPfA], ru[kPfA], ry[kPfA];
        auto load = [&](int s, int n) {
            const int64_t ok = (int64_t)max(nr - 1 - n, 0) * P;
            rmC[s] = mCp[ok];
            rrh[s] = rhp[ok];
            if (ADV) rw[s] = wp[ok];
            ru[s] = uc[ok];
            if (NR == 0) ry[s] = yb[ok];
        };
#pragma unroll
        for (int s = 0; s < kPfA; ++s) load(s, s);
        // levels m + 2, m + 1, m of the window (index 0, 1, 2) and the new level m - 1
        double W_m[3] = {0.0, 0.0, 0.0}, W_u[3] = {0.0, 0.0, 0.0}, W_rh[3] = {0.0, 0.0, 0.0}, W_w[3] = {0.0, 0.0, 0.0};
        double W_y = 0.0, u1 = 0.0, u2 = 0.0;
        auto step = [&](int n, int s) {  // takes level l = nr - 1 - n in; finishes m = l + 1
            const int m = nr - n;
            const double nm = rmC[s], nu = ru[s], nrh = rrh[s], nw = ADV ? rw[s] : 0.0;
            if (m < nr) {  // lam(m)
                const double y = NR ? ypR[m < 0 ? 0 : m] : W_y;
                double v;
                if (m == nr - 1)
                    v = y;
                else if (m == nr - 2)
                    v = y - u1 * dpL[(int64_t)m * kImprThreads];
                else
                    v = (y - u1 * dpL[(int64_t)m * kImprThreads]) - u2 * epL[(int64_t)m * kImprThreads];
                yb[m * P] = v;
                const int k = m + 1;
                if (k < nr) {
                    double gk, gw;
                    // mask of level k + 1 clamped to nr - 1, of level k - 2 to 0 (nm repeats level 0 there)
                    const double mP1 = k + 1 < nr ? W_m[0] : W_m[1];
                    adj_params<ADV>(a, lv, nr, k, in, rA, rrA, u1, v, nu, W_u[2], W_u[1], W_u[0], nm, W_m[2], W_m[1], mP1,
                                    W_rh[1], W_rh[2], W_w[1], gk, gw);
                    kb[k * P] = gk;
                    if (ADV) wbp[k * P] = gw;
                }
                u2 = u1;
                u1 = v;
            }
            W_m[0] = W_m[1], W_m[1] = W_m[2], W_m[2] = nm;
            W_u[0] = W_u[1], W_u[1] = W_u[2], W_u[2] = nu;
            W_rh[0] = W_rh[1], W_rh[1] = W_rh[2], W_rh[2] = nrh;
            W_w[0] = W_w[1], W_w[1] = W_w[2], W_w[2] = nw;
            if (NR == 0) W_y = ry[s];
            load(s, n + kPfA);
        };
        // n = 0 takes level nr - 1 in; n = nr (level 0 again) finishes m = 0
        if constexpr (NR != 0) {
#pragma unroll
            for (int n = 0; n <= NR; ++n) step(n, n % kPfA);
        } else {
            int n0 = 0;
            for (; n0 + kPfA - 1 <= nr; n0 += kPfA) {
#pragma unroll
                for (int s = 0; s < kPfA; ++s) step(n0 + s, s);
            }
#pragma unroll
            for (int s = 0; s < kPfA; ++s)
                if (n0 + s <= nr) step(n0 + s, s);
        }
        kb[0] = 0.0;  // level 0 and the surface interface have none
        if (ADV) wbp[0] = 0.0;
    }
}

}  // namespace
}  // namespace mj

extern "C" int mj_gad_implicit_r_adjoint(const mj_impr_grid* g, const mj_impr_config* c, const double* kappaRX,
                                         const double* recip_hFac, const double* wFld, const double* u,
                                         const double* ubar, double* ybar, double* kappaRX_bar, double* wFld_bar,
                                         void* stream) {
    MJ_REQUIRE(g && c, "mj_gad_implicit_r_adjoint: null grid/config");
    MJ_REQUIRE(c->batch >= 1 && c->batch <= 65535 && c->ntiles >= 1 && c->nr >= 2 && c->nr <= 150,
               "mj_gad_implicit_r_adjoint: batch in 1..65535, ntiles >= 1, nr in 2..150");
    MJ_REQUIRE(c->sNx >= 1 && c->sNy >= 1 && c->OL >= 0, "mj_gad_implicit_r_adjoint: bad tile layout");
    const int nx = c->sNx + 2 * c->OL, ny = c->sNy + 2 * c->OL;
    const int64_t plane = (int64_t)nx * ny, member = (int64_t)c->ntiles * c->nr * plane;
    MJ_REQUIRE(c->batch == 1 || (c->member_stride3d >= member && (c->mask_member_stride == 0 ||
                                                                  c->mask_member_stride >= member)),
               "mj_gad_implicit_r_adjoint: member strides smaller than one member's arrays");
    MJ_REQUIRE(kappaRX && recip_hFac && u && ubar && ybar && kappaRX_bar && g->maskC && g->dTtracerLev &&
                   g->recip_drF && g->recip_drC,
               "mj_gad_implicit_r_adjoint: null array or grid field");
    MJ_REQUIRE(!c->implicitAdvection || (wFld && wFld_bar && g->rA && g->recip_rA),
               "mj_gad_implicit_r_adjoint: implicit advection needs wFld, wFld_bar, rA, recip_rA");
    const double* ins[] = {kappaRX, recip_hFac, wFld, u, ubar, g->maskC};
    for (const double* p : ins)
        MJ_REQUIRE(p != ybar && p != kappaRX_bar && (!wFld_bar || p != wFld_bar),
                   "mj_gad_implicit_r_adjoint: an output aliases an input");
    ImprArgs a;
    a.T = c->ntiles;
    a.nx = nx;
    a.ny = ny;
    a.sNx = c->sNx;
    a.sNy = c->sNy;
    a.OL = c->OL;
    a.nr = c->nr;
    a.adv = c->implicitAdvection ? 1 : 0;
    a.plane = plane;
    a.ms3 = c->member_stride3d;
    a.mms = c->mask_member_stride;
    a.maskC = g->maskC;
    a.rA = g->rA;
    a.recip_rA = g->recip_rA;
    a.dt = g->dTtracerLev;
    a.rdrF = g->recip_drF;
    a.rdrC = g->recip_drC;
    a.rkSign = g->rkSign;
    a.kap = kappaRX;
    a.rh = recip_hFac;
    a.w = c->implicitAdvection ? wFld : kappaRX;
    a.y = nullptr;
    a.out = nullptr;
    hipStream_t st = as_stream(stream);
    const size_t lds = ((size_t)2 * c->nr * kImprThreads + 3 * (size_t)c->nr) * sizeof(double);
    using Kern = void (*)(ImprArgs, const double*, const double*, double*, double*, double*);
    const Kern kern = c->nr == 50 ? (a.adv ? impr_adjoint_kernel<true, 50> : impr_adjoint_kernel<false, 50>)
                                  : (a.adv ? impr_adjoint_kernel<true, 0> : impr_adjoint_kernel<false, 0>);
    if (lds > 65536)
        MJ_HIP(hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
    const int64_t cols = (int64_t)c->ntiles * plane;
    const dim3 grid((unsigned)((cols + kImprThreads - 1) / kImprThreads), (unsigned)c->batch);
    hipLaunchKernelGGL(kern, grid, dim3(kImprThreads), lds, st, a, u, ubar, ybar, kappaRX_bar,
                       a.adv ? wFld_bar : (double*)nullptr);
    MJ_HIP(hipGetLastError());
    return MJ_OK;
}
