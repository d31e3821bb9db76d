// GAD DST3 tracer advection on gfx950.
//
// Horizontal part: the reference's GAD_ADVECTION with implicitAdvection (pkgs/gad.py:460-539, gad_advection.F):
// three passes, each an X and a Y block whose action per tile comes from the facet pass table (which direction
// sweeps, overlap-only / interior-only update regions, FILL_CS_CORNER_TR_RL corner fills before/after the flux).
// Everything is tile-local, so one workgroup owns one (member, tile, level): the 98x98 FP64 working tracer
// (localTij) and the input tracer live in LDS (2 x 76.8 KB, gfx950's 160 KB LDS); each interface is evaluated once
// (twice in the small overlap sweeps), velocities and metrics are read once per sweep that needs them, and only the
// tendency is written. The reference evaluates all six flux arrays on every tile and
// masks; here each tile evaluates only the sweeps its table runs (2-3 of 6).
//
// Vertical part (R, only when wFld is given): a DST3 flux through the level interfaces applied after the
// horizontal passes, with the same non-divergent update form. It is not in the reference (which runs the vertical
// implicitly); its definition is written out at gad_vert_kernel.
#include <string.h>

#include <algorithm>

#include "mj_common.h"
#include "mj_internal.h"

namespace mj {

constexpr int GNY = 98, GNX = 98, GPLANE = GNY * GNX;  // LLC90 tiles with OL = 4

struct GadDev {
    int B, T, K, OLx, OLy, sNx, sNy;
    int64_t ms3, mms;
    const int32_t* mask_index;  // device [B]: mask slot of each member, or NULL (slot = member)
    int lpb;                    // levels per block of the horizontal launch (consecutive levels of one tile)
    const MjTilePlan* tiles;
    const double *dyG, *dxG, *recip_dxC, *recip_dyC, *recip_rA, *rA, *maskInC;
    const double *maskW, *maskS, *maskC;
    const double *dTlev, *drF, *recip_drF, *rhoFacC, *recip_rhoFacC, *deepFacC, *recip_deepFacC, *recip_deepFac2C,
        *recip_drC;
    double oneSixth;
    const double *u, *v, *w, *tr, *hFacW, *hFacS, *recip_hFacC;
    double* out;  // gTracer (no R flux) or localTij after the horizontal passes (R flux follows)
    const int32_t* nlev;
    unsigned* mbits;  // maskLocW / maskLocS bit planes per (mask slot, tile, level), gad_pre_kernel
    double2* g2;  // per tile, the 2-D metrics a sweep point reads, in pairs (gad_pre_kernel): [3][T][GPLANE]
                  // {dyG, recip_dxC} (X faces), {dxG, recip_dyC} (Y faces), {recip_rA, maskInC}
};

// Mask slot of member m: members of one level class share their grid masks.
__device__ __forceinline__ int64_t mask_slot(const GadDev& a, int m) { return a.mask_index ? a.mask_index[m] : m; }
// A bit plane in LDS: four words a row, bit i of a row in its word i / 32 (one column has the same shift in all rows). In
// memory its points follow one another (kPlaneBits words; a plane in rows would take 30 % more).
constexpr int kRowWords = 4, kMaskWords = GNY * kRowWords, kPlaneBits = 2 * ((GPLANE + 63) / 64);
static_assert(GNX > 96 && GNX < 32 * kRowWords, "words of a row");
// The bit planes of member m's masks at (tile t, level k): maskLocW's kPlaneBits words, then maskLocS's.
__device__ __forceinline__ const unsigned* unit_bits(const GadDev& a, int m, int t, int k) {
    const int64_t s = a.mms ? mask_slot(a, m) : 0;
    return a.mbits + ((s * a.T + t) * a.K + k) * 2 * kPlaneBits;
}
// Word i of a plane's rows, from the plane in memory.
__device__ __forceinline__ unsigned row_word(const unsigned* plane, int i) {
    const int w = i % kRowWords, bit = i / kRowWords * GNX + 32 * w;
    const unsigned v = __builtin_amdgcn_alignbit(plane[(bit >> 5) + 1], plane[bit >> 5], bit & 31);
    return w == kRowWords - 1 ? v & ((1u << (GNX - 96)) - 1) : v;
}
static_assert(((GNY - 1) * GNX + 96) / 32 + 1 < kPlaneBits, "the last row's words");

// maskLocW / maskLocS: maskW / maskS with FILL_CS_CORNER_UV_RS(.FALSE.) applied (gad.py:263-281, :489-490).
// (ia, ja) array indices; returns the corner-filled mask value at that point.
__device__ __forceinline__ double mask_loc(const GadDev& a, const MjTilePlan& tp, const double* mW, const double* mS,
                                           int ja, int ia, bool want_u) {
    const int fi = ia - a.OLx + 1, fj = ja - a.OLy + 1;  // Fortran indices
    const int sNx = a.sNx, sNy = a.sNy;
    auto at = [&](const double* f, int i, int j) { return f[(j - 1 + a.OLy) * GNX + (i - 1 + a.OLx)]; };
    if (fi <= 0 && fj <= 0 && tp.sw) {
        const int i = 1 - fi, j = 1 - fj;
        return want_u ? at(mS, 1 - j, 1 + i) : at(mW, 1 + j, 1 - i);
    }
    if (fi >= sNx + 1 && fj <= 0 && tp.se) {
        const int i = fi - sNx, j = 1 - fj;
        if (want_u) return i >= 2 ? at(mS, sNx + j, i) : at(mW, fi, fj);
        return at(mW, sNx + 1 - j, 1 - i);
    }
    if (fi <= 0 && fj >= sNy + 1 && tp.nw) {
        const int i = 1 - fi, j = fj - sNy;
        if (want_u) return at(mS, 1 - j, sNy + 1 - i);
        return j >= 2 ? at(mW, j, sNy + i) : at(mS, fi, fj);
    }
    if (fi >= sNx + 1 && fj >= sNy + 1 && tp.ne) {
        const int i = fi - sNx, j = fj - sNy;
        if (want_u) return i >= 2 ? at(mS, sNx + j, sNy + 2 - i) : at(mW, fi, fj);
        return j >= 2 ? at(mW, sNx + 2 - j, sNy + i) : at(mS, fi, fj);
    }
    return want_u ? at(mW, fi, fj) : at(mS, fi, fj);
}

// FILL_CS_CORNER_TR_RL(fill4dir, withSigns=.FALSE.) (gad.py:241-260): the (dst, src) pair of thread tid, for each
// corner present and i, j = 1..OL (false: no pair). Destinations are distinct, sources are distinct, and no
// source is a destination.
__device__ __forceinline__ bool corner_pair(const GadDev& a, const MjTilePlan& tp, int dir, int tid, int& dst,
                                            int& src) {
    const int OL = a.OLx;  // OLx == OLy checked on the host
    if (tid >= 4 * OL * OL) return false;
    const int c = tid / (OL * OL), r = tid - c * OL * OL;
    const int j = r / OL + 1, i = r % OL + 1;
    const int sNx = a.sNx, sNy = a.sNy;
    const bool on = c == 0 ? tp.sw : c == 1 ? tp.se : c == 2 ? tp.nw : tp.ne;
    if (!on) return false;
    int di, dj, si, sj;
    if (dir == 1) {
        if (c == 0) { di = 1 - i; dj = 1 - j; si = 1 - j; sj = i; }
        else if (c == 1) { di = sNx + i; dj = 1 - j; si = sNx + j; sj = i; }
        else if (c == 2) { di = 1 - i; dj = sNy + j; si = 1 - j; sj = sNy + 1 - i; }
        else { di = sNx + i; dj = sNy + j; si = sNx + j; sj = sNy + 1 - i; }
    } else {
        if (c == 0) { di = 1 - i; dj = 1 - j; si = j; sj = 1 - i; }
        else if (c == 1) { di = sNx + i; dj = 1 - j; si = sNx + 1 - j; sj = 1 - i; }
        else if (c == 2) { di = 1 - i; dj = sNy + j; si = j; sj = sNy + i; }
        else { di = sNx + i; dj = sNy + j; si = sNx + 1 - j; sj = sNy + i; }
    }
    dst = (dj - 1 + a.OLy) * GNX + (di - 1 + a.OLx);
    src = (sj - 1 + a.OLy) * GNX + (si - 1 + a.OLx);
    return true;
}

// The fill on a tile (LDS or the block's own global plane): all reads precede all writes.
__device__ __forceinline__ void corner_fill(double* loc, const GadDev& a, const MjTilePlan& tp, int dir, int tid) {
    for (int n0 = 0; n0 < 4 * a.OLx * a.OLx; n0 += blockDim.x) {
        int dst = -1, src = -1;
        double v = 0.0;
        const bool on = corner_pair(a, tp, dir, n0 + tid, dst, src);
        if (on) v = loc[src];
        __syncthreads();
        if (on) loc[dst] = v;
        __syncthreads();
    }
}

// Transpose of the fill on a cotangent plane: the destination's cotangent moves to its source.
__device__ __forceinline__ void corner_fill_T(double* bar, const GadDev& a, const MjTilePlan& tp, int dir, int tid) {
    for (int n0 = 0; n0 < 4 * a.OLx * a.OLx; n0 += blockDim.x) {
        int dst = -1, src = -1;
        double v = 0.0;
        const bool on = corner_pair(a, tp, dir, n0 + tid, dst, src);
        if (on) v = bar[dst];
        __syncthreads();
        if (on) {
            bar[src] = bar[src] + v;
            bar[dst] = 0.0;
        }
        __syncthreads();
    }
}

// Unit (tile, member, level block) of a DST3 launch of gridDim.x >= B*T*ceil(K/L) blocks (a multiple of 8, L =
// a.lpb levels per block): units ordered tile-major (tile, member, level block) and cut into 8 contiguous ranges, one
// per XCD (block b runs on XCD b % 8), so each XCD works through about T/8 tiles and their 2-D metrics stay in its L2
// across members and levels. k is the block's first level.
__device__ __forceinline__ bool gad_unit(const GadDev& a, int& t, int& m, int& k) {
    const int nkb = (a.K + a.lpb - 1) / a.lpb;
    const int n = a.B * a.T * nkb;
    const int chunk = (n + 7) / 8;
    const int pos = blockIdx.x / 8;
    const int u = (blockIdx.x % 8) * chunk + pos;
    if (pos >= chunk || u >= n) return false;
    k = (u % nkb) * a.lpb;
    const int tm = u / nkb;
    m = tm % a.B;
    t = tm / a.B;
    return true;
}

// The tables of a call. First maskLocW / maskLocS of every (mask slot, tile, level) as bit planes in global memory: the
// DST3 blocks of the members that share a slot load its words instead of the two mask planes (2 x 77 KB). The masks are 0/1
// by construction (hFac != 0), so a bit and its double 0.0/1.0 carry the same value. Off the four corner halo squares
// mask_loc is the plain mask, so every wave ballots rows of maskW / maskS, a pair of points a lane; then the points of the
// corner squares of the corners the tile has are set from mask_loc. Then, in the blocks behind them, the 2-D metrics in the
// pairs the sweeps load together (one 16-byte load instead of two 8-byte ones).
//
// Bound by HBM: one workgroup per mask plane, all its loads in flight at once. One member of 50 levels (100 MB) took 49 us
// with both planes in a workgroup of 256 threads and 16 words at a time, 38 us with single points, and the metrics 5 us in
// a launch of their own; 25 us together now (4 TB/s).
constexpr int kPreThreads = 512;
__device__ __forceinline__ unsigned spread16(unsigned x) {  // bit i to bit 2 i
    x = (x | x << 8) & 0x00ff00ffu;
    x = (x | x << 4) & 0x0f0f0f0fu;
    x = (x | x << 2) & 0x33333333u;
    return (x | x << 1) & 0x55555555u;
}
__global__ void __launch_bounds__(kPreThreads) gad_pre_kernel(GadDev a, int nplanes) {
    const int tid = threadIdx.x;
    if ((int)blockIdx.x >= nplanes) {
        const int64_t n = (int64_t)a.T * GPLANE, q = (int64_t)(blockIdx.x - nplanes) * kPreThreads + tid;
        if (q >= n) return;
        a.g2[q] = make_double2(a.dyG[q], a.recip_dxC[q]);
        a.g2[n + q] = make_double2(a.dxG[q], a.recip_dyC[q]);
        a.g2[2 * n + q] = make_double2(a.recip_rA[q], a.maskInC[q]);
        return;
    }
    __shared__ unsigned b[kMaskWords];
    const int u = blockIdx.x >> 1, want_u = !(blockIdx.x & 1);
    const int k = u % a.K, st = u / a.K, t = st % a.T, sl = st / a.T;
    const MjTilePlan& tp = a.tiles[t];
    const int64_t bm = sl * a.mms + ((int64_t)t * a.K + k) * GPLANE;
    const double *const mW = a.maskW + bm, *const mS = a.maskS + bm, *const mk = want_u ? mW : mS;
    const int lane = tid & 63, wave = tid >> 6;
    constexpr int NW = kPreThreads / 64, N = (GNY + NW - 1) / NW;  // rows of a wave
    static_assert(GNX % 2 == 0 && GNX / 2 <= 64, "a pair of points a lane");
    const bool on = lane < GNX / 2;
    double2 v[N];
    if (((uintptr_t)mk & 15) == 0) {
#pragma unroll
        for (int r = 0; r < N; ++r) {
            const int j = wave + r * NW;
            v[r] = on && j < GNY ? *(const double2*)(mk + j * GNX + 2 * lane) : make_double2(0.0, 0.0);
        }
    } else {
#pragma unroll
        for (int r = 0; r < N; ++r) {
            const int j = wave + r * NW;
            const double* const p = mk + j * GNX + 2 * lane;
            v[r] = on && j < GNY ? make_double2(p[0], p[1]) : make_double2(0.0, 0.0);
        }
    }
#pragma unroll
    for (int r = 0; r < N; ++r) {
        const int j = wave + r * NW;
        const unsigned long long e = __ballot(v[r].x != 0.0), o = __ballot(v[r].y != 0.0);
        if (lane < kRowWords && j < GNY)
            b[j * kRowWords + lane] = spread16((unsigned)(e >> (16 * lane)) & 0xffffu) |
                                      spread16((unsigned)(o >> (16 * lane)) & 0xffffu) << 1;
    }
    __syncthreads();
    // corner c (sw, se, nw, ne), point p of its OL x OL square
    const int OL = a.OLx, n = 4 * OL * OL;
    for (int r = tid; r < n; r += kPreThreads) {
        const int c = r / (OL * OL), pp = r % (OL * OL);
        const bool has = c == 0 ? tp.sw : c == 1 ? tp.se : c == 2 ? tp.nw : tp.ne;
        if (has) {
            const int dj = pp / OL, di = pp % OL;
            const int ja = (c < 2) ? dj : a.OLy + a.sNy + dj, ia = (c % 2 == 0) ? di : a.OLx + a.sNx + di;
            unsigned* word = b + ja * kRowWords + (ia >> 5);
            const unsigned bit = 1u << (ia & 31);
            if (mask_loc(a, tp, mW, mS, ja, ia, want_u) != 0.0)
                atomicOr(word, bit);
            else
                atomicAnd(word, ~bit);
        }
    }
    __syncthreads();
    unsigned* o = a.mbits + (int64_t)blockIdx.x * kPlaneBits;
    static_assert(kPlaneBits <= kPreThreads, "a word a thread");
    if (tid < kPlaneBits) {
        const int j = 32 * tid / GNX, c = 32 * tid % GNX, w = c >> 5;
        unsigned v = 0;
        if (j < GNY) {
            const unsigned* const row = b + j * kRowWords;
            v = __builtin_amdgcn_alignbit(w + 1 < kRowWords ? row[w + 1] : 0, row[w], c & 31);
            if (c > GNX - 32 && j + 1 < GNY) v |= row[kRowWords] << (GNX - c);
        }
        o[tid] = v;
    }
}

// Box point idx (row-major, width bw) of box B: array index.
template <class Box>
__device__ __forceinline__ int box_point(const Box& B, int bw, float inv_bw, int idx) {
    const int r = (int)(((float)idx + 0.5f) * inv_bw);  // idx / bw, exact for idx < 2^14 and bw <= 128
    return (B.j0 + r) * GNX + B.i0 + (idx - r * bw);
}

// The value of the next lane; `last` (uniform) in lane 63.
__device__ __forceinline__ double next_lane(double v, double last) {
    const int lo = __builtin_amdgcn_update_dpp(__double2loint(last), __double2loint(v), 0x130, 0xf, 0xf, false);
    const int hi = __builtin_amdgcn_update_dpp(__double2hiint(last), __double2hiint(v), 0x130, 0xf, 0xf, false);
    return __hiloint2double(hi, lo);
}
__device__ __forceinline__ double lane_value(double v, int lane) {
    return __hiloint2double(__builtin_amdgcn_readlane(__double2hiint(v), lane),
                            __builtin_amdgcn_readlane(__double2loint(v), lane));
}
// Bit p of b as 0.0 / 1.0.
__device__ __forceinline__ double bit01(unsigned b, int p) {
    return __hiloint2double((((int)(b << (31 - p))) >> 31) & 0x3ff00000, 0);
}
// Bits i - 1, i, i + 1 of a row of a bit plane (0 before its first).
__device__ __forceinline__ unsigned three_bits(const unsigned* row, int i) {
    const int w = max(i - 1, 0) >> 5;
    const unsigned long long v = ((unsigned long long)row[min(w + 1, kRowWords - 1)] << 32) | row[w];
    return (unsigned)((i > 0 ? v >> ((i - 1) & 31) : v << 1) & 7u);
}


// The plan of the block's tile is kept in LDS (a byte or half word of global memory is a vector load, and would wait for
// all loads issued before it). A sweep's entry, read uniformly; index s = 2 pass + dir.
constexpr int kSweepWords = sizeof(MjSweep) / 4, kPlanWords = sizeof(MjTilePlan) / 4;
static_assert(sizeof(MjSweep) == 20 && sizeof(MjTilePlan) == 124, "plan words");
struct HzBox {
    int i0, i1, j0, j1;
    __device__ __forceinline__ int points() const { return (i1 - i0) * (j1 - j0); }
    __device__ __forceinline__ bool has(int j, int i) const { return (i >= i0) & (i < i1) & (j >= j0) & (j < j1); }
};
struct HzSweep {
    int fill_before, fill_after;
    HzBox box[2];  // empty where the sweep has fewer
    __device__ __forceinline__ HzSweep(const MjTilePlan& lp, int s) {
        const int* w = (const int*)&lp + s * kSweepWords;
        auto u = [&](int i) { return __builtin_amdgcn_readfirstlane(w[i]); };
        const int f = u(0), nbox = f >> 24;
        fill_before = (f >> 8) & 0xff;
        fill_after = (f >> 16) & 0xff;
        for (int b = 0; b < 2; ++b) {
            const int i = u(1 + 2 * b), j = u(2 + 2 * b);
            box[b] = b < nbox ? HzBox{i & 0xffff, i >> 16, j & 0xffff, j >> 16} : HzBox{0, 0, 0, 0};
        }
    }
    __device__ __forceinline__ int points() const { return box[0].points() + box[1].points(); }
    // the rows j0 .. j0 + n - 1, the columns i0 .. i0 + n - 1: is one in a box's range?
    __device__ __forceinline__ bool rows(int j, int n) const {
        return ((j < box[0].j1) & (j + n > box[0].j0)) | ((j < box[1].j1) & (j + n > box[1].j0));
    }
    __device__ __forceinline__ bool cols(int i, int n) const {
        return ((i < box[0].i1) & (i + n > box[0].i0)) | ((i < box[1].i1) & (i + n > box[1].i0));
    }
    __device__ __forceinline__ bool has(int j, int i) const { return box[0].has(j, i) | box[1].has(j, i); }
};
// The next sweep from index s on that runs, 6: none.
__device__ __forceinline__ int next_sweep(const MjTilePlan& lp, int s) {
    while (s < 6 && !(__builtin_amdgcn_readfirstlane(((const int*)&lp)[s * kSweepWords]) & 0xff)) ++s;
    return s;
}

// The value of the lane before; `first` (uniform) in lane 0.
__device__ __forceinline__ double prev_lane(double v, double first) {
    const int lo = __builtin_amdgcn_update_dpp(__double2loint(first), __double2loint(v), 0x138, 0xf, 0xf, false);
    const int hi = __builtin_amdgcn_update_dpp(__double2hiint(first), __double2hiint(v), 0x138, 0xf, 0xf, false);
    return __hiloint2double(hi, lo);
}

// Element i of a plane: base in scalar registers, 32-bit offset.
template <class T>
__device__ __forceinline__ T ld(const T* p, int i) {
    return *(const T*)((const char*)p + (unsigned)(i * (int)sizeof(T)));
}

// Forms v here: the compiler would move the arithmetic behind all loads that follow, and spill what it reads.
__device__ __forceinline__ void pin(double& v) { asm volatile("" : "+v"(v)); }

// Element q + r GNX, r = 0 .. 13, of a plane: 32-bit offsets and an immediate (which ends at 4095 bytes).
__device__ __forceinline__ double plane8(const double* p, int q, int r) {
    const int c = r < 7 ? 3 : 10;
    return ((const double*)((const char*)p + (unsigned)(q + c * GNX) * 8))[(r - c) * GNX];
}
__device__ __forceinline__ double2 plane16(const double2* p, int q, int r) {
    const int c = r / 5 * 5 + 2;
    return ((const double2*)((const char*)p + (unsigned)(q + c * GNX) * 16))[(r - c) * GNX];
}
// A level's factor, in scalar registers.
__device__ __forceinline__ double level_value(const double* p, int k) {
    const double v = p[k];
    return __hiloint2double(__builtin_amdgcn_readfirstlane(__double2hiint(v)),
                            __builtin_amdgcn_readfirstlane(__double2loint(v)));
}

// One workgroup of 704 threads per (member, tile, level). Thread (seg, col) = (tid / 98, tid % 98) owns the rows 14 seg ..
// 14 seg + 13 of column col through all sweeps: the coefficient of its points' updates is formed once and stays in
// registers. A face's transport and interface value are evaluated once, by the owner of the point behind it: in X a point
// takes those of its other face from the lane of the next column (a DPP shift; the faces beside a wave's last lane are
// evaluated by its lanes 0 .. 13, a row each), in Y a thread walks down its rows and evaluates one face more, the first of
// the segment below. The values are those of one evaluation per face in a flux plane, in the same order of operations. A
// point keeps its increment in a register until every thread has read the tracer plane, and only then updates it. What a
// row reads from memory is loaded kHzAhead rows before it. LDS: the working plane, the input tracer (read by every update
// and by the output) and the mask bits, 156 KB.
//
// Sweeps with at most 1024 points (the overlap strips of passes 1 and 2) run one point a thread over the boxes, both faces
// evaluated by the point: on the columns 94 of 98 lanes would be idle there.
//
// Bound by HBM: a unit moves seven planes (540 KB, 28 us of a CU's share) and takes 37 us, of which some 4 are phases
// without loads; one member of 50 levels is 650 units on 256 CUs. Evaluating both faces at each of ten points a thread, all
// loads of a point behind one another, took 136 us for it (120 now) and 1700 us for 24 members of mixed level counts (1510
// now, 3.7 TB/s). One row ahead instead of two measured 3 % more for both, four 8 % more for the members. recip_rA and maskInC are
// read from their own planes, where half of a pair would be thrown away: a row's loads are 40 bytes instead of 48 (the whole
// step 152 -> 146 us and 3.05 -> 2.95 ms). maskInC as bits, 32 bytes, gave nothing more, nor did loading a sweep's first rows
// before the barriers in front of it (149 us).
constexpr int kHzRows = 14, kHzSegs = GNY / kHzRows, kHzThreads = 704, kHzSmall = 1024;
constexpr int kHzAhead = 2;
static_assert(kHzSegs * kHzRows == GNY && kHzSegs * GNX <= kHzThreads, "a thread per column and segment");

struct HzLds {
    double loc[GPLANE], trc[GPLANE];
    unsigned mlw[kMaskWords], mls[kMaskWords];
    MjTilePlan plan;
};

// One (member, tile, level) plane of the horizontal passes. SNAP: the state before the second, third, ... sweep goes to the
// planes at snap (the reverse mode's), and the result is written only if a.out is given.
template <bool SNAP>
__device__ __forceinline__ void hz_plane(const GadDev& a, int t, int m, int k, HzLds& S, double* snap) {
    constexpr int R = kHzRows, N = kHzAhead + 1;
    double *const loc = S.loc, *const trc = S.trc;
    int tid = threadIdx.x;
    const int64_t b3 = m * a.ms3 + ((int64_t)t * a.K + k) * GPLANE;
    const int64_t b2 = (int64_t)t * GPLANE;
    const double* const rhC = a.recip_hFacC + b3;
    const double2* const am = a.g2 + 2 * (int64_t)a.T * GPLANE + b2;  // {recip_rA, maskInC}
    const double *const rrA = a.recip_rA + b2, *const mIn = a.maskInC + b2;
    const double dt = level_value(a.dTlev, k), deepFacC = level_value(a.deepFacC, k), rdeepC = level_value(a.recip_deepFacC, k);
    const double rdeep2C = level_value(a.recip_deepFac2C, k), rhoFacC = level_value(a.rhoFacC, k);
    const double rrhoFacC = level_value(a.recip_rhoFacC, k), drF = level_value(a.drF, k), rdrF = level_value(a.recip_drF, k);
    const double oneSixth = a.oneSixth;
    const bool own = tid < kHzSegs * GNX;
    const int seg = own ? tid / GNX : 0;
    int col = own ? tid - seg * GNX : 0, j0 = seg * R, q0 = j0 * GNX + col;
    auto at8 = [&](const double* p, int r) { return plane8(p, q0, r); };
    // X: lane r has row r of the point behind the wave's last lane
    int qe;
    {
        const int lane = tid & 63, te = (tid | 63) + 1, sege = te / GNX;
        const bool edge = lane < R && te < kHzSegs * GNX;
        qe = edge ? (sege * R + lane) * GNX + te - sege * GNX : q0;
    }
    auto trans = [&](double V, double G, double H) { return V * (G * deepFacC * drF * H) * rhoFacC; };
    // interface value (gad.py:482-485 transport; 0 outside the Fortran flux loops i = 1-OLx+2 .. sNx+OLx-1,
    // gad_dst3_adv_x.F:80, and j = 1-OLy+2 .. sNy+OLy-1, gad_dst3_adv_y.F:78); bits from bit p on: the masks of the faces
    // before, at and behind it
    auto flux = [&](bool in, double T, double V, double rd, double t_m2, double t_m1, double t_0, double t_p1,
                    unsigned bits, int p) {
        const double Dm1 = (t_m1 - t_m2) * bit01(bits, p), D0 = (t_0 - t_m1) * bit01(bits, p + 1),
                     Dp1 = (t_p1 - t_0) * bit01(bits, p + 2);
        const double f = dst3_flux_r(T, fabs(V * dt * rd * rdeepC), oneSixth, t_m1, t_0, Dm1, D0, Dp1);
        return in ? f : 0.0;
    };
    double coef[R];
    {
        const double* const tr = a.tr + b3;
        double tv[R], rh[R], ra[R];
        const int pw = tid < kPlanWords ? ((const int*)&a.tiles[t])[tid] : 0;
        static_assert(kMaskWords <= kHzThreads, "a word of each plane per thread");
        const unsigned* gb = unit_bits(a, m, t, k);
        const int wi = min(tid, kMaskWords - 1);
        const unsigned w0 = row_word(gb, wi), w1 = row_word(gb + kPlaneBits, wi);
#pragma unroll
        for (int r = 0; r < R; ++r) {
            tv[r] = at8(tr, r);
            rh[r] = at8(rhC, r);
            ra[r] = at8(rrA, r);
        }
        if (tid < kPlanWords) ((int*)&S.plan)[tid] = pw;
        if (tid < kMaskWords) S.mlw[tid] = w0, S.mls[tid] = w1;
#pragma unroll
        for (int r = 0; r < R; ++r) {
            coef[r] = dt * rrhoFacC * rh[r] * rdrF * ra[r] * rdeep2C;  // gad.py:494
            pin(coef[r]);
        }
        if (own) {
#pragma unroll
            for (int r = 0; r < R; ++r) loc[q0 + r * GNX] = trc[q0 + r * GNX] = tv[r];
        }
    }
    __syncthreads();
    // masks of the thread's Y faces: rows j0 - 1 .. j0 + R + 1
    unsigned my = 0;
#pragma unroll
    for (int r = 0; r < R + 3; ++r)
        my |= (S.mls[max(min(j0 - 1 + r, GNY - 1), 0) * kRowWords + (col >> 5)] >> (col & 31) & 1u) << r;
    int ns = 0;
    for (int s = next_sweep(S.plan, 0); s < 6;) {
        // positions and masks made anew for each sweep: the compiler would keep all that is derived from them in registers
        asm volatile("" : "+v"(tid), "+v"(q0), "+v"(col), "+v"(j0), "+v"(qe), "+v"(my));
        const int dir = s & 1;
        const HzSweep P(S.plan, s);
        const int npt = P.points();
        const double* const vel = (dir == 0 ? a.u : a.v) + b3;
        const double* const hf = (dir == 0 ? a.hFacW : a.hFacS) + b3;
        const double2* const gr = a.g2 + dir * (int64_t)a.T * GPLANE + b2;  // {dyG|dxG, recip_dxC|dyC}
        struct RowIn {
            double V, H, MI;
            double2 G;
        } in[N];
        if (P.fill_before) corner_fill(loc, a, S.plan, P.fill_before, tid);
        // local - coef*(d(af) - tracer*d(trans))*maskInC (gad.py:511-514)
        if (npt <= kHzSmall) {
            const int d = dir == 0 ? 1 : GNX;
            constexpr int C = (kHzSmall + kHzThreads - 1) / kHzThreads;
            double inc[C];
            int qq[C];
#pragma unroll
            for (int n = 0; n < C; ++n) {
                const int idx = tid + n * kHzThreads;
                if (idx >= npt) continue;
                const int n0 = P.box[0].points(), bw0 = P.box[0].i1 - P.box[0].i0, bw1 = P.box[1].i1 - P.box[1].i0;
                const int q = idx < n0 ? box_point(P.box[0], bw0, 1.0f / (float)max(bw0, 1), idx)
                                       : box_point(P.box[1], bw1, 1.0f / (float)max(bw1, 1), idx - n0);
                qq[n] = q;
                const double2 G0 = ld(gr, q), G1 = ld(gr, q + d), A = ld(am, q);
                const double V0 = ld(vel, q), H0 = ld(hf, q), V1 = ld(vel, q + d), H1 = ld(hf, q + d), RH = ld(rhC, q);
                const unsigned* mb = dir == 0 ? S.mlw : S.mls;
                const int j = q / GNX, i = q - j * GNX, c = dir == 0 ? i : j, cmax = (dir == 0 ? GNX : GNY) - 2;
                const double T0 = trans(V0, G0.x, H0), T1 = trans(V1, G1.x, H1);
                auto at = [&](int o) { return loc[max(min(q + o * d, GPLANE - 1), 0)]; };
                auto bit = [&](int o) {
                    const int jb = min(max(j + (dir == 0 ? 0 : o), 0), GNY - 1), ib = min(max(i + (dir == 0 ? o : 0), 0), GNX - 1);
                    return (mb[jb * kRowWords + (ib >> 5)] >> (ib & 31)) & 1u;
                };
                const unsigned bits = bit(-1) | bit(0) << 1 | bit(1) << 2 | bit(2) << 3;
                const double f0 = flux(c >= 2 && c <= cmax, T0, V0, G0.y, at(-2), at(-1), at(0), at(1), bits, 0);
                const double f1 = flux(c + 1 >= 2 && c + 1 <= cmax, T1, V1, G1.y, at(-1), at(0), at(1), at(2), bits, 1);
                const double daf = f1 - f0, dtr = T1 - T0, cf = dt * rrhoFacC * RH * rdrF * A.x * rdeep2C;
                inc[n] = cf * (daf - trc[q] * dtr) * A.y;
            }
            __syncthreads();  // every read of the plane precedes the updates
            if (P.fill_after) corner_fill(loc, a, S.plan, P.fill_after, tid);
#pragma unroll
            for (int n = 0; n < C; ++n)
                if (tid + n * kHzThreads < npt) loc[qq[n]] = loc[qq[n]] - inc[n];
        } else {
            double inc[R];
            if (dir == 0) {
                auto load = [&](int r) {
                    if (r < R) in[r % N] = RowIn{at8(vel, r), at8(hf, r), at8(mIn, r), plane16(gr, q0, r)};
                };
                const double Ve = ld(vel, qe), He = ld(hf, qe);
                const double2 Ge = ld(gr, qe);
#pragma unroll
                for (int r = 0; r < kHzAhead; ++r) load(r);
                const int je = qe / GNX, ie = qe - je * GNX;  // columns 0, 1 and 97 have no flux: their lanes read beside them
                const double* const le = loc + max(min(qe, GPLANE - 2), 2);
                const double Te = trans(Ve, Ge.x, He);
                const double fe = flux(ie >= 2 && ie <= GNX - 2, Te, Ve, Ge.y, le[-2], le[-1], le[0], le[1],
                                       three_bits(S.mlw + je * kRowWords, ie), 0);
                const bool inx = col >= 2 && col <= GNX - 2;
                const double* const l0 = loc + j0 * GNX + max(min(col, GNX - 2), 2);
#pragma unroll
                for (int r = 0; r < R; ++r) {
                    __builtin_amdgcn_sched_barrier(0);
                    load(r + kHzAhead);
                    const RowIn I = in[r % N];
                    const double* const l = l0 + r * GNX;
                    const double T0 = trans(I.V, I.G.x, I.H);
                    const double f0 = flux(inx, T0, I.V, I.G.y, l[-2], l[-1], l[0], l[1],
                                           three_bits(S.mlw + (j0 + r) * kRowWords, col), 0);
                    const double f1 = next_lane(f0, lane_value(fe, r)), T1 = next_lane(T0, lane_value(Te, r));
                    const double daf = f1 - f0, dtr = T1 - T0;
                    inc[r] = coef[r] * (daf - trc[q0 + r * GNX] * dtr) * I.MI;
                    pin(inc[r]);
                }
            } else {
                // rows beside the thread's own
                auto beside = [&](int r) { return max(min(j0 + r, GNY - 1), 0) * GNX + col; };
                auto lds = [&](int r) { return r >= 0 && r < R ? loc[q0 + r * GNX] : loc[beside(r)]; };
                auto load = [&](int r) {
                    if (r < R)
                        in[r % N] = RowIn{at8(vel, r), at8(hf, r), at8(mIn, r), plane16(gr, q0, r)};
                    else if (r == R)
                        in[r % N] = RowIn{ld(vel, beside(r)), ld(hf, beside(r)), 0.0, ld(gr, beside(r))};
                };
#pragma unroll
                for (int r = 0; r < kHzAhead; ++r) load(r);
                double tm2 = lds(-2), tm1 = lds(-1), t0 = lds(0), T0 = 0.0, f0 = 0.0, MI = 0.0;
#pragma unroll
                for (int r = 0; r <= R; ++r) {
                    __builtin_amdgcn_sched_barrier(0);
                    load(r + kHzAhead);
                    const RowIn I = in[r % N];
                    const double tp1 = lds(r + 1);
                    const double T1 = trans(I.V, I.G.x, I.H);
                    const double f1 = flux(j0 + r >= 2 && j0 + r <= GNY - 2, T1, I.V, I.G.y, tm2, tm1, t0, tp1, my, r);
                    if (r > 0) {
                        const double daf = f1 - f0, dtr = T1 - T0;
                        inc[r - 1] = coef[r - 1] * (daf - trc[q0 + (r - 1) * GNX] * dtr) * MI;
                        pin(inc[r - 1]);
                    }
                    tm2 = tm1, tm1 = t0, t0 = tp1, T0 = T1, f0 = f1, MI = I.MI;
                }
            }
            __syncthreads();  // every read of the plane precedes the updates
            if (P.fill_after) corner_fill(loc, a, S.plan, P.fill_after, tid);
            if (own) {
#pragma unroll
                for (int r = 0; r < R; ++r) {
                    const double l = loc[q0 + r * GNX];
                    loc[q0 + r * GNX] = P.has(j0 + r, col) ? l - inc[r] : l;
                }
            }
        }
        __syncthreads();
        s = next_sweep(S.plan, s + 1);
        if (SNAP && s < 6 && own) {
            double* const sp = snap + (size_t)ns * GPLANE;
#pragma unroll
            for (int r = 0; r < R; ++r) sp[q0 + r * GNX] = loc[q0 + r * GNX];
            ++ns;
        }
    }
    if (!own || (SNAP && !a.out)) return;
    double* const out = a.out + b3;
    if (a.w) {
#pragma unroll
        for (int r = 0; r < R; ++r) out[q0 + r * GNX] = loc[q0 + r * GNX];
    } else {
#pragma unroll
        for (int r = 0; r < R; ++r) out[q0 + r * GNX] = (loc[q0 + r * GNX] - trc[q0 + r * GNX]) / dt;  // gad.py:539
    }
}

// The plane as a call of its own (the multi-level blocks: inlined into the level loop it spills registers).
__device__ __noinline__ void hz_plane_call(const GadDev& a, int t, int m, int k, HzLds& S) {
    hz_plane<false>(a, t, m, k, S, nullptr);
}

// One workgroup per (member, tile, level block): LEVELS false, one level per block (a.lpb == 1); true, a.lpb
// consecutive levels, one after the other in the same LDS planes.
template <bool LEVELS>
__global__ void __launch_bounds__(kHzThreads, 3) gad_hz_kernel(GadDev a) {
    __shared__ HzLds S;
    int t, m, k0;
    if (!gad_unit(a, t, m, k0)) return;
    if (!LEVELS) {
        if (a.nlev && k0 >= a.nlev[m]) return;
        hz_plane<false>(a, t, m, k0, S, nullptr);
        return;
    }
    const int kend = min(k0 + a.lpb, a.nlev ? min(a.nlev[m], a.K) : a.K);
    for (int k = k0; k < kend; ++k) {
        if (k > k0) __syncthreads();  // the previous level's output has read the LDS planes
        hz_plane_call(a, t, m, k, S);
    }
}

// ------------------------------------------------------------------------------------------------ reverse mode
constexpr int kAdjChunk = 1024;  // (member, tile, level)s per reverse launch, in whole columns (at least one)
constexpr int kAdjSnaps = 5;     // snapshots of one: six sweeps, the first from the tracer itself
constexpr int kAdjPlanes = 7;    // planes of one in the workspace query's answer, which callers know; kAdjSnaps are used
// Partial derivatives of one DST3 interface value f = A (t_m1 + d0 Rj + d1 Rjm) + Bm (t_0 - d0 Rj - d1 Rjp)
// (A = (tr + |tr|)/2, Bm = (tr - |tr|)/2, d0 = (2-c)(1-c)/6, d1 = (1-c^2)/6): w[0..3] = df/dt_m2, df/dt_m1,
// df/dt_0, df/dt_p1 (independent of the tracer), dtr = df/dtr, dc = df/dcfl. The derivative of |x| at 0 is taken
// as 0 (sign(0) = 0), which is what a central difference across x = 0 gives.
struct FluxPartials {
    double w[4], dtr, dc;
};
__device__ __forceinline__ FluxPartials dst3_partials(double tr_, double cfl, double oneSixth, double t_m2,
                                                      double t_m1, double t_0, double t_p1, double m_m1, double m_0,
                                                      double m_p1) {
    const double Rjp = (t_p1 - t_0) * m_p1;
    const double Rj = (t_0 - t_m1) * m_0;
    const double Rjm = (t_m1 - t_m2) * m_m1;
    const double d0 = (2. - cfl) * (1. - cfl) * oneSixth;
    const double d1 = (1. - cfl * cfl) * oneSixth;
    const double A = 0.5 * (tr_ + fabs(tr_)), Bm = 0.5 * (tr_ - fabs(tr_));
    const double sg = tr_ > 0.0 ? 1.0 : (tr_ < 0.0 ? -1.0 : 0.0);
    FluxPartials P;
    P.w[0] = -A * d1 * m_m1;
    P.w[1] = A * (1.0 - d0 * m_0 + d1 * m_m1) + Bm * (d0 * m_0);
    P.w[2] = A * (d0 * m_0) + Bm * (1.0 - d0 * m_0 + d1 * m_p1);
    P.w[3] = -Bm * d1 * m_p1;
    const double Pv = t_m1 + (d0 * Rj + d1 * Rjm), Nv = t_0 - (d0 * Rj + d1 * Rjp);
    P.dtr = 0.5 * (1.0 + sg) * Pv + 0.5 * (1.0 - sg) * Nv;
    const double d0c = (2.0 * cfl - 3.0) * oneSixth, d1c = -2.0 * cfl * oneSixth;
    P.dc = A * (d0c * Rj + d1c * Rjm) - Bm * (d0c * Rj + d1c * Rjp);
    return P;
}

// Unit of a reverse launch: n (member, tile, level)s from u0 on, level fastest, cut into 8 contiguous ranges, one per XCD
// (gad_unit's reason). i: its number in the launch.
__device__ __forceinline__ bool adj_unit(const GadDev& a, int u0, int n, int& i, int& t, int& m, int& k) {
    const int chunk = (n + 7) / 8, pos = blockIdx.x / 8;
    i = (blockIdx.x % 8) * chunk + pos;
    if (pos >= chunk || i >= n) return false;
    k = (u0 + i) % a.K;
    const int mt = (u0 + i) / a.K;
    t = mt % a.T;
    m = mt / a.T;
    return true;
}

// The forward sweeps for the reverse mode: snapshots, and localTij at a.out if given.
__global__ void __launch_bounds__(kHzThreads, 3) gad_hz_snap_kernel(GadDev a, int u0, int n, double* snap) {
    __shared__ HzLds S;
    int i, t, m, k;
    if (!adj_unit(a, u0, n, i, t, m, k)) return;
    if (a.nlev && k >= a.nlev[m]) return;
    hz_plane<true>(a, t, m, k, S, snap + (size_t)i * kAdjSnaps * GPLANE);
}

// Reverse mode of gad_hz_kernel (horizontal DST3 without R flux) for one (member, tile, level): given the cotangent gbar
// of gTracer, writes the cotangents of the tracer, uFld and vFld planes (every padded point; the grid, hFac and mask inputs
// are treated as constants). The sweeps are reversed, each from the snapshot of the tile before it: the box update (af,
// tracer and transport terms), the corner fill after the flux, the flux (weights of the four tracer values, transport and
// CFL terms), the corner fill before it.
//
// With lbar (the R flux's reverse mode) the sweeps start from lbar, the cotangent of localTij after the horizontal passes,
// instead of from gbar, and the tracer cotangent already holds the vertical part (added to, not set).
//
// Thread (seg, col) = (tid / 98, tid % 98) owns the rows 14 seg .. 14 seg + 13 of column col. Every face's partials are
// evaluated once, by its owner: in X the four points that they go to take them from the lanes beside (DPP shifts; the three
// faces beside a wave's 64 points are evaluated by lanes 3 r + 0 .. 2 for row r), in Y a thread walks up its column and
// evaluates the faces of three rows more. The update's cotangents are formed from localTij's cotangent before a barrier,
// which is then updated in place behind it. LDS: the tile and that cotangent, 154 KB, one workgroup of 11 waves a CU.
//
// What a row reads from memory is loaded a row ahead, and no row has a branch: the loads of all rows issued together spill,
// and a load issued behind a row's stores waits for them too (both count in order). Bound by HBM (one
// member of 50 levels moves 1.13 GB, 22 planes of 77 KB a unit of two or three sweeps, at 3.9 TB/s) and the rounds of its
// 650 units on 256 CUs, the last one half empty.
//
// Evaluating all five partials that a point needs, with a second flux plane and no more than a point's loads in flight,
// took 958 us for one member of 50 levels together with the replay of the forward sweeps (two of three, each with a
// snapshot); 291 us now, and 128 us for the replay, whose launch with the R flux also makes the localTij that took another
// 136 us. Ten rows a thread (1024 threads, 128 VGPRs) and twenty (512, 256) measured 540 to 560 us in the form without the
// loads ahead, as did fourteen; two rows ahead spill (400 us).
constexpr int kAdjRows = 14, kAdjSegs = GNY / kAdjRows, kAdjThreads = 704;
static_assert(kAdjSegs * kAdjRows == GNY && kAdjSegs * GNX <= kAdjThreads && 3 * kAdjRows <= 64, "a thread per column and segment, a lane per edge face");

struct AdjLds {
    double loc[GPLANE], lb[GPLANE];
    unsigned mlw[kMaskWords], mls[kMaskWords];
    MjTilePlan plan;
};

__global__ void __launch_bounds__(kAdjThreads, 3)
    gad_hz_adjoint_kernel(GadDev a, const double* gbar, double* trb, double* ub, double* vb, const double* snap, int u0,
                          int n, const double* lbar) {
    constexpr int R = kAdjRows;
    __shared__ AdjLds S;
    int unit, t, m, k;
    if (!adj_unit(a, u0, n, unit, t, m, k)) return;
    int tid = threadIdx.x;
    const int64_t b3 = m * a.ms3 + ((int64_t)t * a.K + k) * GPLANE;
    const bool own = tid < kAdjSegs * GNX;
    const int seg = own ? tid / GNX : 0;
    int col = own ? tid - seg * GNX : 0, j0 = seg * R;
    int q0 = j0 * GNX + col;
    double *const TB = trb + b3, *const UB = ub + b3, *const VB = vb + b3;
    if (a.nlev && k >= a.nlev[m]) {  // no dependence: zero cotangents
        for (int r = 0; own && r < R; ++r) TB[q0 + r * GNX] = UB[q0 + r * GNX] = VB[q0 + r * GNX] = 0.0;
        return;
    }
    const int64_t b2 = (int64_t)t * GPLANE;
    const double *const tr = a.tr + b3, *const rhC = a.recip_hFacC + b3;
    const double2* const am = a.g2 + 2 * (int64_t)a.T * GPLANE + b2;  // {recip_rA, maskInC}
    const double dt = level_value(a.dTlev, k), deepFacC = level_value(a.deepFacC, k), rdeepC = level_value(a.recip_deepFacC, k);
    const double rdeep2C = level_value(a.recip_deepFac2C, k), rhoFacC = level_value(a.rhoFacC, k), rrhoFacC = level_value(a.recip_rhoFacC, k);
    const double drF = level_value(a.drF, k), rdrF = level_value(a.recip_drF, k), oneSixth = a.oneSixth;
    snap += (size_t)unit * kAdjSnaps * GPLANE;
    auto update_coef = [&](double RH, double2 AM) { return dt * rrhoFacC * RH * rdrF * AM.x * rdeep2C * AM.y; };

    auto at8 = [&](const double* p, int q, int r) { return plane8(p, q, r); };
    auto at16 = [&](const double2* p, int q, int r) { return plane16(p, q, r); };
    {
        double x[R];
#pragma unroll
        for (int r = 0; r < R; ++r) x[r] = at8(lbar ? lbar + b3 : gbar + b3, q0, r);
        if (!lbar) {
#pragma unroll
            for (int r = 0; r < R; ++r) x[r] = x[r] / dt;
        }
        if (own) {
#pragma unroll
            for (int r = 0; r < R; ++r) S.lb[q0 + r * GNX] = x[r];
            if (!lbar) {
#pragma unroll
                for (int r = 0; r < R; ++r) TB[q0 + r * GNX] = -x[r];
            }
        }
        const unsigned* gb = unit_bits(a, m, t, k);
        static_assert(kMaskWords <= kAdjThreads, "a word of each plane per thread");
        if (tid < kMaskWords) {
            S.mlw[tid] = row_word(gb, tid);
            S.mls[tid] = row_word(gb + kPlaneBits, tid);
        }
        if (tid < kPlanWords) ((int*)&S.plan)[tid] = ((const int*)&a.tiles[t])[tid];
    }
    __syncthreads();
    // masks of the Y faces of the thread's column: rows j0 - 2 .. j0 + R + 2, from bit 0 on
    unsigned my = 0;
#pragma unroll
    for (int r = -2; r < R + 3; ++r)
        my |= (S.mls[max(min(j0 + r, GNY - 1), 0) * kRowWords + (col >> 5)] >> (col & 31) & 1u) << (r + 2);
    int left = 0;  // sweeps to reverse
    for (int s = 0; s < 6; ++s) left += next_sweep(S.plan, s) == s;
    bool first[2] = {true, true};  // no cotangent of this velocity written yet
    for (int s = 5; s >= 0; --s) {
        if (next_sweep(S.plan, s) != s) continue;
        --left;
        // positions made anew for each sweep: the compiler would keep every address derived from them in registers
        asm volatile("" : "+v"(tid), "+v"(q0), "+v"(col), "+v"(j0), "+v"(my));
        const int dir = s & 1, lane = tid & 63;
        const HzSweep P(S.plan, s);
        const double* const sn = left ? snap + (size_t)(left - 1) * GPLANE : tr;
        const double* const vel = (dir == 0 ? a.u : a.v) + b3;
        const double* const hf = (dir == 0 ? a.hFacW : a.hFacS) + b3;
        const double2* const gr = a.g2 + dir * (int64_t)a.T * GPLANE + b2;  // {dyG|dxG, recip_dxC|dyC}
        double* const vbar = dir == 0 ? UB : VB;
        const bool init = dir == 0 ? first[0] : first[1];
        if (dir == 0) first[0] = false; else first[1] = false;
        // box update: loc[q] -= c_q (af[q+d] - af[q] - tr[q] (T[q+d] - T[q])), c_q = coef(q) maskInC(q); cg: the cotangent
        // c_q lb[q] of the increment, 0 off the boxes
        auto update_bar = [&](bool in, double c, double lb) {
            double x = c * lb;
            pin(x);  // else the loads move behind a branch, one after the other
            return in ? x : 0.0;
        };
        // a face whose interface value has the cotangent g: c[0..3] to the tracer values q - 2d .. q + d, vv to the velocity
        // (its transport T = V L rhoFacC); bits from bit p on: the masks of the faces before, at and behind it
        auto face = [&](bool in, double g, double V, double L, double T, double rd, double tm2, double tm1, double t0,
                        double tp1, unsigned bits, int p, double (&c)[4], double& vv) {
            const double arg = V * dt * rd * rdeepC;
            const FluxPartials F = dst3_partials(T, fabs(arg), oneSixth, tm2, tm1, t0, tp1, bit01(bits, p),
                                                 bit01(bits, p + 1), bit01(bits, p + 2));
            const bool act = in && g != 0.0;
            const double sgn = arg > 0.0 ? 1.0 : (arg < 0.0 ? -1.0 : 0.0);
#pragma unroll
            for (int i = 0; i < 4; ++i) c[i] = act ? F.w[i] * g : 0.0;
            vv = act ? (F.dtr * g) * (L * rhoFacC) + (F.dc * g) * (sgn * dt * rd * rdeepC) : 0.0;
        };
        // the velocity's cotangent at row r: the transport's tb, then the flux part; o: what is there from a sweep before
        auto put_vel = [&](int r, double tb, double L, double vv, double o) {
            const double x = tb != 0.0 ? tb * (L * rhoFacC) : 0.0, b = init ? 0.0 : o;
            vbar[q0 + r * GNX] = (b + x) + vv;
        };
        const double* const old = init ? vel : vbar;  // not looked at when there is nothing yet
        // ---- before the barrier: the tile, the update's cotangents of the thread's rows (in Y of two more on each side)
        // and in X of the points beside the wave
        // strips: most wavefronts (X) or lanes (Y, whose columns have nothing to do with each other) have no point of them
        const bool act = dir == 0 ? __any(P.rows(j0, R)) : P.cols(col, 1);
        auto beside = [&](int r) { return max(min(j0 + r, GNY - 1), 0) * GNX + col; };  // rows beside the thread's own
        auto at = [&](const double* p, int r) { return r >= 0 && r < R ? at8(p, q0, r) : ld(p, beside(r)); };
        auto at2 = [&](const double2* p, int r) { return r >= 0 && r < R ? at16(p, q0, r) : ld(p, beside(r)); };
        auto lds = [&](int r) { return r >= 0 && r < R ? q0 + r * GNX : beside(r); };
        // X: lane 3 r + f has row r of the point before the wave's first (f = 0), of the two behind its last (1, 2)
        const int er = lane / 3, ef = lane - er * 3, te = ef == 0 ? (tid & ~63) - 1 : (tid | 63) + ef;
        const bool edge = er < R && te >= 0 && te < kAdjSegs * GNX;
        const int eseg = edge ? te / GNX : 0, ei = edge ? te - eseg * GNX : 0, ej = edge ? eseg * R + er : 0;
        const int eq = ej * GNX + ei, em = max(eq - 1, 0);
        double cg[R + 4], ecg = 0.0, ecm = 0.0;
        unsigned inb = 0;  // bit r + 2: row r is in a box
        {
            double sv[R];
#pragma unroll
            for (int r = 0; r < R; ++r) sv[r] = at8(sn, q0, r);
            if (act) {
                double RH[R];
                double2 A[R];
#pragma unroll
                for (int r = 0; r < R; ++r) {
                    RH[r] = at8(rhC, q0, r);
                    A[r] = at16(am, q0, r);
                }
#pragma unroll
                for (int r = 0; r < R; ++r) {
                    const bool inp = P.has(j0 + r, col);
                    inb |= (unsigned)inp << (r + 2);
                    cg[r + 2] = update_bar(inp, update_coef(RH[r], A[r]), S.lb[q0 + r * GNX]);
                    pin(cg[r + 2]);
                }
                if (dir == 0) {
                    ecg = update_bar(edge & P.has(ej, ei), update_coef(ld(rhC, eq), ld(am, eq)), S.lb[eq]);
                    ecm = update_bar(edge & (ei > 0) & P.has(ej, ei - 1), update_coef(ld(rhC, em), ld(am, em)), S.lb[em]);
                } else {
#pragma unroll
                    for (int i = 0; i < 4; ++i) {
                        const int r = i < 2 ? i - 2 : R + i - 2;
                        const bool inp = (j0 + r >= 0) & P.has(j0 + r, col);
                        inb |= (unsigned)inp << (r + 2);
                        cg[r + 2] = update_bar(inp, update_coef(at(rhC, r), at2(am, r)), S.lb[lds(r)]);
                    }
                }
            }
            if (own) {
#pragma unroll
                for (int r = 0; r < R; ++r) S.loc[q0 + r * GNX] = sv[r];
            }
        }
        __syncthreads();  // the tile is loaded; every read of the cotangent precedes its updates
        if (P.fill_before) corner_fill(S.loc, a, S.plan, P.fill_before, tid);
        if (P.fill_after) corner_fill_T(S.lb, a, S.plan, P.fill_after, tid);
        // ---- the faces; what a row reads is loaded kAhead rows before it
        constexpr int kAhead = 1;
        struct RowIn {
            double V, H, TR, old, tb;
            double2 G;
        } in[kAhead + 1];
        if (dir == 0 && act) {
            double ec[4], eT, ect;
            {
                const double* const l = S.loc + max(min(eq, GPLANE - 2), 2);
                const double2 G = ld(gr, eq);
                const double V = ld(vel, eq), L = G.x * deepFacC * drF * ld(hf, eq);
                double vv;
                eT = V * L * rhoFacC;
                ect = ecg * ld(tr, eq);
                pin(ect);
                ect = edge & P.has(ej, ei) ? ect : 0.0;
                face(edge && ei >= 2 && ei <= GNX - 2, ecg - ecm, V, L, eT, G.y, l[-2], l[-1], l[0], l[1],
                     three_bits(S.mlw + ej * kRowWords, ei), 0, ec, vv);
            }
            auto load = [&](int r) {
                if (r < R) in[r % (kAhead + 1)] = RowIn{at8(vel, q0, r), at8(hf, q0, r), at8(tr, q0, r),
                                                           at8(old, q0, r), at8(TB, q0, r), at16(gr, q0, r)};
            };
#pragma unroll
            for (int r = 0; r < kAhead; ++r) load(r);
            const bool inx = col >= 2 && col <= GNX - 2;  // columns 0, 1 and 97 have no flux: they read beside them
            const double* const l0 = S.loc + j0 * GNX + max(min(col, GNX - 2), 2);
            if (own) {
#pragma unroll
                for (int r = 0; r < R; ++r) {
                    __builtin_amdgcn_sched_barrier(0);
                    load(r + kAhead);
                    const int q = q0 + r * GNX;
                    const RowIn I = in[r % (kAhead + 1)];
                    const double L = I.G.x * deepFacC * drF * I.H, T = I.V * L * rhoFacC, g = cg[r + 2];
                    const bool inp = inb >> (r + 2) & 1;
                    const double ct = inp ? g * I.TR : 0.0;
                    const double cm = prev_lane(g, lane_value(ecg, 3 * r)), cmt = prev_lane(ct, lane_value(ect, 3 * r));
                    const double* const l = l0 + r * GNX;
                    double c[4], vv;
                    face(inx, g - cm, I.V, L, T, I.G.y, l[-2], l[-1], l[0], l[1],
                         three_bits(S.mlw + (j0 + r) * kRowWords, col), 0, c, vv);
                    // to this point from the faces q + 2, q + 1, q, q - 1
                    const double c0 =
                        next_lane(next_lane(c[0], lane_value(ec[0], 3 * r + 1)), lane_value(ec[0], 3 * r + 2));
                    const double c1 = next_lane(c[1], lane_value(ec[1], 3 * r + 1));
                    const double c3 = prev_lane(c[3], lane_value(ec[3], 3 * r));
                    const double T1 = next_lane(T, lane_value(eT, 3 * r + 1));
                    S.lb[q] = S.lb[q] + (((c0 + c1) + c[2]) + c3);
                    TB[q] = inp ? I.tb + g * (T1 - T) : I.tb;
                    put_vel(r, (0.0 - ct) + cmt, L, vv, I.old);
                }
            }
        } else if (dir != 0 && act) {
            // up the column: face r gives to the rows r - 2 .. r + 1; a0: row r + 1, complete with it, a1, a2: r, r - 1;
            // ct: of row r
            auto load = [&](int r) {
                if (r >= -1)
                    in[(r + 1) % (kAhead + 1)] = RowIn{at(vel, r), at(hf, r), r >= 0 && r <= R ? at(tr, r - 1) : 0.0,
                                                       r >= 0 && r < R ? at8(old, q0, r) : 0.0,
                                                       r >= 0 && r < R ? at8(TB, q0, r) : 0.0, at2(gr, r)};
            };
#pragma unroll
            for (int r = R + 1; r > R + 1 - kAhead; --r) load(r);
            if (own) {
                double a0 = 0.0, a1 = 0.0, a2 = 0.0, T1 = 0.0, ct = 0.0;
                double t0 = S.loc[lds(R + 1)], tp1 = S.loc[lds(R + 2)], tm1 = S.loc[lds(R)];
#pragma unroll
                for (int r = R + 1; r >= -1; --r) {
                    __builtin_amdgcn_sched_barrier(0);
                    load(r - kAhead);
                    const RowIn I = in[(r + 1) % (kAhead + 1)];
                    const int j = j0 + r;
                    const double L = I.G.x * deepFacC * drF * I.H, T = I.V * L * rhoFacC;
                    const double tm2 = S.loc[lds(r - 2)];
                    double c[4], vv;
                    face(j >= 2 && j <= GNY - 2, cg[r + 2] - cg[r + 1], I.V, L, T, I.G.y, tm2, tm1, t0, tp1, my, r + 1, c, vv);
                    if (r >= -1 && r + 1 < R) {
                        const int ql = q0 + (r + 1) * GNX;
                        S.lb[ql] = S.lb[ql] + (a0 + c[3]);
                    }
                    if (r >= 0 && r <= R) {
                        const double cmt = inb >> (r + 1) & 1 ? cg[r + 1] * I.TR : 0.0;
                        if (r < R) {
                            TB[q0 + r * GNX] = inb >> (r + 2) & 1 ? I.tb + cg[r + 2] * (T1 - T) : I.tb;
                            put_vel(r, (0.0 - ct) + cmt, L, vv, I.old);
                        }
                        ct = cmt;
                    }
                    a0 = a1 + c[2];
                    a1 = a2 + c[1];
                    a2 = c[0];
                    T1 = T;
                    tp1 = t0, t0 = tm1, tm1 = tm2;
                }
            }
        } else {
            if (init && own) {
#pragma unroll
                for (int r = 0; r < R; ++r) vbar[q0 + r * GNX] = 0.0;
            }
        }
        __syncthreads();
        if (P.fill_before) corner_fill_T(S.lb, a, S.plan, P.fill_before, tid);
    }
#pragma unroll
    for (int r = 0; r < R; ++r) {
        if (!own) continue;
        const int q = q0 + r * GNX;
        TB[q] = TB[q] + S.lb[q];
        if (first[0]) UB[q] = 0.0;
        if (first[1]) VB[q] = 0.0;
    }
}

// Vertical DST3 (R) sweep after the horizontal passes, per column (member, tile, j, i), k = 0..nlev-1 downward.
// Interface k (0..K) is the top of cell k; w(k) = wFld at interface k, positive upward; the transport is
// rTrans(k) = w(k) * rA * mk(k), mk(k) = maskC(k-1) * maskC(k) for 1 <= k <= K-1, and 0 at the surface (k = 0)
// and the bottom (k = K). The interface value is the DST3 formula with the upstream side below for rTrans > 0:
//   Rj = (t(k-1) - t(k)) mk(k), Rjm = (t(k) - t(k+1)) mk(k+1), Rjp = (t(k-2) - t(k-1)) mk(k-1),
//   c = |w(k) dt(k) recip_drC(k)|, d0 = (2-c)(1-c)/6, d1 = (1-c^2)/6,
//   wT(k) = (rT+|rT|)/2 (t(k) + d0 Rj + d1 Rjm) + (rT-|rT|)/2 (t(k-1) - (d0 Rj + d1 Rjp)),
// with t = localTij after the horizontal passes. Update (the horizontal form, net outflow wT(k) - wT(k+1)):
//   local(k) <- local(k) - coef(k) ((wT(k) - wT(k+1)) - tracer(k) (rTrans(k) - rTrans(k+1))) maskC(k),
// gTracer = (local - tracer)/dt(k) on the whole tile array.
//
// Bound by HBM: one walk down the column, step k takes level k in, evaluates interface k - 1 and completes level k - 2; the
// level data are loaded kVertAhead steps ahead. With one step's loads in flight one member of 50 levels (300 MB) took 98 us;
// 75 us now, 4 TB/s. 24 members, which fill the card by themselves, take 1.01 ms either way (4.6 TB/s). One, two and four steps ahead measure the same, six 2 us more.
constexpr int kVertAhead = 2;
__global__ void __launch_bounds__(256) gad_vert_kernel(GadDev a, const double* __restrict__ loc_h) {
    const int q = blockIdx.x * blockDim.x + threadIdx.x;
    const int mt = blockIdx.y;
    if (q >= GPLANE) return;
    const int t = mt % a.T, m = mt / a.T;
    const int K = a.K;
    const int kmax = a.nlev ? a.nlev[m] : K;
    const int64_t b2 = (int64_t)t * GPLANE + q;
    const double rA = a.rA[b2], rrA = a.recip_rA[b2];
    const int64_t c3 = m * a.ms3 + (int64_t)t * K * GPLANE + q;
    const double* __restrict__ w = a.w + c3;
    const double* __restrict__ tr = a.tr + c3;
    const double* __restrict__ rhC = a.recip_hFacC + c3;
    const double* __restrict__ lh = loc_h + c3;
    const double* __restrict__ mc = a.maskC + mask_slot(a, m) * a.mms + (int64_t)t * K * GPLANE + q;
    double* __restrict__ out = a.out + c3;
    auto L = [](int k) { return (int64_t)k * GPLANE; };
    double rw[kVertAhead], rtr[kVertAhead], rrh[kVertAhead], rlh[kVertAhead], rmc[kVertAhead];
    auto load = [&](int s, int k) {
        const int64_t o = L(max(min(k, kmax - 1), 0));
        rw[s] = w[o];
        rtr[s] = tr[o];
        rrh[s] = rhC[o];
        rlh[s] = lh[o];
        rmc[s] = mc[o];
    };
#pragma unroll
    for (int s = 0; s < kVertAhead; ++s) load(s, s);
    // levels k - 1, k - 2, k - 3 (1, 2, 3), 0 outside 0 .. kmax - 1; wT2, rT2: interface k - 2
    double T1 = 0.0, T2 = 0.0, T3 = 0.0, M1 = 0.0, M2 = 0.0, mk1 = 0.0, mk2 = 0.0, w1 = 0.0, tr1 = 0.0, tr2 = 0.0, rh1 = 0.0,
           rh2 = 0.0, wT2 = 0.0, rT2 = 0.0;
    auto step = [&](int k, int s) {
        const bool wet = k < kmax;
        const double T0 = wet ? rlh[s] : 0.0, M0 = wet ? rmc[s] : 0.0, w0 = rw[s], tr0 = rtr[s], rh0 = rrh[s];
        load(s, k + kVertAhead);
        const double mk0 = k >= 1 ? M1 * M0 : 0.0;
        // interface k - 1: upstream for positive (upward) transport: cell k-1, then k; downstream: k-2, then k-3
        double wT1 = 0.0, rT1 = 0.0;
        const int ki = k - 1;
        if (ki >= 1 && ki <= kmax - 1) {
            rT1 = w1 * rA * mk1;
            const double cfl = fabs(w1 * a.dTlev[ki] * a.recip_drC[ki]);
            wT1 = dst3_flux(rT1, cfl, a.oneSixth, T0, T1, T2, T3, mk0, mk1, mk2);
        }
        const int l = k - 2;
        if (l >= 0) {
            const double cf = a.dTlev[l] * a.recip_rhoFacC[l] * rh2 * a.recip_drF[l] * rrA * a.recip_deepFac2C[l];
            const double loc = T2 - cf * ((wT2 - wT1) - tr2 * (rT2 - rT1)) * M2;
            out[L(l)] = (loc - tr2) / a.dTlev[l];
        }
        T3 = T2, T2 = T1, T1 = T0;
        M2 = M1, M1 = M0;
        mk2 = mk1, mk1 = mk0;
        w1 = w0, tr2 = tr1, tr1 = tr0, rh2 = rh1, rh1 = rh0, wT2 = wT1, rT2 = rT1;
    };
    // steps 0 .. kmax + 1, the last two to complete the column
    for (int k0 = 0; k0 < kmax + 2; k0 += kVertAhead) {
#pragma unroll
        for (int s = 0; s < kVertAhead; ++s)
            if (k0 + s < kmax + 2 && kmax > 0) step(k0 + s, s);
    }
}

// Reverse mode of gad_vert_kernel for one column (member, tile, q): from gbar, the cotangent of gTracer, and loc_h,
// the forward's localTij after the horizontal passes, it writes every level of the column of
//   locbar = the cotangent of loc_h (the identity term gbar/dt plus the interface values' tracer weights),
//   trb    = the vertical part of the tracer cotangent: -gbar/dt + e(k) (rTrans(k) - rTrans(k+1)),
//   wb     = the cotangent of w at interfaces 1 .. nlev-1 (0 at the surface and below the member's levels),
// with e(k) = coef(k) maskC(k) gbar(k)/dt(k). Through the update of level k the interface value wT(k) has the
// cotangent e(k-1) - e(k) and rTrans(k) e(k) tracer(k) - e(k-1) tracer(k-1); the interface value's partials
// (dst3_partials: the four tracer weights, d/dtransport, d/dcfl) carry them on to loc_h and to w through
// rTrans = w rA mk and cfl = |w dt recip_drC| (d|x|/dx = sign x, 0 at 0).
//
// One walk down the column: step k takes level k in, evaluates interface k - 1 (which reads the levels k - 3 .. k) and
// writes what is complete, so each of the six arrays is read once and each of the three written once; the level data are
// loaded kVertAhead steps ahead. Bound by HBM: reading them as needed, with locbar updated in memory, took 240 us for one
// member of 50 levels; 84 us now (470 MB, 5.6 TB/s).
__global__ void __launch_bounds__(256) gad_vert_adjoint_kernel(GadDev a, int col0, const double* __restrict__ loc_h,
                                                               const double* __restrict__ gbar,
                                                               double* __restrict__ locbar, double* __restrict__ trb,
                                                               double* __restrict__ wb) {
    const int q = blockIdx.x * blockDim.x + threadIdx.x;
    const int mt = col0 + blockIdx.y;
    if (q >= GPLANE) return;
    const int t = mt % a.T, m = mt / a.T;
    const int K = a.K;
    const int kmax = a.nlev ? a.nlev[m] : K;
    const int64_t b2 = (int64_t)t * GPLANE + q;
    const double rA = a.rA[b2], rrA = a.recip_rA[b2];
    const int64_t c3 = m * a.ms3 + (int64_t)t * K * GPLANE + q;
    const double* __restrict__ w = a.w + c3;
    const double* __restrict__ tr = a.tr + c3;
    const double* __restrict__ rhC = a.recip_hFacC + c3;
    const double* __restrict__ lh = loc_h + c3;
    const double* __restrict__ gb = gbar + c3;
    const double* __restrict__ mc = a.maskC + mask_slot(a, m) * a.mms + (int64_t)t * K * GPLANE + q;
    double* __restrict__ lb = locbar + c3;
    double* __restrict__ tb = trb + c3;
    double* __restrict__ wbar = wb + c3;
    auto L = [](int k) { return (int64_t)k * GPLANE; };
    double rw[kVertAhead], rtr[kVertAhead], rrh[kVertAhead], rlh[kVertAhead], rgb[kVertAhead], rmc[kVertAhead];
    auto load = [&](int s, int k) {
        const int64_t o = L(max(min(k, kmax - 1), 0));
        rw[s] = w[o];
        rtr[s] = tr[o];
        rrh[s] = rhC[o];
        rlh[s] = lh[o];
        rgb[s] = gb[o];
        rmc[s] = mc[o];
    };
#pragma unroll
    for (int s = 0; s < kVertAhead; ++s) load(s, s);
    // levels k - 1, k - 2, k - 3 (1, 2, 3)
    double T1 = 0.0, T2 = 0.0, T3 = 0.0, M1 = 0.0, mk1 = 0.0, mk2 = 0.0, e1 = 0.0, e2 = 0.0, w1 = 0.0,
           tr1 = 0.0, tr2 = 0.0, rT1 = 0.0, tv1 = 0.0, l1 = 0.0, l2 = 0.0, l3 = 0.0;
    auto step = [&](int k, int s) {
        const bool wet = k < kmax;
        const double T0 = wet ? rlh[s] : 0.0, M0 = wet ? rmc[s] : 0.0, w0 = rw[s], tr0 = rtr[s], g = rgb[s], rh = rrh[s];
        load(s, k + kVertAhead);
        const bool inner = k >= 1 && wet;
        const double mk0 = inner ? M1 * M0 : 0.0, rT0 = inner ? w0 * rA * mk0 : 0.0;
        double e0 = 0.0, l0 = 0.0, tv0 = 0.0;
        if (wet) {
            const double cf = a.dTlev[k] * a.recip_rhoFacC[k] * rh * a.recip_drF[k] * rrA * a.recip_deepFac2C[k];
            l0 = g / a.dTlev[k];
            e0 = cf * M0 * l0;
            tv0 = -l0;
        }
        if (k >= 1 && k - 1 < kmax) tb[L(k - 1)] = tv1 + e1 * (rT1 - rT0);
        const int ki = k - 1;
        if (ki >= 1 && ki <= kmax - 1) {
            const double wTb = e2 - e1;
            const double arg = w1 * a.dTlev[ki] * a.recip_drC[ki];
            const FluxPartials P = dst3_partials(rT1, fabs(arg), a.oneSixth, T0, T1, T2, T3, mk0, mk1, mk2);
            if (wet) l0 = l0 + P.w[0] * wTb;
            l1 = l1 + P.w[1] * wTb;
            l2 = l2 + P.w[2] * wTb;
            l3 = l3 + P.w[3] * wTb;
            const double rTb = e1 * tr1 - e2 * tr2 + P.dtr * wTb;
            const double sgn = arg > 0.0 ? 1.0 : (arg < 0.0 ? -1.0 : 0.0);
            wbar[L(ki)] = rTb * (rA * mk1) + (P.dc * wTb) * (sgn * a.dTlev[ki] * a.recip_drC[ki]);
        } else if (ki == 0) {
            wbar[0] = 0.0;
        }
        if (k >= 3 && k - 3 < kmax) lb[L(k - 3)] = l3;
        T3 = T2, T2 = T1, T1 = T0;
        M1 = M0, mk2 = mk1, mk1 = mk0;
        e2 = e1, e1 = e0;
        w1 = w0, tr2 = tr1, tr1 = tr0, rT1 = rT0, tv1 = tv0;
        l3 = l2, l2 = l1, l1 = l0;
    };
    // steps 0 .. kmax + 2, the last three to complete the column
    for (int k0 = 0; k0 < kmax + 3; k0 += kVertAhead) {
#pragma unroll
        for (int s = 0; s < kVertAhead; ++s)
            if (k0 + s < kmax + 3) step(k0 + s, s);
    }
    for (int k = kmax; k < K; ++k) lb[L(k)] = tb[L(k)] = wbar[L(k)] = 0.0;
}

}  // namespace mj

using namespace mj;

mj_gad_plan::~mj_gad_plan() {
    if (d_tiles) (void)hipFree(d_tiles);
}

// ------------------------------------------------------------------------------------------------ plan (host)
// Per-facet pass table of gad_advection.F:333-351 (reference gad.py:217-235) and the update regions / fill calls
// of :376-774 (gad.py:339-375), as boxes. Array index of Fortran i is i - 1 + OLx.
static void pass_table(int face, int pass, bool* overlapOnly, bool* interiorOnly, bool* cX, bool* cY) {
    auto in = [&](int a, int b, int c) { return face == a || face == b || face == c; };
    if (pass == 1) {
        *overlapOnly = face % 3 == 0;
        *interiorOnly = face % 3 != 0;
        *cX = in(6, 1, 2);
        *cY = in(3, 4, 5);
    } else if (pass == 2) {
        *overlapOnly = face % 3 == 2;
        *interiorOnly = face % 3 == 1;
        *cX = in(2, 3, 4);
        *cY = in(5, 6, 1);
    } else {
        *overlapOnly = false;
        *interiorOnly = true;
        *cX = face == 5 || face == 6;
        *cY = face == 2 || face == 3;
    }
}

// Fills P's host tables from the topology (no device work).
static int build_plan_host(mj_gad_plan* P, int ntiles, const int32_t* face, const uint8_t* edges, int sNx, int sNy,
                           int OLx, int OLy) {
    P->ntiles = ntiles;
    P->sNx = sNx;
    P->sNy = sNy;
    P->OLx = OLx;
    P->OLy = OLy;
    P->tiles.resize(ntiles);
    auto ix = [&](int i) { return (int16_t)(i - 1 + OLx); };
    auto jx = [&](int j) { return (int16_t)(j - 1 + OLy); };
    for (int t = 0; t < ntiles; ++t) {
        const bool N = edges[4 * t] != 0, S = edges[4 * t + 1] != 0, E = edges[4 * t + 2] != 0,
                   W = edges[4 * t + 3] != 0;
        MjTilePlan& tp = P->tiles[t];
        memset(&tp, 0, sizeof(tp));
        tp.sw = W && S;  // fill_cs_corner_tr_rl.F:78-85
        tp.se = E && S;
        tp.nw = W && N;
        tp.ne = E && N;
        for (int pass = 1; pass <= 3; ++pass) {
            bool ov, io, cX, cY;
            pass_table(face[t], pass, &ov, &io, &cX, &cY);
            MjSweep& X = tp.sweep[pass - 1][0];
            MjSweep& Y = tp.sweep[pass - 1][1];
            if (cX) {  // gad_advection.F:376-565
                const bool doflux = !ov || N || S;
                X.fill_before = (doflux && ov) ? 1 : 0;
                X.fill_after = (doflux && ov && pass == 1) ? 2 : 0;
                if (ov) {
                    int iMin = 1 - OLx + 1, iMax = sNx + OLx - 1;
                    if (W) iMin = 1;
                    if (E) iMax = sNx;
                    if (S) X.box[X.nbox++] = MjBox{ix(iMin), (int16_t)(ix(iMax) + 1), jx(1 - OLy), (int16_t)(jx(0) + 1)};
                    if (N)
                        X.box[X.nbox++] =
                            MjBox{ix(iMin), (int16_t)(ix(iMax) + 1), jx(sNy + 1), (int16_t)(jx(sNy + OLy) + 1)};
                } else {
                    int jMin = 1 - OLy, jMax = sNy + OLy;
                    if (io && S) jMin = 1;
                    if (io && N) jMax = sNy;
                    X.box[X.nbox++] =
                        MjBox{ix(1 - OLx + 1), (int16_t)(ix(sNx + OLx - 1) + 1), jx(jMin), (int16_t)(jx(jMax) + 1)};
                }
                X.run = X.nbox > 0 || X.fill_before || X.fill_after;
            }
            if (cY) {  // gad_advection.F:585-774
                const bool doflux = !ov || E || W;
                Y.fill_before = (doflux && ov) ? 2 : 0;
                Y.fill_after = (doflux && ov && pass == 1) ? 1 : 0;
                if (ov) {
                    int jMin = 1 - OLy + 1, jMax = sNy + OLy - 1;
                    if (S) jMin = 1;
                    if (N) jMax = sNy;
                    if (W) Y.box[Y.nbox++] = MjBox{ix(1 - OLx), (int16_t)(ix(0) + 1), jx(jMin), (int16_t)(jx(jMax) + 1)};
                    if (E)
                        Y.box[Y.nbox++] =
                            MjBox{ix(sNx + 1), (int16_t)(ix(sNx + OLx) + 1), jx(jMin), (int16_t)(jx(jMax) + 1)};
                } else {
                    int iMin = 1 - OLx, iMax = sNx + OLx;
                    if (io && W) iMin = 1;
                    if (io && E) iMax = sNx;
                    Y.box[Y.nbox++] =
                        MjBox{ix(iMin), (int16_t)(ix(iMax) + 1), jx(1 - OLy + 1), (int16_t)(jx(sNy + OLy - 1) + 1)};
                }
                Y.run = Y.nbox > 0 || Y.fill_before || Y.fill_after;
            }
        }
    }
    return MJ_OK;
}

// What the kernels rely on: the update boxes of a sweep are disjoint and lie in the plane together with the face q + d of
// each of their points.
static int check_boxes(const mj_gad_plan& P) {
    for (int t = 0; t < P.ntiles; ++t)
        for (int pass = 0; pass < 3; ++pass)
            for (int dir = 0; dir < 2; ++dir) {
                const MjSweep& S = P.tiles[t].sweep[pass][dir];
                bool ok = S.nbox >= 0 && S.nbox <= 2;
                for (int b = 0; ok && b < S.nbox; ++b) {
                    const MjBox& B = S.box[b];
                    ok = B.i0 >= 0 && B.j0 >= 0 && B.i0 < B.i1 && B.j0 < B.j1 && B.i1 + (dir == 0) <= GNX &&
                         B.j1 + (dir == 1) <= GNY;
                }
                if (ok && S.nbox == 2) {
                    const MjBox &A = S.box[0], &B = S.box[1];
                    ok = A.i1 <= B.i0 || B.i1 <= A.i0 || A.j1 <= B.j0 || B.j1 <= A.j0;
                }
                if (!ok) {
                    set_error("gad plan: tile %d pass %d dir %d: update boxes overlap or leave the plane", t, pass + 1,
                              dir);
                    return MJ_ERR_ARG;
                }
            }
    return MJ_OK;
}

extern "C" int mj_gad_plan_create(int ntiles, const int32_t* face, const uint8_t* edges, int sNx, int sNy, int OLx,
                                  int OLy, mj_gad_plan** out) {
    MJ_REQUIRE(out && face && edges && ntiles > 0, "mj_gad_plan_create: bad argument");
    MJ_REQUIRE(sNx + 2 * OLx == GNX && sNy + 2 * OLy == GNY && OLx == OLy,
               "mj_gad_plan_create: the kernels are built for %dx%d tiles with equal halos (got sNx %d sNy %d OL %d,%d)",
               GNY, GNX, sNx, sNy, OLx, OLy);
    mj_gad_plan* P = new mj_gad_plan();
    build_plan_host(P, ntiles, face, edges, sNx, sNy, OLx, OLy);
    if (check_boxes(*P) != MJ_OK) {
        delete P;
        return MJ_ERR_ARG;
    }
    hipError_t e = hipMalloc((void**)&P->d_tiles, sizeof(MjTilePlan) * ntiles);
    if (e == hipSuccess)
        e = hipMemcpy(P->d_tiles, P->tiles.data(), sizeof(MjTilePlan) * ntiles, hipMemcpyHostToDevice);
    if (e != hipSuccess) {
        delete P;
        set_error("mj_gad_plan_create: %s", hipGetErrorString(e));
        return MJ_ERR_HIP;
    }
    *out = P;
    return MJ_OK;
}

extern "C" int mj_gad_plan_destroy(mj_gad_plan* plan) {
    delete plan;
    return MJ_OK;
}

static int describe(const mj_gad_plan* P, uint8_t* masks, int32_t* fills);

extern "C" int mj_gad_plan_describe(const mj_gad_plan* P, uint8_t* masks, int32_t* fills) {
    MJ_REQUIRE(P, "mj_gad_plan_describe: null plan");
    return describe(P, masks, fills);
}

extern "C" int mj_gad_tables_host(int ntiles, const int32_t* face, const uint8_t* edges, int sNx, int sNy, int OLx,
                                  int OLy, uint8_t* masks, int32_t* fills) {
    MJ_REQUIRE(face && edges && ntiles > 0, "mj_gad_tables_host: bad argument");
    MJ_REQUIRE(sNx + 2 * OLx == GNX && sNy + 2 * OLy == GNY && OLx == OLy, "mj_gad_tables_host: unsupported layout");
    mj_gad_plan P;
    P.ntiles = ntiles;
    P.sNx = sNx;
    P.sNy = sNy;
    P.OLx = OLx;
    P.OLy = OLy;
    build_plan_host(&P, ntiles, face, edges, sNx, sNy, OLx, OLy);
    if (check_boxes(P) != MJ_OK) return MJ_ERR_ARG;
    return describe(&P, masks, fills);
}

static int describe(const mj_gad_plan* P, uint8_t* masks, int32_t* fills) {
    const int T = P->ntiles, plane = GPLANE;
    if (masks) memset(masks, 0, (size_t)6 * T * plane);
    for (int t = 0; t < T; ++t)
        for (int pass = 0; pass < 3; ++pass)
            for (int dir = 0; dir < 2; ++dir) {
                const MjSweep& S = P->tiles[t].sweep[pass][dir];
                if (masks)
                    for (int b = 0; b < S.nbox; ++b)
                        for (int j = S.box[b].j0; j < S.box[b].j1; ++j)
                            for (int i = S.box[b].i0; i < S.box[b].i1; ++i)
                                masks[((size_t)(pass * 2 + dir) * T + t) * plane + j * GNX + i] = 1;
                if (fills) {
                    fills[(pass * 4 + dir * 2 + 0) * T + t] = S.fill_before;
                    fills[(pass * 4 + dir * 2 + 1) * T + t] = S.fill_after;
                }
            }
    return MJ_OK;
}

namespace {
size_t al256(size_t v) { return (v + 255) & ~(size_t)255; }
// Mask slots: one shared set (mask_member_stride 0), one per member, or mask_slots sets picked by mask_index.
int mask_slots_of(const mj_gad_config* c) {
    return c->mask_member_stride == 0 ? 1 : (c->mask_index ? c->mask_slots : c->batch);
}
// The bit planes of every (mask slot, tile, level), then the packed 2-D metrics.
size_t mask_bits_bytes(const mj_gad_config* c, int ntiles) {
    return (size_t)mask_slots_of(c) * ntiles * c->nr * 2 * kPlaneBits * sizeof(unsigned);
}
size_t pre_bytes(const mj_gad_config* c, int ntiles) {
    return al256(mask_bits_bytes(c, ntiles)) + al256((size_t)3 * ntiles * GPLANE * sizeof(double2));
}
// One member-strided FP64 3-D array of the batch (the R flux's localTij, the reverse mode's replay planes).
size_t batch3_bytes(const mj_gad_config* c, int ntiles) {
    return (size_t)c->batch * (size_t)std::max<int64_t>(c->member_stride3d, (int64_t)ntiles * c->nr * GPLANE) *
           sizeof(double);
}
// (member, tile)s of one reverse launch.
int adjoint_columns(const mj_gad_config* c, int ntiles) {
    return (int)std::min<int64_t>((int64_t)c->batch * ntiles, std::max(1, kAdjChunk / c->nr));
}
// The reverse mode's part of its workspace (before the bit planes): the snapshots of a launch (more than kAdjChunk units
// if one column is more), and with the R flux localTij and its cotangent, from adjoint_snap_bytes on.
size_t adjoint_snap_bytes(const mj_gad_config* c, int ntiles) {
    const size_t unit = (size_t)GPLANE * sizeof(double);
    return std::max((size_t)kAdjChunk * kAdjPlanes * unit, (size_t)adjoint_columns(c, ntiles) * c->nr * kAdjSnaps * unit);
}
size_t adjoint_scratch_bytes(const mj_gad_config* c, int ntiles, int with_w) {
    return al256(adjoint_snap_bytes(c, ntiles) + (with_w ? 2 * batch3_bytes(c, ntiles) : 0));
}
// The per-call tables at `pre` (pre_bytes): the bit planes of maskLocW / maskLocS for every (mask slot, tile,
// level) and the packed 2-D metrics; sets a.mbits and a.g2.
int launch_pre(GadDev& a, const mj_gad_config* c, void* pre, hipStream_t st) {
    const int nslots = mask_slots_of(c);
    a.mbits = (unsigned*)pre;
    a.g2 = (double2*)((char*)pre + al256(mask_bits_bytes(c, a.T)));
    const int nplanes = 2 * nslots * a.T * a.K;
    const int npack = (a.T * GPLANE + kPreThreads - 1) / kPreThreads;
    hipLaunchKernelGGL(gad_pre_kernel, dim3((unsigned)(nplanes + npack)), dim3(kPreThreads), 0, st, a, nplanes);
    MJ_HIP(hipGetLastError());
    return MJ_OK;
}
int check_mask_slots(const mj_gad_config* c, int ntiles) {
    MJ_REQUIRE(c->mask_member_stride == 0 || c->mask_index == nullptr || c->mask_slots >= 1,
               "mj_gad: mask_slots (the number of mask slots) is required with mask_index");
    MJ_REQUIRE((int64_t)mask_slots_of(c) * ntiles * c->nr < (1ll << 30), "mj_gad: too many mask slots");
    return MJ_OK;
}

// Device arguments of the DST3 kernels shared by the forward and reverse entry points.
GadDev gad_dev(const mj_gad_plan* P, const mj_gad_grid* g, const mj_gad_config* c, const double* uFld,
               const double* vFld, const double* wFld, const double* tracer, const double* hFacW, const double* hFacS,
               const double* recip_hFacC) {
    GadDev a{};
    a.B = c->batch;
    a.T = P->ntiles;
    a.K = c->nr;
    a.OLx = P->OLx;
    a.OLy = P->OLy;
    a.sNx = P->sNx;
    a.sNy = P->sNy;
    a.ms3 = c->member_stride3d;
    a.mms = c->mask_member_stride;
    a.mask_index = c->mask_member_stride ? c->mask_index : nullptr;
    a.lpb = c->levels_per_block > 0 ? c->levels_per_block : 1;
    a.tiles = P->d_tiles;
    a.dyG = g->dyG;
    a.dxG = g->dxG;
    a.recip_dxC = g->recip_dxC;
    a.recip_dyC = g->recip_dyC;
    a.recip_rA = g->recip_rA;
    a.rA = g->rA;
    a.maskInC = g->maskInC;
    a.maskW = g->maskW;
    a.maskS = g->maskS;
    a.maskC = g->maskC;
    a.dTlev = g->dTlev;
    a.drF = g->drF;
    a.recip_drF = g->recip_drF;
    a.rhoFacC = g->rhoFacC;
    a.recip_rhoFacC = g->recip_rhoFacC;
    a.deepFacC = g->deepFacC;
    a.recip_deepFacC = g->recip_deepFacC;
    a.recip_deepFac2C = g->recip_deepFac2C;
    a.recip_drC = g->recip_drC;
    a.oneSixth = g->oneSixth;
    a.u = uFld;
    a.v = vFld;
    a.w = wFld;
    a.tr = tracer;
    a.hFacW = hFacW;
    a.hFacS = hFacS;
    a.recip_hFacC = recip_hFacC;
    a.nlev = c->nlev;
    return a;
}
}  // namespace

extern "C" size_t mj_gad_dst3_workspace_bytes(const mj_gad_config* c, int ntiles, int with_w) {
    if (!c || c->batch < 1 || c->nr < 1 || ntiles < 1) return 0;
    return (with_w ? al256(batch3_bytes(c, ntiles)) : 0) + pre_bytes(c, ntiles);
}

extern "C" int mj_gad_dst3(const mj_gad_plan* P, const mj_gad_grid* g, const mj_gad_config* c, const double* uFld,
                           const double* vFld, const double* wFld, const double* tracer, const double* hFacW,
                           const double* hFacS, const double* recip_hFacC, double* gTracer, void* work,
                           size_t work_bytes, void* stream) {
    MJ_REQUIRE(P && g && c, "mj_gad_dst3: null plan/grid/config");
    MJ_REQUIRE(uFld && vFld && tracer && hFacW && hFacS && recip_hFacC && gTracer, "mj_gad_dst3: null field");
    MJ_REQUIRE(g->dyG && g->dxG && g->recip_dxC && g->recip_dyC && g->recip_rA && g->maskInC && g->maskW && g->maskS,
               "mj_gad_dst3: null grid field");
    MJ_REQUIRE(g->dTlev && g->drF && g->recip_drF && g->rhoFacC && g->recip_rhoFacC && g->deepFacC &&
                   g->recip_deepFacC && g->recip_deepFac2C,
               "mj_gad_dst3: null vertical grid field");
    MJ_REQUIRE(c->batch >= 1 && c->nr >= 1, "mj_gad_dst3: batch and nr must be >= 1");
    MJ_REQUIRE(c->member_stride3d >= (int64_t)P->ntiles * c->nr * GPLANE || c->batch == 1,
               "mj_gad_dst3: member_stride3d too small");
    MJ_REQUIRE((int64_t)c->batch * P->ntiles * c->nr < (1ll << 31), "mj_gad_dst3: too many (member, tile, level)s");
    int rc = check_mask_slots(c, P->ntiles);
    if (rc) return rc;
    if (wFld) MJ_REQUIRE(g->maskC && g->rA && g->recip_drC, "mj_gad_dst3: the R flux needs maskC, rA, recip_drC");
    const size_t need = mj_gad_dst3_workspace_bytes(c, P->ntiles, wFld != nullptr);
    MJ_REQUIRE(work && work_bytes >= need, "mj_gad_dst3: work %zu < %zu bytes", work ? work_bytes : 0, need);
    MJ_REQUIRE(((uintptr_t)work & 255) == 0, "mj_gad_dst3: work must be 256-byte aligned");
    {
        const char *w0 = (const char*)work, *w1 = w0 + need;
        const char *g0 = (const char*)gTracer, *g1 = g0 + batch3_bytes(c, P->ntiles);
        MJ_REQUIRE(w1 <= g0 || g1 <= w0, "mj_gad_dst3: work must not overlap gTracer");
    }
    double* loc_h = (double*)work;
    GadDev a = gad_dev(P, g, c, uFld, vFld, wFld, tracer, hFacW, hFacS, recip_hFacC);
    a.out = wFld ? loc_h : gTracer;
    hipStream_t st = as_stream(stream);
    if ((rc = launch_pre(a, c, (char*)work + (wFld ? al256(batch3_bytes(c, P->ntiles)) : 0), st))) return rc;
    const int nkb = (c->nr + a.lpb - 1) / a.lpb;
    const unsigned nblk = (unsigned)((c->batch * P->ntiles * nkb + 7) / 8 * 8);
    if (a.lpb > 1)
        hipLaunchKernelGGL(gad_hz_kernel<true>, dim3(nblk), dim3(kHzThreads), 0, st, a);
    else
        hipLaunchKernelGGL(gad_hz_kernel<false>, dim3(nblk), dim3(kHzThreads), 0, st, a);
    MJ_HIP(hipGetLastError());
    if (wFld) {
        a.out = gTracer;
        hipLaunchKernelGGL(gad_vert_kernel, dim3((GPLANE + 255) / 256, (unsigned)(c->batch * P->ntiles)), dim3(256), 0,
                           st, a, (const double*)loc_h);
        MJ_HIP(hipGetLastError());
    }
    return MJ_OK;
}

extern "C" size_t mj_gad_dst3_adjoint_workspace_bytes(const mj_gad_config* c, int ntiles, int with_w) {
    if (!c || c->batch < 1 || c->nr < 1 || ntiles < 1) return 0;
    return adjoint_scratch_bytes(c, ntiles, with_w) + pre_bytes(c, ntiles);
}

extern "C" int mj_gad_dst3_adjoint(const mj_gad_plan* P, const mj_gad_grid* g, const mj_gad_config* c,
                                   const double* uFld, const double* vFld, const double* wFld, const double* tracer,
                                   const double* hFacW, const double* hFacS, const double* recip_hFacC,
                                   const double* gTracer_bar, double* tracer_bar, double* uFld_bar, double* vFld_bar,
                                   double* wFld_bar, double* work, size_t work_bytes, void* stream) {
    MJ_REQUIRE(P && g && c, "mj_gad_dst3_adjoint: null plan/grid/config");
    MJ_REQUIRE(uFld && vFld && tracer && hFacW && hFacS && recip_hFacC && gTracer_bar && tracer_bar && uFld_bar &&
                   vFld_bar && work,
               "mj_gad_dst3_adjoint: null field");
    MJ_REQUIRE(g->dyG && g->dxG && g->recip_dxC && g->recip_dyC && g->recip_rA && g->maskInC && g->maskW && g->maskS,
               "mj_gad_dst3_adjoint: null grid field");
    MJ_REQUIRE(c->batch >= 1 && c->nr >= 1, "mj_gad_dst3_adjoint: batch and nr must be >= 1");
    MJ_REQUIRE(c->member_stride3d >= (int64_t)P->ntiles * c->nr * GPLANE || c->batch == 1,
               "mj_gad_dst3_adjoint: member_stride3d too small");
    MJ_REQUIRE((int64_t)c->batch * P->ntiles * c->nr < (1ll << 31), "mj_gad_dst3_adjoint: too many blocks");
    if (wFld) {
        MJ_REQUIRE(wFld_bar && g->maskC && g->rA && g->recip_drC,
                   "mj_gad_dst3_adjoint: the R flux needs wFld_bar, maskC, rA, recip_drC");
        for (const double* o : {(const double*)tracer_bar, (const double*)uFld_bar, (const double*)vFld_bar})
            MJ_REQUIRE(o != wFld_bar, "mj_gad_dst3_adjoint: wFld_bar aliases another output");
    }
    int rc = check_mask_slots(c, P->ntiles);
    if (rc) return rc;
    const size_t need = mj_gad_dst3_adjoint_workspace_bytes(c, P->ntiles, wFld != nullptr);
    MJ_REQUIRE(work_bytes >= need, "mj_gad_dst3_adjoint: work %zu < %zu bytes", work_bytes, need);
    MJ_REQUIRE(((uintptr_t)work & 255) == 0, "mj_gad_dst3_adjoint: work must be 256-byte aligned");
    hipStream_t st = as_stream(stream);
    GadDev a = gad_dev(P, g, c, uFld, vFld, nullptr, tracer, hFacW, hFacS, recip_hFacC);
    if ((rc = launch_pre(a, c, (char*)work + adjoint_scratch_bytes(c, P->ntiles, wFld != nullptr), st))) return rc;
    GadDev f = a;  // the forward replay, with the R flux localTij after the horizontal passes
    f.w = wFld;
    f.out = nullptr;
    double* lbar = nullptr;
    if (wFld) {
        f.out = (double*)((char*)work + adjoint_snap_bytes(c, P->ntiles));
        lbar = (double*)((char*)f.out + batch3_bytes(c, P->ntiles));
    }
    const int ncol = c->batch * P->ntiles, step = adjoint_columns(c, P->ntiles);
    for (int c0 = 0; c0 < ncol; c0 += step) {
        const int nc = std::min(step, ncol - c0), n = nc * c->nr;
        const unsigned nblk = (unsigned)((n + 7) / 8 * 8);
        hipLaunchKernelGGL(gad_hz_snap_kernel, dim3(nblk), dim3(kHzThreads), 0, st, f, c0 * c->nr, n, work);
        MJ_HIP(hipGetLastError());
        if (wFld) {
            hipLaunchKernelGGL(gad_vert_adjoint_kernel, dim3((GPLANE + 255) / 256, (unsigned)nc), dim3(256), 0, st, f, c0,
                               (const double*)f.out, gTracer_bar, lbar, tracer_bar, wFld_bar);
            MJ_HIP(hipGetLastError());
        }
        hipLaunchKernelGGL(gad_hz_adjoint_kernel, dim3(nblk), dim3(kAdjThreads), 0, st, a, gTracer_bar, tracer_bar,
                           uFld_bar, vFld_bar, (const double*)work, c0 * c->nr, n, (const double*)lbar);
        MJ_HIP(hipGetLastError());
    }
    return MJ_OK;
}
