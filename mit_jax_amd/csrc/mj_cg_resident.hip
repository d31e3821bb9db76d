// CG2D on gfx950, resident form: the whole solve of a member runs in 13 workgroups (one per tile) that keep every
// vector of the recurrence on chip, for 90 x 90 tiles.
//
// What bounds the other launch shapes: the phase launches stream 11 FP64 vectors per iteration through HBM, and the
// grid barriers of the persistent launch cost about 10 us each (device-scope fences write back and invalidate the L2s).
// Here a workgroup of 512 threads owns a (member, tile): x, r, s and z / q are registers (18 points per thread, 256
// registers at two waves per SIMD), the stencil operand is an LDS tile, aW sits in LDS and the other coefficients
// stream from L2. What the tiles of a member tell each other per phase is small: the ring values their neighbours read
// and one or two partial sums. These go through device memory as tagged 8-byte words, {tag, half of a double} (the tag
// is the number of the exchange): a reader polls a word until its tag arrives, so no fence, no barrier and no separate
// flag is needed. A round (publish, poll, workgroup barrier) takes 1.5-2.0 us for 1 to 19 members in flight.
//
// Members are taken from a queue by groups of workgroups (one per tile), as many groups as fit the device at one
// workgroup per CU: a member's tiles never wait for another member. Launched cooperatively (all workgroups resident).
//
// Arithmetic, operation order and the sums are those of mj_cg2d.hip, bit for bit (see unit_I1, group_phase_B / _C).
//
// Thread mapping: lane l of a half-wave holds columns l, l + 32 and l + 64 of six consecutive rows, so the first two
// steps of the row tree (v[l] + v[l + 64], then + v[l + 32]) are within the thread and 94 % of the lanes work (column
// pairs on a wave: 70 %). Lanes whose third column would be 90..95 repeat column 89, and the 16th half-wave repeats the
// 15th's rows: same loads, same values, the same values written to the same places, and counted once in the sums.
#include <algorithm>
#include <type_traits>

#include "mj_cg_sweep.h"
#include "mj_common.h"
#include "mj_internal.h"
#include "mj_resident_dev.h"

namespace mj {
namespace {

constexpr int kN = 90;                    // tile side
constexpr int kOL = 4, kNX = kN + 2 * kOL, kPlane = kNX * kNX;  // the arrays' padded tiles
constexpr int kPitch = kN + 2;            // LDS tile: rows and columns -1..90
constexpr int kTile = kPitch * kPitch;    // doubles
constexpr int kWaves = 8, kThreads = 64 * kWaves;
constexpr int kRows = 6, kPts = 3 * kRows;   // rows of a half-wave, points of a thread
constexpr int kRingLanes = 4 * kN / kWaves;  // ring points per wave, in its first lanes
static_assert(kRingLanes <= 64, "poll lanes");
static_assert(15 * kRows == kN && 2 * kWaves == 16, "rows");

struct ResDev {
    int B;
    int64_t ms, oms;
    const double *aW, *aS, *aC, *pW, *pS, *pC;
    const double *b, *x0;
    double* x;
    const double* norm;
    double tol_sq;
    int max_iters;
    const int32_t *full_off, *full_dst, *full_src;
    const int8_t* full_sign;
    const int32_t* op_index;
    const int4* ring;    // [T][360] {slot, LDS offset | neg << 30, padded source or -1, padded destination}
    const int32_t* pub;  // [T][4][90] slots of the tile's south and north rows and west and east columns, -1: not read
    ResSync y;
    mj_cg2d_diag* diag;
};

// p[off / 8 + k]: a uniform base, a lane's byte offset and a constant, the form of one load's address.
__device__ __forceinline__ double at(const double* p, unsigned off, int k) {
    return *reinterpret_cast<const double*>(reinterpret_cast<const char*>(p + k) + off);
}
__device__ __forceinline__ void put_at(double* p, unsigned off, int k, double v) {
    *reinterpret_cast<double*>(reinterpret_cast<char*>(p + k) + off) = v;
}

// ---------------------------------------------------------------------------------------------------- row trees
// The row trees of a half-wave's six rows, both halves at once: w[i] is lane l's v[l] (+ v[l + 64]) + v[l + 32] of row
// i. The steps 16, 8 and 4 run on two rows at a time in the lanes they leave idle; the sums end in the lanes of
// row_of_lane.
__device__ __forceinline__ double row_trees(double (&w)[kRows]) {
    swap16(w[0], w[1]);
    swap16(w[2], w[3]);
    swap16(w[4], w[5]);
    const double a = w[0] + w[1], b = w[2] + w[3], c = w[4] + w[5];
    // step 8: lanes 0..7 of a row of 16 go on with a, lanes 8..15 with b
    const double ab = dpp<0x118, 0xc>(a, b) + dpp<0x108, 0x3>(b, a), c8 = c + dpp<0x108, 0xf>(c, c);
    // step 4: c goes on in lanes 4..7
    double s = dpp<0x114, 0x2>(ab, c8) + dpp<0x104, 0x5>(c8, ab);
    s = s + dpp<0x102, 0xf>(s, s);
    return s + dpp<0x101, 0xf>(s, s);
}
// Which of its half's six rows a lane ends with, -1: none.
__device__ __forceinline__ int row_of_lane(int lane) {
    const int l = lane & 15, pair = l == 0 ? 0 : l == 8 ? 1 : l == 4 ? 2 : -1;
    return pair < 0 ? -1 : 2 * pair + (lane >> 4 & 1);
}

// ---------------------------------------------------------------------------------------------------- Fortran order
// Two chains of 16 additions at a time (their additions alternate: each hides the other's latency).
__device__ __forceinline__ void add16x2(double& s, double v, double& t, double w) {
    const double one = 1.0;
#define MJ_ADD2(i)                                                                    \
    "v_fmac_f64_dpp %0, %2, %4 row_newbcast:" #i " row_mask:0xf bank_mask:0xf\n"     \
    "v_fmac_f64_dpp %1, %3, %4 row_newbcast:" #i " row_mask:0xf bank_mask:0xf\n"
    asm volatile("s_nop 1\n" MJ_ADD2(0) MJ_ADD2(1) MJ_ADD2(2) MJ_ADD2(3) MJ_ADD2(4) MJ_ADD2(5) MJ_ADD2(6) MJ_ADD2(7)
                     MJ_ADD2(8) MJ_ADD2(9) MJ_ADD2(10) MJ_ADD2(11) MJ_ADD2(12) MJ_ADD2(13) MJ_ADD2(14) MJ_ADD2(15)
                 : "+&v"(s), "+&v"(t)
                 : "v"(v), "v"(w), "v"(one));
#undef MJ_ADD2
}

// The strictly sequential sums ((0 + v[0]) + v[1]) + ... of NS staged arrays of kN * kN values, bitwise.
//
// A chain of 8,100 dependent additions is bound by the latency of an FP64 addition (8.5 cycles: 29 us a sum; 12-16
// cycles with operands from LDS, 45 us). So the chain is cut into chunks that run at the same time, one to the 16 lanes of
// a row, two instruction streams a wave: a chunk needs the running sum it starts from, which is only known approximately.
// Its 16 lanes therefore run the chunk from the 16 consecutive doubles around an estimate, and the chunks are put together
// by following, chunk after chunk, which of the next one's starts an end is: a walk over small integers, by lane reads.
// Where an end is none of them, the chunks from there on run again around better estimates: the first of them around its
// true start, the others moved by the same distance. Every pass settles at least one chunk, so the result is always the
// chain's, whatever the data.
//
// The estimates have to know the rounding of the chain so far (some tens of units in the last place at its end), not only
// its sum: each thread runs a link of 17 values from the scan of the links' sums before it, and the scan of what the links
// add, rounded as they round, is within a few units of the running sum. (An addition rounds s + v alike from starts that
// lie some units apart, but for ties and where the sum passes a power of two.)
//
// The pass is bound by the issue of the additions. 64 starts around the tree sums, in 16 chunks (8 a sum for two) with the
// ends looked up one after the other in LDS, took 8.2 us a sum and 13.4 us for
// two; 5.1 and 7.4 us now, of which the estimates are 1.7 and 3.1, the pass 1.3 and 2.2.
// All threads call it; sum[q] is valid in every thread.
constexpr int kStarts = 16, kChunks = 8 * kWaves, kLink = 17, kLinks = (kN * kN + kLink - 1) / kLink;
static_assert(kLinks <= kThreads && kLink % 2 == 1, "a link a thread, no two lanes of a bank group in one bank");
struct ChainLds {
    double ends[kChunks * kStarts], center[kChunks], part[2][2][kWaves], sum[2];
    // which start of the next chunk c the end is, plus 16 (c % 4): a lane number, if the start is one of those run
    int next[kChunks * kStarts];
    int from[2];                  // first chunk of a sum that has to run (again); all of them: done
};
// The sum of the lanes before this one; all: of all lanes. DPP: shifts within the rows of 16, then the last lane of a row
// and of a half to what follows.
template <int CTRL, int ROWS>
__device__ __forceinline__ double dpp_or_zero(double v) {
    const int lo = __builtin_amdgcn_update_dpp(0, __double2loint(v), CTRL, ROWS, 0xf, false);
    const int hi = __builtin_amdgcn_update_dpp(0, __double2hiint(v), CTRL, ROWS, 0xf, false);
    return __hiloint2double(hi, lo);
}
__device__ __forceinline__ double wave_scan(double v, double& all) {
    double s = v;
    s = s + dpp_or_zero<0x111, 0xf>(s);
    s = s + dpp_or_zero<0x112, 0xf>(s);
    s = s + dpp_or_zero<0x114, 0xf>(s);
    s = s + dpp_or_zero<0x118, 0xf>(s);
    s = s + dpp_or_zero<0x142, 0xa>(s);
    s = s + dpp_or_zero<0x143, 0xc>(s);
    all = lane_double(s, 63);
    return dpp_or_zero<0x138, 0xf>(s);
}
template <int NS>
__device__ __forceinline__ void tile_chain(const double* st0, const double* st1, ChainLds& C) {
    constexpr int NC = kChunks / NS, n = kN * kN;  // chunks of a sum
    constexpr int links = (kLinks + NC - 1) / NC, len = links * kLink, steps = (len + 15) / 16;
    constexpr int mid = kStarts / 2, kNone = 1 << 28;
    static_assert(kStarts == 16 && NC % 4 == 0 && NC * links <= kThreads, "a chunk a row of lanes (the last may be empty)");
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, l16 = lane & 15;
    auto bits = [](double x) { return __double_as_longlong(x); };
    // ---- the estimates
    {
        auto link = [&](int w, double s) {
            const int base = min(tid * kLink, n - kLink);  // the last link is short, some threads have none
            const double* const p = (w ? st1 : st0) + base;
            const int skip = tid < kLinks ? tid * kLink - base : kLink;
#pragma unroll
            for (int k = 0; k < kLink; ++k) {
                const double x = p[k];
                s = s + (k >= skip ? x : -0.0);  // s + -0.0 is s
            }
            return s;
        };
        double start[NS], add[NS];
#pragma unroll
        for (int w = 0; w < NS; ++w) add[w] = link(w, 0.0);
#pragma unroll
        for (int round = 0; round < 2; ++round) {
#pragma unroll
            for (int w = 0; w < NS; ++w) {
                double all;
                start[w] = wave_scan(add[w], all);
                if (lane == 0) C.part[round][w][wave] = all;
            }
            __syncthreads();
#pragma unroll
            for (int w = 0; w < NS; ++w) {
                double g = 0.0;
#pragma unroll
                for (int k = 0; k < kWaves; ++k) g = k < wave ? g + C.part[round][w][k] : g;
                start[w] = g + start[w];
                if (round == 0) add[w] = link(w, start[w]) - start[w];
            }
        }
#pragma unroll
        for (int w = 0; w < NS; ++w)
            if (tid % links == 0 && tid / links < NC) C.center[w * NC + tid / links] = start[w];
        if (tid < NS) C.from[tid] = 0;
    }
    __syncthreads();
    const int q = NS == 2 && wave >= kWaves / 2 ? 1 : 0;
    const int g0 = 8 * wave + (lane >> 4), g1 = g0 + 4, c0 = g0 - q * NC, c1 = c0 + 4;  // this lane's chunks
    const double* const v = (q ? st1 : st0) + c0 * len;
    const int n0 = min(len, n - c0 * len), n1 = min(len, n - c1 * len);
    auto val = [&](int h, int k) { return k < (h ? n1 : n0) ? v[4 * h * len + k] : -0.0; };
    for (;;) {
        if (8 * wave + 7 - q * NC >= C.from[q]) {
            double s = __longlong_as_double(bits(C.center[g0]) + (l16 - mid));
            double t = __longlong_as_double(bits(C.center[g1]) + (l16 - mid));
            if (c0 == 0) s = 0.0;
            double v0 = val(0, l16), v1 = val(1, l16);
            for (int k = 0; k < steps; ++k) {
                const double a = v0, b = v1;
                v0 = val(0, 16 * (k + 1) + l16);
                v1 = val(1, 16 * (k + 1) + l16);
                add16x2(s, a, t, b);
            }
            auto put = [&](int g, int c, double end) {
                C.ends[g * kStarts + l16] = end;
                const long long d = c + 1 < NC ? bits(end) - bits(C.center[g + 1]) : 0;
                C.next[g * kStarts + l16] = mid + (int)(d < -kNone ? -kNone : d > kNone ? kNone : d) + ((c + 1) & 3) * 16;
            };
            put(g0, c0, s);
            put(g1, c1, t);
        }
        __syncthreads();
        const int w = wave;  // the sum that this wave puts together
        const int f0 = w < NS ? __builtin_amdgcn_readfirstlane(C.from[w]) : NC;
        if (f0 < NC) {
            int off = ~0, last = 0;  // off: bits that are not those of a lane of the next chunk's, of any step
            if (f0 == 0) {
                int nx[NC / 4];  // chunk 4 k + j in the lanes 16 j .. 16 j + 15
#pragma unroll
                for (int k = 0; k < NC / 4; ++k) nx[k] = C.next[(w * NC + 4 * k) * kStarts + lane];
                int at = mid;
                off = 0;
#pragma unroll
                for (int c = 0; c < NC; ++c) {
                    off |= at ^ (c & 3) * 16;
                    last = at;
                    at = __builtin_amdgcn_readlane(nx[c / 4], at);
                }
            }
            if ((off & ~(kStarts - 1)) == 0) {
                if (lane == 0) {
                    C.sum[w] = C.ends[(w * NC + NC - 1) * kStarts + (last & (kStarts - 1))];
                    C.from[w] = NC;
                }
            } else if (lane == 0) {
                int c = f0, run = mid;
                double s = 0.0;
                while (c < NC && run >= 0 && run < kStarts) {
                    s = C.ends[(w * NC + c) * kStarts + run];
                    run = C.next[(w * NC + c) * kStarts + run] - ((c + 1) & 3) * 16;
                    ++c;
                }
                if (c == NC) C.sum[w] = s;
                C.from[w] = c;
                // chunk c starts from s: move its estimate there and the later ones along
                double g = s;
                for (int k = c; k < NC; ++k) {
                    const double old = C.center[w * NC + k], e = C.ends[(w * NC + k) * kStarts + mid];
                    C.center[w * NC + k] = g;
                    g = e + (g - old);
                }
            }
        }
        __syncthreads();
        if (C.from[0] >= NC && (NS == 1 || C.from[1] >= NC)) return;
    }
}

// ---------------------------------------------------------------------------------------------------- the kernel
// A thread's points, k = 3 i + c: row row0 + i, column l + 32 c (the third clamped to 89); in the padded arrays at
// go[c > 1] bytes + gk(k), in the LDS tile at lo[c > 1] + lk(k). Derived anew wherever it is used (the thread number
// passes through an empty asm statement), so that no derived address stays in registers across the phases.
struct Pos {
    int tid, l, row0, col2;
    unsigned go[2];
    int lo[2];
    __device__ __forceinline__ explicit Pos(int tid_) : tid(tid_) {
        asm volatile("" : "+v"(tid));
        l = tid & 31;
        row0 = kRows * min(tid >> 5, 14);
        col2 = min(l + 64, kN - 1);
        const int cols[2] = {l, col2};
#pragma unroll
        for (int c = 0; c < 2; ++c) {
            go[c] = 8u * (unsigned)(row0 * kNX + cols[c]);
            lo[c] = (row0 + 1) * kPitch + 1 + cols[c];
        }
    }
    static __device__ __forceinline__ constexpr int gk(int k) { return k / 3 * kNX + (k % 3 == 1 ? 32 : 0); }
    static __device__ __forceinline__ constexpr int lk(int k) { return k / 3 * kPitch + (k % 3 == 1 ? 32 : 0); }
    __device__ __forceinline__ bool third() const { return l + 64 < kN; }
    __device__ __forceinline__ int col(int k) const { return k % 3 == 2 ? col2 : l + 32 * (k % 3); }
    // p: column 0 of the tile's first interior row
    __device__ __forceinline__ double ld(const double* p, int k, int d = 0) const {
        return at(p, go[k % 3 == 2], gk(k) + d);
    }
    __device__ __forceinline__ void st(double* p, int k, double v) const { put_at(p, go[k % 3 == 2], gk(k), v); }
};

// The coefficients of one row of a thread's points: W here and at the next column, S of the next row, C.
struct Coef {
    double w[3], e[3], n[3], c[3];
};

// LDS. Tree order: the tile, then aW of the tile's rows (columns 0..90). Fortran order: the tile, over which one sum's
// values are staged, then a second sum's.
constexpr int kWPitch = kN + 1;
constexpr int kLdsTree = kTile + kN * kWPitch, kLdsFort = kTile + kN * kN;

template <int MODE>
__global__ void __launch_bounds__(kThreads, 2) cg2d_resident_kernel(ResDev a) {
    constexpr bool kFort = MODE == MJ_SUM_FORTRAN;
    extern __shared__ __align__(16) double lds[];
    double* const tile = lds;
    double* const cacheW = lds + kTile;
    __shared__ double rows[2][128], edge[4][kN];
    __shared__ typename std::conditional<kFort, ChainLds, int>::type chain;
    __shared__ int s_bad, s_next;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    int g, t;
    resident_unit(a.y.G, g, t);
    const int T = a.y.T;
    const int tbase = t * kPlane + kOL * kNX + kOL;
    // this lane's ring point (lanes below kRingLanes): where its value comes from and goes
    const int epos = wave * kRingLanes + lane;
    const int4 re = lane < kRingLanes ? a.ring[t * 4 * kN + epos] : make_int4(0, 0, -1, 0);
    const bool rneed = lane < kRingLanes && re.z >= 0;
    const int rlds = re.y;
    const int eslot = lane < kRingLanes ? a.pub[t * 4 * kN + epos] : -1;
    uint64_t* const words = a.y.words + (size_t)g * a.y.group_words;
    const unsigned ring_words = 4u * (unsigned)a.y.nslots;
    const bool pA = lane >= kPartA && lane < kPartA + T, pB = lane >= kPartB && lane < kPartB + T;
    const unsigned ring_src = 2u * (unsigned)re.x;
    const unsigned part_src = ring_words + (pB ? 4u * (unsigned)(lane - kPartB) + 2u : pA ? 4u * (unsigned)(lane - kPartA) : 0u);
    unsigned seq = 0;  // number of the last exchange
    unsigned members = 0;

    if (tid == 0) s_bad = 0;
    // the last exchange: ring value (lanes below kRingLanes) and the sums of the partials A, B of every tile
    auto receive = [&](bool ring, bool A, bool B, double& v, double& sA, double& sB, bool largest = false) {
        double w[1] = {0.0};
        const unsigned odd = seq & 1;
        const uint64_t* const p[1] = {words + (ring_src + odd * (ring_words >> 1))};
        const bool need[1] = {ring && rneed};
        double part = -0.0;
        if (!wait_words<2, 1>(a.y, p, need, w, words + (part_src + odd * 4u * (unsigned)T), (A && pA) || (B && pB),
                              part, seq) &&
            lane == 0)
            s_bad = 1;
        v = w[0];
        if (largest)
            sA = part_max(part, T);
        else
            part_sums(part, sA, sB);
    };
    auto publish_part = [&](int q, double v) {
        put_double(words + (ring_words + ((seq & 1) * (unsigned)T + (unsigned)t) * 4 + 2 * q), v, seq);
    };
    // the tile's outermost rows and columns of v, for send_edges to publish after a barrier
    auto keep_edges = [&](const double (&v)[kPts]) {
        const Pos P(tid);
        if (P.row0 == 0) {
#pragma unroll
            for (int c = 0; c < 3; ++c) edge[0][P.col(c)] = v[c];
        }
        if (P.row0 == kN - kRows) {
#pragma unroll
            for (int c = 0; c < 3; ++c) edge[1][P.col(c)] = v[kPts - 3 + c];
        }
        if (P.l == 0) {
#pragma unroll
            for (int i = 0; i < kRows; ++i) edge[2][P.row0 + i] = v[3 * i];
        }
        if (P.l == kN - 65) {
#pragma unroll
            for (int i = 0; i < kRows; ++i) edge[3][P.row0 + i] = v[3 * i + 2];
        }
    };
    auto send_edges = [&]() {
        if (eslot >= 0)
            put_double(words + ((seq & 1) * (ring_words >> 1) + 2u * (unsigned)eslot), edge[0][epos], seq);
    };
    // the products f(k) of the thread's points into the row sums q, or into a staging area (Fortran order)
    auto row_sums = [&](int q, auto&& f) {
        const Pos P(tid);
        const bool third = P.third();
        double w[kRows];
#pragma unroll
        for (int i = 0; i < kRows; ++i) {
            const double v0 = f(3 * i), v1 = f(3 * i + 1), v2 = f(3 * i + 2);
            w[i] = (third ? v0 + v2 : v0) + v1;
        }
        const double s = row_trees(w);
        const int i = row_of_lane(lane);
        if (i >= 0) rows[q][P.row0 + i] = s;
    };
    auto stage = [&](double* st, auto&& f) {
        const Pos P(tid);
#pragma unroll
        for (int k = 0; k < kPts; ++k) st[(P.row0 + k / 3) * kN + P.col(k)] = f(k);
    };
    // exchange seq: the edges of v, and the tile's sum of f as part q; every thread calls it
    auto send_sum = [&](const double (&v)[kPts], int q, auto&& f) {
        keep_edges(v);
        if constexpr (kFort) {
            __syncthreads();  // the staging area lies over the tile: every wave has read it
            send_edges();
            stage(tile, f);
            __syncthreads();
            tile_chain<1>(tile, nullptr, chain);
            if (tid == 0) publish_part(q, chain.sum[0]);
        } else {
            row_sums(0, f);
            __syncthreads();
            send_edges();
            if (wave == 0) {
                const bool h = lane + 64 < kN;
                const double s = wave_tree(rows[0][lane], h ? rows[0][lane + 64] : 0.0, h);
                if (lane == 0) publish_part(q, s);
            }
        }
    };
    // the edges of v, and the tile's sums of f0 and f1 as parts 0 and 1
    auto send_sums = [&](const double (&v)[kPts], auto&& f0, auto&& f1) {
        keep_edges(v);
        if constexpr (kFort) {
            __syncthreads();
            send_edges();
            stage(tile, f0);
            stage(lds + kTile, f1);
            __syncthreads();
            tile_chain<2>(tile, lds + kTile, chain);
            if (tid < 2) publish_part(tid, chain.sum[tid]);
        } else {
            row_sums(0, f0);
            row_sums(1, f1);
            __syncthreads();
            send_edges();
            if (wave < 2) {
                const bool h = lane + 64 < kN;
                const double s = wave_tree(rows[wave][lane], h ? rows[wave][lane + 64] : 0.0, h);
                if (lane == 0) publish_part(wave, s);
            }
        }
    };
    auto put_tile = [&](const double (&v)[kPts], double ring) {
        const Pos P(tid);
#pragma unroll
        for (int k = 0; k < kPts; ++k) tile[P.lo[k % 3 == 2] + P.lk(k)] = v[k];
        if (lane < kRingLanes) tile[rlds & ((1 << 30) - 1)] = (rlds >> 30) & 1 ? -ring : ring;
    };
    // o = A v (isA) or M v of the LDS tile at the thread's points, v its own values; W, S, C the slot's coefficients.
    // The next row's coefficients are loaded while a row is computed; the first row's come from the caller (first_row),
    // loaded before the wait for the other tiles.
    auto row_coef = [&](const Pos& P, auto isA, const double* W, const double* S, const double* C, int i) {
        constexpr bool kCached = decltype(isA)::value && !kFort;
        Coef r;
#pragma unroll
        for (int c = 0; c < 3; ++c) {
            const int k = 3 * i + c;
            r.w[c] = kCached ? 0.0 : P.ld(W, k);
            r.e[c] = kCached ? 0.0 : P.ld(W, k, 1);
            r.n[c] = P.ld(S, k, kNX);
            r.c[c] = P.ld(C, k);
        }
        return r;
    };
    struct First {
        Coef r;
        double s[3];
    };
    auto first_row = [&](auto isA, const double* W, const double* S, const double* C) {
        const Pos P(tid);
        First f;
        f.r = row_coef(P, isA, W, S, C, 0);
#pragma unroll
        for (int c = 0; c < 3; ++c) f.s[c] = P.ld(S, c);
        return f;
    };
    auto stencil = [&](auto isA, const double* W, const double* S, const double* C, const First& f,
                       const double (&v)[kPts], double (&o)[kPts]) {
        constexpr bool kA = decltype(isA)::value, kCached = kA && !kFort;
        const Pos P(tid);
        Coef r = f.r;
        double sn[3] = {f.s[0], f.s[1], f.s[2]};
#pragma unroll
        for (int i = 0; i < kRows; ++i) {
            Coef nx;
            if (i + 1 < kRows) nx = row_coef(P, isA, W, S, C, i + 1);
#pragma unroll
            for (int c = 0; c < 3; ++c) {
                const int k = 3 * i + c, lq = P.lo[c == 2] + P.lk(k);
                const double* cw = cacheW + (P.row0 + i) * kWPitch + P.col(c);
                const double w = kCached ? cw[0] : r.w[c], e = kCached ? cw[1] : r.e[c];
                const double s0 = sn[c], s1 = r.n[c], cc = r.c[c];
                const double vm = i > 0 ? v[k - 3] : tile[lq - kPitch];
                const double vp = i + 1 < kRows ? v[k + 3] : tile[lq + kPitch];
                const double vl = tile[lq - 1], vr = tile[lq + 1], vc = v[k];
                sn[c] = s1;
                o[k] = kA ? w * vl + e * vr + s0 * vm + s1 * vp + cc * vc
                          : cc * vc + w * vl + e * vr + s0 * vm + s1 * vp;
            }
            // the row is computed here: the compiler would otherwise move the arithmetic to its first use, behind
            // every row's loads, and spill what they return
            asm volatile("" : "+v"(o[3 * i]), "+v"(o[3 * i + 1]), "+v"(o[3 * i + 2]));
            r = nx;
        }
    };

    for (;;) {
        // ---- the next member of the queue
        ++members;
        if (tid == 0) {
            s_next = next_member(a.y, g, t, members);
            if (s_next < 0) s_bad = 1;
        }
        __syncthreads();
        if (s_bad) break;
        const int m = s_next;
        if (m >= a.B) return;
        const double* const x0 = a.x0 + m * a.ms;
        const double* const b = a.b + m * a.ms + tbase;
        double* const xg = a.x + m * a.ms;
        const int64_t ob = (int64_t)(a.op_index ? a.op_index[m] : m) * a.oms + tbase;
        const double nm = a.norm[m];
        double x[kPts], r[kPts], s[kPts], zq[kPts];
        const double *const aW = a.aW + ob, *const aS = a.aS + ob, *const aC = a.aC + ob;
        const double *const pW = a.pW + ob, *const pS = a.pS + ob, *const pC = a.pC + ob;
        const std::true_type A{};
        const std::false_type M{};
        double rring = 0.0, sring = 0.0;

        // ---- I0: max |b cg2dNorm|
        {
            const Pos P(tid);
            double mx = 0.0;
#pragma unroll
            for (int k = 0; k < kPts; ++k) mx = fmax(mx, fabs(P.ld(b, k) * nm));
            for (int o = 32; o >= 1; o >>= 1) mx = fmax(mx, __shfl_xor(mx, o, 64));
            if (lane == 0) rows[0][wave] = mx;
            if constexpr (!kFort) {
                for (int q = tid; q < kN * kWPitch; q += kThreads) {
                    const int j = q / kWPitch;
                    cacheW[q] = aW[j * kNX + q - j * kWPitch];
                }
            }
        }
        __syncthreads();
        ++seq;
        if (wave == 0) {
            double mx = lane < kWaves ? rows[0][lane] : 0.0;
            for (int o = 8; o >= 1; o >>= 1) mx = fmax(mx, __shfl_xor(mx, o, 64));
            if (lane == 0) publish_part(0, mx);
        }
        // ---- I1: x = the normalised first guess with its exchanged halo, r = b - A x
        double rhsMax, v, unused;
        receive(false, true, false, v, rhsMax, unused, true);
        const double rhsNorm = rhsMax != 0.0 ? 1.0 / rhsMax : 1.0;
        First f = first_row(A, aW, aS, aC);
        {
            const Pos P(tid);
#pragma unroll
            for (int k = 0; k < kPts; ++k) x[k] = P.ld(x0 + tbase, k) * rhsNorm;
            double xr = 0.0;
            if (lane < kRingLanes) xr = re.z >= 0 ? x0[re.z] * rhsNorm : x0[re.w];
            put_tile(x, xr);
        }
        // halo of x: the first guess, then the exchanged points
        for (int q = tid; q < kPlane; q += kThreads) {
            const int j = q / kNX, i = q - j * kNX;
            if (j < kOL || j >= kOL + kN || i < kOL || i >= kOL + kN) xg[t * kPlane + q] = x0[t * kPlane + q];
        }
        __syncthreads();
        if (s_bad) break;
        for (int k = a.full_off[t] + tid; k < a.full_off[t + 1]; k += kThreads) {
            const int sp = a.full_src[k], sq = sp % kPlane, sj = sq / kNX, si = sq - sj * kNX;
            const bool inner = sj >= kOL && sj < kOL + kN && si >= kOL && si < kOL + kN;
            const double v = inner ? x0[sp] * rhsNorm : x0[sp];
            xg[a.full_dst[k]] = a.full_sign[k] < 0 ? -v : v;
        }
        ++seq;
        stencil(A, aW, aS, aC, f, x, zq);
        {
            const Pos P(tid);
#pragma unroll
            for (int k = 0; k < kPts; ++k) {
                s[k] = P.ld(b, k) * nm * rhsNorm;
                r[k] = s[k] - zq[k];
            }
        }
        send_sums(r, [&](int k) { return r[k] * r[k]; }, [&](int k) { return s[k]; });
        // ---- I2: z = M r, eta(1)
        double err, eta, sumRHS, etaP = 1.0;
        f = first_row(M, pW, pS, pC);
        receive(true, true, true, rring, err, sumRHS);
        put_tile(r, rring);
        __syncthreads();
        if (s_bad) break;
        ++seq;
        stencil(M, pW, pS, pC, f, r, zq);
        send_sum(zq, 1, [&](int k) { return zq[k] * r[k]; });
#pragma unroll
        for (int k = 0; k < kPts; ++k) s[k] = 0.0;
        if (t == 0 && tid == 0) {
            a.diag[m].firstResidual = sqrt(err);
            a.diag[m].sumRHS = sumRHS;
            a.diag[m].rhsMax = rhsMax;
            a.diag[m].outerIters = 0;
            a.diag[m].launches = 0;
        }
        bool bad = false;
        int n = 1;
        for (;; ++n) {
            // ---- B(n): stopping rule on err(n-1); s = z + beta s, q = A s, sigma. The rule comes behind the barrier and
            // the look at s_bad: a wave whose wait failed has no err, and all waves must take the same way.
            f = first_row(A, aW, aS, aC);
            {
                double e;
                receive(true, n > 1, true, v, e, eta);
                if (n > 1) err = e;
            }
            const double beta = eta / etaP;
#pragma unroll
            for (int k = 0; k < kPts; ++k) s[k] = zq[k] + beta * s[k];
            sring = rneed ? v + beta * sring : 0.0;
            put_tile(s, sring);
            __syncthreads();
            if ((bad = s_bad)) break;
            if (!(n - 1 < a.max_iters) || err < a.tol_sq) break;
            ++seq;
            stencil(A, aW, aS, aC, f, s, zq);
            send_sum(zq, 0, [&](int k) { return s[k] * zq[k]; });
            // ---- C(n): x += alpha s, r -= alpha q, z = M r, err, eta
            f = first_row(M, pW, pS, pC);
            double sigma;
            receive(true, true, false, v, sigma, unused);
            const double alpha = eta / sigma;
#pragma unroll
            for (int k = 0; k < kPts; ++k) {
                x[k] = x[k] + alpha * s[k];
                r[k] = r[k] - alpha * zq[k];
            }
            rring = rneed ? rring - alpha * v : 0.0;
            put_tile(r, rring);
            __syncthreads();
            if ((bad = s_bad)) break;
            ++seq;
            stencil(M, pW, pS, pC, f, r, zq);
            send_sums(zq, [&](int k) { return r[k] * r[k]; }, [&](int k) { return zq[k] * r[k]; });
            etaP = eta;
        }
        if (bad) break;
        // un-normalise x (cg2d.F:380-395)
        {
            const Pos P(tid);
#pragma unroll
            for (int k = 0; k < kPts; ++k) P.st(xg + tbase, k, x[k] / rhsNorm);
        }
        if (t == 0 && tid == 0) {
            a.diag[m].lastResidual = sqrt(err);
            a.diag[m].numIters = n - 1;
            a.diag[m].converged = err < a.tol_sq ? 1 : 0;
        }
        __syncthreads();  // every wave has looked at s_bad; the next member's first wait may set it
    }
}

__global__ void res_init_kernel(uint64_t* words, size_t n, int* queue, int* error) {
    for (size_t k = (size_t)blockIdx.x * blockDim.x + threadIdx.x; k < n; k += (size_t)gridDim.x * blockDim.x)
        words[k] = 0;
    if (blockIdx.x == 0 && threadIdx.x == 0) {
        *queue = 0;
        *error = 0;
    }
}

// After a launch in which a wait failed, every member's record says so. Not the launch's own business: its workgroups end
// one by one, and one that was served in time may still write a record after the others have left.
__global__ void __launch_bounds__(256) res_failed_kernel(const int* error, mj_cg2d_diag* diag, int B) {
    if (*error == 0) return;
    for (int m = threadIdx.x; m < B; m += 256) diag[m].converged = -2;
}

// The order in which a batch with several operators is taken: the members that need most iterations first, so that the
// last ones to start are short (a group that starts a long member when the others are done leaves them idle). The number
// of iterations grows as the diagonal's excess over the face coefficients (the free-surface term) falls; a sample of
// each member's operator tells (key). It decides nothing but the order.
constexpr int kOrderMax = 4096, kSampleStep = 8;  // largest batch that is ordered; every 8th row is looked at
__global__ void __launch_bounds__(256) res_key_kernel(const double* aW, const double* aS, const double* aC, int64_t oms,
                                                      const int32_t* op_index, int T, unsigned* key) {
    __shared__ float s_sum[2][4];
    const int m = blockIdx.x, tid = threadIdx.x;
    const int64_t ob = (int64_t)(op_index ? op_index[m] : m) * oms;
    constexpr int rows = (kN + kSampleStep - 1) / kSampleStep;
    float excess = 0.0f, diag = 0.0f;
    for (int i = tid; i < T * rows * kN; i += 256) {
        const int t = i / (rows * kN), r = i - t * rows * kN, j = r / kN;
        const int64_t p = ob + t * kPlane + (kOL + j * kSampleStep) * kNX + kOL + (r - j * kN);
        const double c = aC[p];
        excess += (float)fabs(aW[p] + aW[p + 1] + aS[p] + aS[p + kNX] + c);
        diag += (float)fabs(c);
    }
    for (int o = 32; o >= 1; o >>= 1) {
        excess += __shfl_xor(excess, o, 64);
        diag += __shfl_xor(diag, o, 64);
    }
    if ((tid & 63) == 0) {
        s_sum[0][tid >> 6] = excess;
        s_sum[1][tid >> 6] = diag;
    }
    __syncthreads();
    if (tid == 0) {
        for (int w = 1; w < 4; ++w) {
            excess += s_sum[0][w];
            diag += s_sum[1][w];
        }
        key[m] = __float_as_uint(excess / diag);  // >= 0: ordered as its bits (NaN too)
    }
}
__global__ void __launch_bounds__(1024) res_order_kernel(const unsigned* key, int B, int* order) {
    __shared__ unsigned s_key[kOrderMax];
    for (int m = threadIdx.x; m < B; m += 1024) s_key[m] = key[m];
    __syncthreads();
    for (int m = threadIdx.x; m < B; m += 1024) {
        int rank = 0;
        for (int q = 0; q < B; ++q) rank += s_key[q] < s_key[m] || (s_key[q] == s_key[m] && q < m);
        order[rank] = m;
    }
}

}  // namespace

int resident_prepare(const mj_halo_plan* P, const mj_cg2d_ops* ops, const mj_cg2d_config* cfg, const void* kfn,
                     int threads, size_t lds, void* workspace, size_t workspace_bytes, hipStream_t st, ResSync* y,
                     bool* ok) {
    *ok = false;
    int dev = 0, ncu = 0, coop = 0, clk_khz = 0, max_lds = 0, per_cu = 0;
    MJ_HIP(hipGetDevice(&dev));
    MJ_HIP(hipDeviceGetAttribute(&ncu, hipDeviceAttributeMultiprocessorCount, dev));
    MJ_HIP(hipDeviceGetAttribute(&coop, hipDeviceAttributeCooperativeLaunch, dev));
    MJ_HIP(hipDeviceGetAttribute(&clk_khz, hipDeviceAttributeWallClockRate, dev));
    MJ_HIP(hipDeviceGetAttribute(&max_lds, hipDeviceAttributeMaxSharedMemoryPerBlock, dev));
    if (!coop || (size_t)max_lds < lds) return MJ_OK;
    MJ_HIP(hipFuncSetAttribute(kfn, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
    MJ_HIP(hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, kfn, threads, lds));
    y->T = P->ntiles;
    y->nslots = P->res_nslots;
    y->B = cfg->batch;
    y->G = std::min(y->B, per_cu * ncu / y->T);
    if (y->G < 1) return MJ_OK;
    y->group_words = ((size_t)4 * y->nslots + (size_t)8 * y->T + 31) / 32 * 32;
    const size_t next = (size_t)y->G * y->group_words, misc = (next + y->G + 31) / 32 * 32;  // words
    if ((misc + 32 + y->B) * 8 > workspace_bytes) return MJ_OK;
    uint64_t* const w = (uint64_t*)workspace;
    y->words = w;
    y->next = w + next;
    y->queue = (int*)(w + misc);
    y->error = (int*)(w + misc + 8);
    y->limit = (unsigned long long)((clk_khz > 0 ? clk_khz : 100000) * 1000.0 * P->res_wait_s);
    hipLaunchKernelGGL(res_init_kernel, dim3(64), dim3(256), 0, st, w, misc, y->queue, y->error);
    MJ_HIP(hipGetLastError());
    y->order = nullptr;
    if (ops->member_stride != 0 && y->B > y->G && y->B <= kOrderMax) {
        unsigned* const key = (unsigned*)(w + misc + 32);
        int* const order = (int*)key + y->B;
        hipLaunchKernelGGL(res_key_kernel, dim3(y->B), dim3(256), 0, st, ops->aW2d, ops->aS2d, ops->aC2d,
                           ops->member_stride, ops->op_index, y->T, key);
        MJ_HIP(hipGetLastError());
        hipLaunchKernelGGL(res_order_kernel, dim3(1), dim3(1024), 0, st, key, y->B, order);
        MJ_HIP(hipGetLastError());
        y->order = order;
    }
    *ok = true;
    return MJ_OK;
}

int resident_launch(const void* kfn, int threads, void** args, size_t lds, const ResSync& y, mj_cg2d_diag* diag,
                    hipStream_t st) {
    MJ_HIP(hipLaunchCooperativeKernel(kfn, dim3(y.G * y.T), dim3(threads), args, (unsigned)lds, st));
    hipLaunchKernelGGL(res_failed_kernel, dim3(1), dim3(256), 0, st, y.error, diag, y.B);
    MJ_HIP(hipGetLastError());
    return MJ_OK;
}

int stream_capturing(hipStream_t st, bool* capturing) {
    hipStreamCaptureStatus s = hipStreamCaptureStatusNone;
    MJ_HIP(hipStreamIsCapturing(st, &s));
    *capturing = s != hipStreamCaptureStatusNone;
    return MJ_OK;
}

bool resident_fits(const mj_halo_plan* P, const mj_cg2d_config* c) {
    return c->sNx == kN && c->sNy == kN && c->OL == kOL && c->ntiles <= kResMaxTiles && P->res_ok;
}

int resident_solve(mj_halo_plan* P, const mj_cg2d_ops* ops, const double* b, const double* x0, double* x,
                   const double* cg2dNorm, const mj_cg2d_config* cfg, void* workspace, size_t workspace_bytes,
                   mj_cg2d_diag* diag, hipStream_t st, bool* done) {
    *done = false;
    const void* kfn = cfg->sum_order == MJ_SUM_FORTRAN ? (const void*)cg2d_resident_kernel<MJ_SUM_FORTRAN>
                                                       : (const void*)cg2d_resident_kernel<MJ_SUM_TREE>;
    const size_t lds = (cfg->sum_order == MJ_SUM_FORTRAN ? kLdsFort : kLdsTree) * sizeof(double);
    ResDev a{};
    bool ok = false;
    int rc = resident_prepare(P, ops, cfg, kfn, kThreads, lds, workspace, workspace_bytes, st, &a.y, &ok);
    if (rc || !ok) return rc;
    a.B = cfg->batch;
    a.ms = cfg->member_stride;
    a.oms = ops->member_stride;
    a.aW = ops->aW2d;
    a.aS = ops->aS2d;
    a.aC = ops->aC2d;
    a.pW = ops->pW;
    a.pS = ops->pS;
    a.pC = ops->pC;
    a.b = b;
    a.x0 = x0;
    a.x = x;
    a.norm = cg2dNorm;
    a.tol_sq = cfg->tolerance * cfg->tolerance;  // cg2d.F:111
    a.max_iters = cfg->max_iters;
    a.full_off = P->cg_full_off;
    a.full_dst = P->cg_full_dst;
    a.full_src = P->cg_full_src;
    a.full_sign = P->cg_full_sign;
    a.op_index = ops->op_index;
    a.ring = P->res_ring;
    a.pub = P->res_pub;
    a.diag = diag;
    void* args[] = {(void*)&a};
    if ((rc = resident_launch(kfn, kThreads, args, lds, a.y, diag, st))) return rc;
    *done = true;
    return MJ_OK;
}

// The ring entries and publication slots of the resident solves, from the per-tile ring tables of the plan (held lock).
int ensure_resident_tables(mj_halo_plan* P, const std::vector<int32_t>& roff, const std::vector<int32_t>& rdst,
                           const std::vector<int32_t>& rsrc, const std::vector<int8_t>& rsg) {
    const int nx = P->nx, plane = P->nx * P->ny, T = P->ntiles, OL = kOL;
    if (nx != kNX || P->ny != kNX || T > kResMaxTiles) return MJ_OK;
    std::vector<int4> ring((size_t)T * 4 * kN);
    std::vector<int32_t> pub((size_t)T * 4 * kN, -1);
    int nslots = 0;
    for (int t = 0; t < T; ++t) {
        if (roff[t + 1] - roff[t] != 4 * kN) return MJ_OK;
        for (int k = 0; k < 4 * kN; ++k) {
            const int e = roff[t] + k, d = rdst[e] % plane, s = rsrc[e];
            int slot = 0;
            if (s >= 0) {
                const int sq = s % plane, sj = sq / nx - OL, si = sq % nx - OL;
                // sources lie on the outermost rows and columns (the kernel publishes those)
                int pos = -1;
                if (sj == 0) pos = si;
                else if (sj == kN - 1) pos = kN + si;
                else if (si == 0) pos = 2 * kN + sj;
                else if (si == kN - 1) pos = 3 * kN + sj;
                if (pos < 0) return MJ_OK;
                int32_t& p = pub[(size_t)(s / plane) * 4 * kN + pos];
                if (p < 0) p = nslots++;
                slot = p;
            }
            const int lds = (d / nx - OL + 1) * kPitch + (d % nx - OL + 1);
            ring[(size_t)t * 4 * kN + k] = make_int4(slot, lds | (rsg[e] < 0 ? 1 << 30 : 0), s, rdst[e]);
        }
    }
    MJ_HIP(hipMalloc((void**)&P->res_ring, ring.size() * sizeof(int4)));
    MJ_HIP(hipMemcpy(P->res_ring, ring.data(), ring.size() * sizeof(int4), hipMemcpyHostToDevice));
    MJ_HIP(hipMalloc((void**)&P->res_pub, pub.size() * sizeof(int32_t)));
    MJ_HIP(hipMemcpy(P->res_pub, pub.data(), pub.size() * sizeof(int32_t), hipMemcpyHostToDevice));
    P->res_nslots = std::max(nslots, 1);
    P->res_ok = 1;
    return MJ_OK;
}

}  // namespace mj
