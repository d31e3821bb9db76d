// Device building blocks of the resident CG2D solves (FP64 and mixed precision): tagged words between the workgroups of
// a member, the queue of members, and cross-lane sums.
#pragma once

#include "mj_common.h"
#include "mj_resident.h"

namespace mj {

constexpr int kPartA = 32, kPartB = 48;  // lanes that poll the partial sums of tile lane - kPartA / - kPartB
static_assert(kPartB - kPartA >= kResMaxTiles && 64 - kPartB >= kResMaxTiles, "poll lanes");

// ---------------------------------------------------------------------------------------------------- tagged words
__device__ __forceinline__ void put_word(uint64_t* p, uint64_t v) {
    __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ uint64_t get_word(const uint64_t* p) {
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
// A double is two neighbouring words, 16-byte aligned, stored and loaded as one access with the cache policy of the words
// (agent scope): each half carries its tag, so it does not matter whether the access is one. The words of an exchange are
// what bounds it (they go past the L2s): with two accesses a double 64 members to 1e-12 took 20.3 ms and 128 members of the
// mixed solve 8.9; 17.4 and 7.6 with one. Polling more often than a poll takes (two in flight) made 22.7 and 12.8 of it.
typedef unsigned ResPair __attribute__((ext_vector_type(4)));
__device__ __forceinline__ void put_double(uint64_t* p, double v, unsigned tag) {
    const ResPair w = {(unsigned)__double2loint(v), tag, (unsigned)__double2hiint(v), tag};
    // a store of more than 8 bytes must not be followed at once by a write of its data registers (the compiler sees to
    // that for its own stores only)
    asm volatile("global_store_dwordx4 %0, %1, off sc1\n\ts_nop 1" : : "v"(p), "v"(w) : "memory");
}
__device__ __forceinline__ void get_pair(const uint64_t* p, uint64_t& a, uint64_t& b) {
    ResPair w;
    asm volatile("global_load_dwordx4 %0, %1, off sc1\n\ts_waitcnt vmcnt(0)" : "=&v"(w) : "v"(p) : "memory");
    a = (uint64_t)w.y << 32 | w.x;
    b = (uint64_t)w.w << 32 | w.z;
}
// Whether a wait that began at t0 (0: now) is to end: it took too long, or another workgroup gave up. The same answer in
// every lane (one lane's look at the error).
__device__ __forceinline__ bool gave_up(const ResSync& a, unsigned long long& t0) {
    const unsigned long long now = wall_clock64();
    if (t0 == 0) t0 = now;
    const int error = __hip_atomic_load(a.error, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    if (__builtin_amdgcn_readfirstlane(error) == 0 && now - t0 < a.limit) return false;
    __hip_atomic_store(a.error, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    return true;
}
__device__ __forceinline__ void put_float(uint64_t* p, float v, unsigned tag) {
    put_word(p, (uint64_t)tag << 32 | __float_as_uint(v));
}
// The words published with this tag: PW words at each p[i] for the lanes with need_p[i] (a double, or a float in the low
// half of one word) and a double at q for those with need_q; the whole wave waits together. False when the wait timed
// out or another workgroup gave up.
template <int PW, int N>
__device__ __forceinline__ bool wait_words(const ResSync& a, const uint64_t* const (&p)[N], const bool (&need_p)[N],
                                           double (&vp)[N], const uint64_t* q, bool need_q, double& vq, unsigned tag) {
    uint64_t p0[N], p1[N], q0 = 0, q1 = 0;
    unsigned spins = 0;
    unsigned long long t0 = 0;
    bool wp[N], wq = need_q;
#pragma unroll
    for (int i = 0; i < N; ++i) {
        wp[i] = PW > 0 && need_p[i];
        p0[i] = p1[i] = 0;
    }
    for (;;) {
#pragma unroll
        for (int i = 0; i < N; ++i)
            if (wp[i]) {
                if (PW > 1)
                    get_pair(p[i], p0[i], p1[i]);
                else
                    p0[i] = get_word(p[i]);
            }
        if (wq) get_pair(q, q0, q1);
        bool wait = false;
#pragma unroll
        for (int i = 0; i < N; ++i) {
            if (wp[i]) wp[i] = (unsigned)(p0[i] >> 32) != tag || (PW > 1 && (unsigned)(p1[i] >> 32) != tag);
            wait = wait || wp[i];
        }
        if (wq) wq = (unsigned)(q0 >> 32) != tag || (unsigned)(q1 >> 32) != tag;
        if (!__any(wait || wq)) break;
        if (((++spins & 1023u) == 0 || a.limit == 0) && gave_up(a, t0)) return false;
    }
#pragma unroll
    for (int i = 0; i < N; ++i)
        if (PW > 0 && need_p[i]) vp[i] = __hiloint2double((int)(unsigned)p1[i], (int)(unsigned)p0[i]);
    if (need_q) vq = __hiloint2double((int)(unsigned)q1, (int)(unsigned)q0);
    return true;
}
__device__ __forceinline__ double lane_double(double v, int lane) {
    return __hiloint2double(__builtin_amdgcn_readlane(__double2hiint(v), lane),
                            __builtin_amdgcn_readlane(__double2loint(v), lane));
}
// The group's next member (members: which of its members it is, from 1; a.B: none is left), -1 when a wait timed out.
// One thread of a workgroup calls it; tile 0's takes the member from the queue and tells the others.
__device__ __forceinline__ int next_member(const ResSync& a, int g, int t, unsigned members) {
    uint64_t* const w = a.next + g;
    if (t == 0) {
        const int i = atomicAdd(a.queue, 1), m = i >= a.B ? a.B : a.order ? a.order[i] : i;
        put_word(w, (uint64_t)members << 32 | (unsigned)m);
        return m;
    }
    unsigned spins = 0;
    unsigned long long t0 = 0;
    for (;;) {
        const uint64_t v = get_word(w);
        if ((unsigned)(v >> 32) == members) return (int)(unsigned)v;
        if (((++spins & 1023u) == 0 || a.limit == 0) && gave_up(a, t0)) return -1;
    }
}
// Unit of this block: group g, tile t. The blocks of an XCD (b % 8) take consecutive units, tile-major, so that few
// tiles' coefficients pass through an L2.
__device__ __forceinline__ void resident_unit(int G, int& g, int& t) {
    const int n = gridDim.x, xcd = blockIdx.x % 8;
    const int u = xcd * (n / 8) + min(xcd, n % 8) + blockIdx.x / 8;
    t = u / G;
    g = u - t * G;
}
// A value that every lane holds, in scalar registers.
__device__ __forceinline__ double uniform(double v) { return lane_double(v, 0); }

// ---------------------------------------------------------------------------------------------------- cross-lane sums
// a: the even rows of 16 lanes from a, the odd ones from b's even; b: a's odd rows, b's odd rows.
__device__ __forceinline__ void swap16(double& a, double& b) {
    const auto lo = __builtin_amdgcn_permlane16_swap((unsigned)__double2loint(a), (unsigned)__double2loint(b), false, false);
    const auto hi = __builtin_amdgcn_permlane16_swap((unsigned)__double2hiint(a), (unsigned)__double2hiint(b), false, false);
    a = __hiloint2double((int)hi[0], (int)lo[0]);
    b = __hiloint2double((int)hi[1], (int)lo[1]);
}
// a: the lower halves of a and b; b: their upper halves.
__device__ __forceinline__ void swap32(double& a, double& b) {
    const auto lo = __builtin_amdgcn_permlane32_swap((unsigned)__double2loint(a), (unsigned)__double2loint(b), false, false);
    const auto hi = __builtin_amdgcn_permlane32_swap((unsigned)__double2hiint(a), (unsigned)__double2hiint(b), false, false);
    a = __hiloint2double((int)hi[0], (int)lo[0]);
    b = __hiloint2double((int)hi[1], (int)lo[1]);
}
template <int CTRL, int BANKS>
__device__ __forceinline__ double dpp(double old, double v) {
    const int lo = __builtin_amdgcn_update_dpp(__double2loint(old), __double2loint(v), CTRL, 0xf, BANKS, false);
    const int hi = __builtin_amdgcn_update_dpp(__double2hiint(old), __double2hiint(v), CTRL, 0xf, BANKS, false);
    return __hiloint2double(hi, lo);
}
// s = s + v[0], s + v[1], ... over the 16 lanes of the lane's row of 16; fma(v, 1, s) is the addition (one rounding),
// and its operand can be broadcast within the instruction.
__device__ __forceinline__ double add16(double s, double v) {
    double one = 1.0;
#define MJ_ADD1(i) "v_fmac_f64_dpp %0, %1, %2 row_newbcast:" #i " row_mask:0xf bank_mask:0xf\n"
    asm volatile("s_nop 1\n" MJ_ADD1(0) MJ_ADD1(1) MJ_ADD1(2) MJ_ADD1(3) MJ_ADD1(4) MJ_ADD1(5) MJ_ADD1(6) MJ_ADD1(7)
                     MJ_ADD1(8) MJ_ADD1(9) MJ_ADD1(10) MJ_ADD1(11) MJ_ADD1(12) MJ_ADD1(13) MJ_ADD1(14) MJ_ADD1(15)
                 : "+&v"(s)
                 : "v"(v), "v"(one));
#undef MJ_ADD1
    return s;
}
// Tile-order sums of the partials in lanes kPartA.. and kPartB.. (rows 2 and 3 of 16 lanes; -0.0 in those of no tile:
// s + -0.0 is s).
__device__ __forceinline__ void part_sums(double v, double& A, double& B) {
    const double s = add16(0.0, v);
    A = lane_double(s, kPartA);
    B = lane_double(s, kPartB);
}

// The largest of the partials A >= 0 of T tiles.
__device__ __forceinline__ double part_max(double v, int T) {
    double A = 0.0;
    for (int k = 0; k < T; ++k) A = fmax(A, lane_double(v, kPartA + k));
    return A;
}
// An exchange of the mixed solve: the words at p for the lanes with need_p; and the sums of the partials A, B (at q, in the
// lanes with need_q), or with `largest` the largest A >= 0, uniform in every wave. One wave of the workgroup (mine) polls
// the partials and tells the others through LDS: with every wave polling them, the few lines that hold a member's sums were
// read by all its waves, and 128 members took 7.6 ms; 6.7 with one. (In the FP64 solve every wave polls them beside its
// ring values: there the wait for the one costs more, 18.0 ms against 17.4 for 64 members to 1e-12.) A barrier has to lie
// between two calls.
struct PartBox {
    double a, b;
    unsigned tag;
};
template <int PW, int N>
__device__ __forceinline__ bool wait_exchange(const ResSync& a, PartBox& box, bool mine, int lane,
                                              const uint64_t* const (&p)[N], const bool (&need_p)[N], double (&vp)[N],
                                              const uint64_t* q, bool need_q, bool largest, double& sA, double& sB,
                                              unsigned tag) {
    double part = -0.0;
    const bool ok = wait_words<PW, N>(a, p, need_p, vp, q, mine && need_q, part, tag);
    if (mine) {
        sB = 0.0;
        if (largest)
            sA = part_max(part, a.T);
        else
            part_sums(part, sA, sB);
        if (lane == 0) {
            box.a = sA;
            box.b = sB;
        }
        // after a wait that timed out, too: the others go on to the barrier behind which they look at the error
        __hip_atomic_store(&box.tag, tag, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_WORKGROUP);
    } else {
        while (__hip_atomic_load(&box.tag, __ATOMIC_ACQUIRE, __HIP_MEMORY_SCOPE_WORKGROUP) != tag)
            __builtin_amdgcn_s_sleep(1);
        sA = uniform(box.a);
        sB = uniform(box.b);
    }
    return ok;
}

}  // namespace mj
