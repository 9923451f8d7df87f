// rcb_small.h -- whole RCB problems of few points, one workgroup each.
//
// The general path launches a kernel per pass and level and waits for its
// counters: about 15 launches for 3 levels, and a second run when a search
// outlasts the queued passes.  A problem of at most kSmallPoints points fits
// one workgroup's registers, so one launch takes it from the caller's points
// to the caller's ids: box, weight sum and weight kind by a workgroup
// reduction, the levels by sub_levels (rcb_subtree.h), the ids from the slots.
#pragma once

#include "rcb_subtree.h"

namespace coupe_hip {

constexpr uint32_t kSmallPoints = 16384;
constexpr uint32_t kSmallLevels = kSubLevels;

// One small problem: its points and ids at src / src_pt of the caller's arrays.
struct SmallProblem {
    uint64_t src;          // first point in the caller's weights and ids
    uint64_t src_pt;       // offset of its first coordinate in the caller's points
    double tol;
    uint32_t count;
    uint32_t levels;
};

// What a problem reports (report[blockIdx.x]): the weight kinds met (not whole
// numbers or not exactly summable, outside int32, outside [0, 65535]) and
// whether a search did not end.
enum : uint32_t { kSmallReal = 1, kSmallWide = 2, kSmallNot16 = 4, kSmallError = 8, kSmallNegative = 16 };

// Reductions of a workgroup in LDS.
struct SmallShared {
    uint32_t ctr[4];
    uint32_t min_slot;
    uint32_t flags;
    float lo[16][kMaxDim], hi[16][kMaxDim];
    double sf[16], sa[16];
    uint64_t su[16];
};
static_assert(sizeof(SmallShared) <= kSubMisc, "reductions");

// Sum over a wavefront of a 64-bit integer, a double, extremes of floats
// (row shifts, no LDS): rcb_device.h's wave totals; min and max by ordered keys.
__device__ __forceinline__ float wave_low(float v) { return key_f32(wave_total_min(f32_key(v))); }
__device__ __forceinline__ float wave_high(float v) { return key_f32(~wave_total_min(~f32_key(v))); }

// Selects the coordinate of a uniform axis from points in registers: bit masks
// made once per pass (an indexed register array would live in scratch).
template <int D>
struct AxisSelect {
    uint32_t m[D];
    __device__ __forceinline__ explicit AxisSelect(int a) {
#pragma unroll
        for (int k = 0; k < D; k++) {
            m[k] = a == k ? 0xffffffffu : 0u;
            asm volatile("" : "+v"(m[k]));
        }
    }
    __device__ __forceinline__ float operator()(const float (&x)[D]) const {
        uint32_t r = 0;
#pragma unroll
        for (int k = 0; k < D; k++) r |= __builtin_bit_cast(uint32_t, x[k]) & m[k];
        return __builtin_bit_cast(float, r);
    }
};

// Where a point's weight comes from in each pass: a register of the
// accumulator type; half a register (32 points per thread, whole weights in
// [0, 65535]); the caller's array again (32 points per thread, other weights).
enum : int { kWeightAcc, kWeight16, kWeightLoad };

constexpr int kAhead = 4;   // points of a lane whose lookups are issued together
constexpr int kLoad = 8;    // points of a lane loaded together

// The levels of a subtree of `count` points in registers, their weights
// win(i); the slots two to a register.  Points are taken kAhead at a time, up to
// the uniform end.
template <int IT>
struct RegSlots {
    uint32_t two[IT / 2];
    __device__ __forceinline__ uint32_t operator()(int k) const {
        return k & 1 ? two[k / 2] >> 16 : two[k / 2] & 0xffffu;
    }
};
template <int D, int TPB, int IT, int KW, typename WIN, typename Acc, typename Weight, typename Split>
__device__ __forceinline__ bool reg_levels(uint32_t count, const float (&x)[IT][D], Weight &&win,
                                           const SubRoot &R, Acc sum, uint32_t *ctr, RegSlots<IT> &slot,
                                           Split &&split_out) {
    constexpr int B = kAhead;
    static_assert(IT % B == 0, "whole groups of points");
    const uint32_t tid = threadIdx.x;
    SubTree<Acc, TPB> T(sub_slots(R.levels));
    uint32_t w16[KW == kWeight16 ? IT / 2 : 1];
    Acc wacc[KW == kWeightAcc ? IT : 1];
#pragma unroll
    for (int k = 0; k < IT / 2; k++) slot.two[k] = 0;
    if constexpr (KW != kWeightLoad) {
#pragma unroll
        for (int k = 0; k < IT; k++) {
            const uint32_t i = (uint32_t)(k * TPB) + tid;
            const WIN v = win(i < count ? i : count - 1);
            if constexpr (KW == kWeightAcc) wacc[k] = AccOps<Acc>::of(v);
            else w16[k / 2] = k & 1 ? w16[k / 2] | (uint32_t)v << 16 : (uint32_t)v;
        }
    }
    return sub_levels<D, TPB, Acc>(
        T, R, count, sum, ctr,
        [&](int nb, int a) {
            const AxisSelect<D> on(a);
            uint32_t first = tid;   // opaque: what follows from it is not kept across passes
            asm volatile("" : "+v"(first));
#pragma unroll
            for (int k0 = 0; k0 < IT; k0 += B) {
                if ((uint32_t)(k0 * TPB) >= count) continue;   // uniform: no point left
                uint32_t s[B];
                float xa[B];
                Acc w[B];
                bool valid[B];
#pragma unroll
                for (int j = 0; j < B; j++) {
                    const int k = k0 + j;
                    const uint32_t i = (uint32_t)(k * TPB) + first;
                    valid[j] = i < count;
                    s[j] = slot(k);   // opaque like the weights: nothing made of them is kept
                    asm volatile("" : "+v"(s[j]));
                    xa[j] = on(x[k]);
                    if constexpr (KW == kWeightLoad) w[j] = AccOps<Acc>::of(win(valid[j] ? i : count - 1));
                    else if constexpr (KW == kWeight16) {
                        uint32_t v = w16[k / 2];
                        asm volatile("" : "+v"(v));
                        w[j] = (Acc)(k & 1 ? v >> 16 : v & 0xffffu);
                    } else {
                        w[j] = wacc[k];
                        asm volatile("" : "+v"(w[j]));
                    }
                }
                sub_bin<B>(T, s, [&](int j, uint32_t) { return xa[j]; }, w, valid, nb, R.packed);
            }
        },
        [&](int a) {
            const AxisSelect<D> on(a);
#pragma unroll
            for (int k0 = 0; k0 < IT; k0 += B) {
                if ((uint32_t)(k0 * TPB) >= count) continue;
                float t[B];
#pragma unroll
                for (int j = 0; j < B; j++) t[j] = T.at(slot(k0 + j)).win.x;
#pragma unroll
                for (int j = 0; j < B; j += 2) {
                    const int k = k0 + j;
                    const uint32_t s0 = 2 * slot(k) + (on(x[k]) >= t[j] ? 1u : 0u);
                    const uint32_t s1 = 2 * slot(k + 1) + (on(x[k + 1]) >= t[j + 1] ? 1u : 0u);
                    slot.two[k / 2] = s0 | s1 << 16;
                }
            }
        },
        split_out);
}

// One small problem: its levels, then its ids.
template <int D, int TPB, int IT, int KW, typename WIN, typename Acc>
__device__ __forceinline__ void small_run(const SmallProblem &P, const float (&x)[IT][D], const WIN *__restrict__ win,
                                          const SubRoot &R, Acc sum, SmallShared &sh,
                                          uint64_t *__restrict__ out, uint32_t kind, uint32_t *report) {
    const uint32_t tid = threadIdx.x;
    RegSlots<IT> slot;
    const bool ok = reg_levels<D, TPB, IT, KW, WIN, Acc>(P.count, x, [&](uint32_t i) { return win[i]; }, R, sum, sh.ctr,
                                                        slot, [](uint32_t, uint32_t, uint32_t, uint32_t, float) {});
    // ids: the leaf's path less the smallest one present (:589-601, :698-702)
    uint32_t m = 0xffffffffu;
#pragma unroll
    for (int k = 0; k < IT; k++) {
        const uint32_t i = (uint32_t)(k * TPB) + tid;
        m = i < P.count ? min(m, slot(k)) : m;
    }
    m = wave_total_min(m);
    if (lane_id() == 0) atomicMin(&sh.min_slot, m);
    __syncthreads();
    const uint32_t off = sh.min_slot;
#pragma unroll
    for (int k = 0; k < IT; k++) {
        const uint32_t i = (uint32_t)(k * TPB) + tid;
        if (i < P.count) out[P.src + i] = (uint64_t)(slot(k) - off);
    }
    if (tid == 0) *report = kind | (ok ? 0u : kSmallError);
}

// The points of a lane as f32 (`as f32`, :677), clamped to the last one past
// the end: from a resident working copy, mapped by a rotation (Rib), or as given.
template <int D, int TPB, int IT, typename Load>
__device__ __forceinline__ void small_points(uint32_t count, float (&x)[IT][D], Load &&load) {
    constexpr int L = IT < kLoad ? IT : kLoad;
#pragma unroll
    for (int k0 = 0; k0 < IT; k0 += L) {
        if ((uint32_t)(k0 * TPB) >= count) {   // uniform: no point left
#pragma unroll
            for (int j = 0; j < L; j++)
#pragma unroll
                for (int a = 0; a < D; a++) x[k0 + j][a] = 0.0f;
            continue;
        }
#pragma unroll
        for (int j = 0; j < L; j++) {
            const uint32_t i = (uint32_t)((k0 + j) * TPB) + threadIdx.x;
            load((uint64_t)(i < count ? i : count - 1), x[k0 + j]);
        }
    }
}

// What a launch of small problems reads and writes.  c0 (non-null): the f32
// coordinates of a resident working copy replace the points; rot_on: every
// point mapped by rot first (Rib).
template <typename WIN>
struct SmallArrays {
    const double *pts;
    const float *c0, *c1, *c2;
    const WIN *win;
    uint64_t *out;
    int wrap32, rot_on;
    Rotation rot;
};

template <int D, int TPB, int IT, typename WIN>
__device__ __forceinline__ void small_problem(const SmallProblem &P, const SmallArrays<WIN> &A, uint32_t *report) {
    SmallShared &sh = *(SmallShared *)sub_lds_base;
    const float *__restrict__ c0 = A.c0, *__restrict__ c1 = A.c1, *__restrict__ c2 = A.c2;
    uint64_t *__restrict__ out = A.out;
    const Rotation &rot = A.rot;
    const uint32_t tid = threadIdx.x;
    const int lane = lane_id(), wid = (int)(tid >> 6);
    const double *__restrict__ p = A.pts + P.src_pt;
    const WIN *__restrict__ w = A.win + P.src;

    // every point once: coordinates as f32 (:677), box (geometry.rs:42-76;
    // the cast is monotone, so the extremes of the f32 coordinates are the
    // casts of the f64 extremes), weight sums (:684) and kinds
    constexpr double kMax = 1.7976931348623157e308;
    float x[IT][D], mn[D], mx[D];
    if (c0) {
        small_points<D, TPB, IT>(P.count, x, [&](uint64_t i, float (&q)[D]) {
            q[0] = c0[P.src + i];
            q[1] = c1[P.src + i];
            if constexpr (D == 3) q[2] = c2[P.src + i];
        });
    } else if (A.rot_on) {
        small_points<D, TPB, IT>(P.count, x, [&](uint64_t i, float (&q)[D]) {
            double v[D];
#pragma unroll
            for (int a = 0; a < D; a++) v[a] = p[i * D + a];
#pragma unroll
            for (int a = 0; a < D; a++) {
                double r = rot.m[a * D] * v[0];
#pragma unroll
                for (int b = 1; b < D; b++) r = r + rot.m[a * D + b] * v[b];
                q[a] = (float)r;
            }
        });
    } else {
        small_points<D, TPB, IT>(P.count, x, [&](uint64_t i, float (&q)[D]) {
#pragma unroll
            for (int a = 0; a < D; a++) q[a] = (float)p[i * D + a];
        });
    }
#pragma unroll
    for (int a = 0; a < D; a++) { mn[a] = (float)kMax; mx[a] = -(float)kMax; }
    uint64_t su = 0;
    double sf = 0.0, sa = 0.0;
    uint32_t fl = 0;
    constexpr int L = IT < kLoad ? IT : kLoad;
#pragma unroll
    for (int k0 = 0; k0 < IT; k0 += L) {
        if ((uint32_t)(k0 * TPB) >= P.count) continue;   // uniform: no point left
        WIN v[L];
#pragma unroll
        for (int j = 0; j < L; j++) {
            const uint32_t i = (uint32_t)((k0 + j) * TPB) + tid;
            v[j] = w[i < P.count ? i : P.count - 1];
        }
#pragma unroll
        for (int j = 0; j < L; j++) {
            const int k = k0 + j;
            const bool here = (uint32_t)(k * TPB) + tid < P.count;
#pragma unroll
            for (int a = 0; a < D; a++) {
                mn[a] = x[k][a] < mn[a] ? x[k][a] : mn[a];
                mx[a] = mx[a] < x[k][a] ? x[k][a] : mx[a];
            }
            if constexpr (std::is_same<WIN, double>::value) {
                const double av = fabs(v[j]);
                const bool whole = (v[j] == trunc(v[j])) & (av <= 9007199254740992.0);
                su += (here & whole) ? (uint64_t)(int64_t)v[j] : 0ull;
                sf += here ? v[j] : 0.0;
                sa += here ? av : 0.0;
                fl |= whole ? 0u : (uint32_t)(kSmallReal | kSmallWide | kSmallNot16);
                fl |= ((v[j] >= -2147483648.0) & (v[j] <= 2147483647.0)) ? 0u : (uint32_t)kSmallWide;
                fl |= ((v[j] >= 0.0) & (v[j] <= 65535.0)) ? 0u : (uint32_t)kSmallNot16;
                fl |= v[j] >= 0.0 ? 0u : (uint32_t)kSmallNegative;   // or NaN
            } else {
                const int64_t u = (int64_t)v[j];
                su += here ? (uint64_t)u : 0ull;
                sa += here ? fabs((double)u) : 0.0;
                fl |= ((u < INT32_MIN) | (u > INT32_MAX)) ? (uint32_t)kSmallWide : 0u;
                fl |= ((u < 0) | (u > 65535)) ? (uint32_t)kSmallNot16 : 0u;
                fl |= u < 0 ? (uint32_t)kSmallNegative : 0u;
            }
        }
    }
#pragma unroll
    for (int a = 0; a < D; a++) {
        mn[a] = wave_low(mn[a]);
        mx[a] = wave_high(mx[a]);
    }
    su = wave_total(su);
    if constexpr (std::is_same<WIN, double>::value) sf = wave_total(sf);
    sa = wave_total(sa);
    if (tid == 0) {
        sh.flags = 0;
        sh.min_slot = 0xffffffffu;
    }
    __syncthreads();
    if (fl) atomicOr(&sh.flags, fl);
    if (lane == 0) {
#pragma unroll
        for (int a = 0; a < D; a++) { sh.lo[wid][a] = mn[a]; sh.hi[wid][a] = mx[a]; }
        sh.su[wid] = su;
        sh.sf[wid] = sf;
        sh.sa[wid] = sa;
    }
    __syncthreads();
    SubRoot R;
    for (int a = 0; a < kMaxDim; a++) R.lo[a] = R.hi[a] = 0.0f;
#pragma unroll
    for (int a = 0; a < D; a++) { R.lo[a] = sh.lo[0][a]; R.hi[a] = sh.hi[0][a]; }
    su = sh.su[0];
    sf = sh.sf[0];
    sa = sh.sa[0];
#pragma unroll 1
    for (int v = 1; v < TPB / 64; v++) {
#pragma unroll
        for (int a = 0; a < D; a++) {
            R.lo[a] = sh.lo[v][a] < R.lo[a] ? sh.lo[v][a] : R.lo[a];
            R.hi[a] = R.hi[a] < sh.hi[v][a] ? sh.hi[v][a] : R.hi[a];
        }
        su += sh.su[v];
        sf += sh.sf[v];
        sa += sh.sa[v];
    }
    const uint32_t all = sh.flags;
    R.axis = 0;
    R.levels = P.levels;
    R.tol = P.tol;
    R.wrap32 = A.wrap32;
    // exact sums: integers, and integer-valued doubles whose sums stay exact
    const bool real = (all & kSmallReal) || (std::is_same<WIN, double>::value &&
                                            !(sa <= 9007199254740992.0 * (1.0 - 1e-6)));
    R.packed = !real && !(all & kSmallNegative) && sa < (double)(1ull << (kSubPack - 1));
    const uint32_t kind = (all & 7u) | (real ? kSmallReal : 0u);
    if constexpr (IT <= 16) {
        if constexpr (std::is_same<WIN, double>::value) {
            if (real) {
                small_run<D, TPB, IT, kWeightAcc, WIN, double>(P, x, w, R, sf, sh, out, kind, report);
                return;
            }
        }
        small_run<D, TPB, IT, kWeightAcc, WIN, uint64_t>(P, x, w, R, su, sh, out, kind, report);
    } else {
        if constexpr (std::is_same<WIN, double>::value) {
            if (real) {
                small_run<D, TPB, IT, kWeightLoad, WIN, double>(P, x, w, R, sf, sh, out, kind, report);
                return;
            }
        }
        if (all & kSmallNot16)
            small_run<D, TPB, IT, kWeightLoad, WIN, uint64_t>(P, x, w, R, su, sh, out, kind, report);
        else
            small_run<D, TPB, IT, kWeight16, WIN, uint64_t>(P, x, w, R, su, sh, out, kind, report);
    }
}

// Problem q of a launch: `one` (a launch of one) or table[q], largest first so
// that the long ones start first.  Workgroups of 256 threads take 8 points per
// thread; those of 512 threads 4, 16 or 32, by the problem's size.
template <int D, int TPB, typename WIN>
__global__ void __launch_bounds__(TPB)
k_small(SmallProblem one, const SmallProblem *__restrict__ table, SmallArrays<WIN> A, uint32_t *report) {
    SmallProblem P = one;
    if (table) P = table[blockIdx.x];
    P.levels = __builtin_amdgcn_readfirstlane(P.levels);   // uniform: kept in scalar registers
    P.count = __builtin_amdgcn_readfirstlane(P.count);
    report += blockIdx.x;
    if constexpr (TPB == 256) {
        small_problem<D, TPB, 8, WIN>(P, A, report);
    } else {
        if (P.count <= TPB * 4) small_problem<D, TPB, 4, WIN>(P, A, report);
        else if (P.count <= TPB * 16) small_problem<D, TPB, 16, WIN>(P, A, report);
        else small_problem<D, TPB, 32, WIN>(P, A, report);
    }
}
static_assert(512 * 32 == kSmallPoints, "the last shape takes every small problem");

}  // namespace coupe_hip
