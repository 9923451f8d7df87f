// rcb_subtree.h -- a bisection tree (or the bottom of one) by one workgroup.
//
// A problem whose points fit a workgroup's registers is split level by level
// without moving a point, without a launch per pass and without a host check:
// every point keeps the index of its part within the level (its *slot*, the
// path bits from the root), a search pass bins the points of every part still
// searching in LDS, the prefix sums and the f64 tests of every candidate are
// taken in parallel, and one lane per part replays coupe's split loop
// (par_rcb_split, recursive_bisection.rs:470-571) over them.  What bounds it
// is the chain of a pass: three barriers, the points' LDS lookup and atomic
// (one each), the scan's shuffles and the replay's lookups.
#pragma once

#include "rcb_device.h"

namespace coupe_hip {

constexpr int kSubLevels = 12;            // most levels of a subtree (2048 parts at the last one)
constexpr int kSubMaxNb = 256;            // bins per part and pass (8 bisection steps)
constexpr uint32_t kSubMisc = 1024;       // bytes of LDS for the reductions
constexpr uint32_t kSubLds = 160 * 1024;  // LDS of a CU
constexpr int kSubPasses = 4096;          // f32 bisection ends within a few hundred candidates
constexpr int kSubPack = 40;              // packed bins: count in the bits above, weight below

// Flags of a slot's window (its upper half word; the lower one is the place
// of its bins).  kSubLo / kSubHi: the window's end is a candidate visited
// before, so what lies beyond it is known.  kSubMin: this pass also takes the
// smallest coordinate at or above every candidate.
enum : uint32_t { kSubOpen = 1u << 16, kSubLo = 2u << 16, kSubHi = 4u << 16, kSubMin = 8u << 16 };

// A scanned candidate's word: the points below it, and what the replay asks.
enum : uint32_t { kCandCount = (1u << 29) - 1, kCandLeft = 1u << 29, kCandStop = 1u << 30, kCandFull = 1u << 31 };

// The LDS of a subtree.  Every array but the last two lies at an offset known
// when compiling, so that the accesses need no base registers.
extern __shared__ __align__(16) char sub_lds_base[];

// 1 / (hi - lo) of a window, for sub_bin's estimate; NaN (no estimate: every
// point walks the midpoints) where an end is 2^124 or more.  Below, every sum
// of two values of the window is finite, so the midpoints are evenly spaced,
// and the reciprocal is a normal number (one below 2^-126 is flushed to 0,
// which would put every point into bin 0).
__device__ __forceinline__ float window_scale(float lo, float hi) {
    const float r = __builtin_amdgcn_rcpf(hi - lo);
    return fmaxf(fabsf(lo), fabsf(hi)) < 0x1p124f ? r : __builtin_nanf("");
}

// One part of the level.
template <typename Acc>
struct SubSlot {
    float4 win;       // lo, hi (par_rcb_split's min, max; lo is the split once closed), window_scale, flags
    Acc sum;          // weight of the part
    Acc bw;           // weight below the window; of the left side once closed
    uint32_t n;       // points of the part
    uint32_t prev;    // prev_count_left
    uint32_t bc;      // points below the window; of the left side once closed
    uint32_t nhi;     // key of the smallest coordinate at or above the window (kSubMin passes)
};

constexpr uint32_t kSubSlotBytes = 48 + 4 + 2 * 2;   // SubSlot, and its entries of heap and list
constexpr uint32_t kSubBinBytes = 8 + 2 * 4;

// Bins of a pass: one per searching part at least; more give more bisection
// steps per pass, small workgroups take fewer so that several fit a CU.
__host__ __device__ constexpr uint32_t sub_bins(int tpb) { return tpb >= 512 ? 2944 : 2048; }
// Slots of the last level of `levels`, and the bytes of LDS.
__host__ __device__ constexpr uint32_t sub_slots(uint32_t levels) { return levels ? 1u << (levels - 1) : 1u; }
__host__ __device__ constexpr uint32_t sub_lds(uint32_t levels, int tpb) {
    return kSubMisc + sub_bins(tpb) * kSubBinBytes + sub_slots(levels) * kSubSlotBytes;
}
static_assert(sub_lds(kSubLevels, 512) <= kSubLds && sub_lds(kSubLevels, 256) <= kSubLds, "LDS of a CU");
static_assert(sub_bins(256) >= sub_slots(kSubLevels) && sub_bins(512) >= sub_slots(kSubLevels), "a bin per part");

// Per bin, one per candidate: entry q holds bin q (the points below candidate
// q and not below q - 1) and the smallest key of bin q + 1; once scanned, the
// weight below candidate q, its word (kCand*) and the smallest key at or
// above it.
template <typename Acc, int TPB>
struct SubTree {
    static constexpr uint32_t bins = sub_bins(TPB);
    static_assert(sizeof(SubSlot<Acc>) == 48, "slot layout");
    float *heap;         // splits of the levels above, heap order
    uint16_t *list[2];   // searching slots, by place

    __device__ explicit SubTree(uint32_t slots) {
        char *p = sub_lds_base + kSubMisc + bins * kSubBinBytes + slots * 48u;
        heap = (float *)p;
        list[0] = (uint16_t *)(p + slots * 4u);
        list[1] = list[0] + slots;
    }
    // weight of a bin (packed: count << kSubPack | weight), count, smallest key
    static __device__ Acc &binw(uint32_t e) { return ((Acc *)(sub_lds_base + kSubMisc))[e]; }
    static __device__ uint32_t &binc(uint32_t e) { return ((uint32_t *)(sub_lds_base + kSubMisc + bins * 8))[e]; }
    static __device__ uint32_t &binm(uint32_t e) { return ((uint32_t *)(sub_lds_base + kSubMisc + bins * 12))[e]; }
    static __device__ SubSlot<Acc> &at(uint32_t s) {
        return ((SubSlot<Acc> *)(sub_lds_base + kSubMisc + bins * kSubBinBytes))[s];
    }
};

// What is known of the root of a subtree.
struct SubRoot {
    float lo[kMaxDim], hi[kMaxDim];   // inherited box
    uint32_t axis;                    // axis of its split
    uint32_t levels;                  // levels to split
    double tol;
    int wrap32;                       // i32 weights (wrapping sums)
    bool packed;                      // weights >= 0 whose sum stays below 2^kSubPack, fewer than 2^24 points
};

// B points of each lane in a search pass of nb bins per part: the lookups of
// the B points are issued together.  Called by whole wavefronts; `valid[j]`
// excludes a lane's point.  The bin is (x - lo) nb / (hi - lo) where that is
// further from a whole number than the candidates (midpoints taken in f32,
// within a few ulps of the window's magnitude of even spacing) and the
// estimate itself can be off; the other points (and all of a window that is
// only a few ulps wide, or that has no estimate: window_scale) walk the
// midpoints par_rcb_split computes (:472).
// coord(j, flags): point j's coordinate on its window's axis.
template <int B, typename Tree, typename Coord, typename Acc>
__device__ __forceinline__ void sub_bin(const Tree &T, const uint32_t (&s)[B], Coord &&coord, const Acc (&w)[B],
                                        const bool (&valid)[B], int nb, bool packed) {
    float4 v[B];
    float x[B];
#pragma unroll
    for (int j = 0; j < B; j++) v[j] = T.at(s[j]).win;
#pragma unroll
    for (int j = 0; j < B; j++) x[j] = coord(j, __builtin_bit_cast(uint32_t, v[j].w));
    bool in[B], any = false, mins = false;
#pragma unroll
    for (int j = 0; j < B; j++) {
        const uint32_t f = __builtin_bit_cast(uint32_t, v[j].w);
        // (bitwise: branches for these tests would cost more than the tests)
        const bool live = valid[j] & ((f & kSubOpen) != 0), low = (f & kSubLo) != 0, high = (f & kSubHi) != 0;
        const bool above = x[j] >= v[j].y;
        in[j] = live & (!low | (x[j] >= v[j].x)) & !(high & above);
        any |= in[j];
        mins |= live & ((f & kSubMin) != 0);
    }
    if (__ballot(mins)) {   // rare: the smallest coordinate beyond the window
#pragma unroll
        for (int j = 0; j < B; j++) {
            const uint32_t f = __builtin_bit_cast(uint32_t, v[j].w), key = f32_key(x[j]);
            if (valid[j] && (f & kSubOpen) && (f & kSubMin) && (f & kSubHi) && x[j] >= v[j].y &&
                key < __atomic_load_n(&T.at(s[j]).nhi, __ATOMIC_RELAXED))
                atomicMin(&T.at(s[j]).nhi, key);
        }
    }
    if (__ballot(any) == 0) return;
    const float fnb = (float)nb;
    int b[B];
    bool unsure[B], walk = false;
#pragma unroll
    for (int j = 0; j < B; j++) {
        const float inv = v[j].z * fnb, e = (x[j] - v[j].x) * inv;
        const float off = fmaxf(fabsf(v[j].x), fabsf(v[j].y)) * inv * 9.5367431640625e-7f + 2.44140625e-4f;
        const float c = fminf(fmaxf(e, 0.0f), fnb - 1.0f);   // NaN: 0
        b[j] = (int)c;
        const float fr = e - (float)b[j];   // outside [0, 1) past either end
        // off is NaN or large where the estimate is worthless
        const bool sure = (off < 0.25f) & ((fr > off) | (b[j] == 0)) & ((fr < 1.0f - off) | (b[j] == nb - 1));
        unsure[j] = in[j] & !sure;
        walk |= unsure[j];
    }
    if (__ballot(walk)) {
#pragma unroll
        for (int j = 0; j < B; j++) {
            if (!unsure[j]) continue;
            float lo = v[j].x, hi = v[j].y;
            b[j] = 0;
            for (int step = nb >> 1; step >= 1; step >>= 1) {
                const float t = (lo + hi) / 2.0f;
                const bool r = x[j] >= t;
                lo = r ? t : lo;
                hi = r ? hi : t;
                b[j] += r ? step : 0;
            }
        }
    }
    uint32_t e[B];
#pragma unroll
    for (int j = 0; j < B; j++) {
        e[j] = (__builtin_bit_cast(uint32_t, v[j].w) & 0xffffu) * (uint32_t)(nb - 1) + (uint32_t)b[j];
        if (!in[j] || b[j] == nb - 1) continue;   // the last bin's sums are the part's less the others
        bool done = false;
        if constexpr (std::is_same<Acc, uint64_t>::value) {
            if (packed) {
                atomicAdd((unsigned long long *)&T.binw(e[j]), (1ull << kSubPack) + (unsigned long long)w[j]);
                done = true;
            }
        }
        if (!done) {
            atomicAdd(&T.binc(e[j]), 1u);
            atomic_add_acc(&T.binw(e[j]), w[j]);
        }
    }
    if (__ballot(mins)) {
#pragma unroll
        for (int j = 0; j < B; j++) {
            if (!in[j] || b[j] == 0 || !(__builtin_bit_cast(uint32_t, v[j].w) & kSubMin)) continue;
            const uint32_t key = f32_key(x[j]);
            if (key < __atomic_load_n(&T.binm(e[j] - 1), __ATOMIC_RELAXED)) atomicMin(&T.binm(e[j] - 1), key);
        }
    }
}

// Clears the bins of a pass.
template <int TPB, typename Acc>
__device__ __forceinline__ void sub_clear(const SubTree<Acc, TPB> &T, uint32_t used) {
    for (uint32_t e = threadIdx.x; e < used; e += (uint32_t)TPB) {
        T.binw(e) = (Acc)0;
        T.binc(e) = 0;
        T.binm(e) = 0xffffffffu;
    }
}

// imb <= tol of coupe's loop, imb = |(wl - ideal) / ideal| (:545-551): the
// division only where a product does not settle it (a quotient and its
// rounding differ by less than 2^-52 of it).
__device__ __forceinline__ bool within(double wl, double ideal, double tol) {
    const double a = fabs(wl - ideal), b = fabs(ideal), p = tol * b;
    if (p > 1e-280 && p < 1e280 && b > 1e-280) {
        if (a < p * (1.0 - 1e-14)) return true;
        if (a > p * (1.0 + 1e-14)) return false;
    }
    return fabs((wl - ideal) / ideal) <= tol;
}

// Inclusive sums within groups of `width` consecutive lanes (a power of two,
// uniform): whole wavefronts by row shifts and row broadcasts (no LDS),
// narrower groups by shuffles.
template <int Ctrl, int Rows>
__device__ __forceinline__ uint64_t dpp_rows64(uint64_t v) {   // 0 in the rows not written
    const uint32_t lo = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)(uint32_t)v, Ctrl, Rows, 0xf, false);
    const uint32_t hi = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)(uint32_t)(v >> 32), Ctrl, Rows, 0xf, false);
    return (uint64_t)lo | (uint64_t)hi << 32;
}
template <typename T>
__device__ __forceinline__ T group_incl_add(T v, int width, int l) {
    if (width == 64) {
        auto step = [&](uint64_t u) {
            if constexpr (sizeof(T) == 8) v += __builtin_bit_cast(T, u);
            else v += (T)u;
        };
        auto bits = [&]() {
            if constexpr (sizeof(T) == 8) return __builtin_bit_cast(uint64_t, v);
            else return (uint64_t)v;
        };
        step(dpp_row64<0x111>(bits()));          // row_shr:1
        step(dpp_row64<0x112>(bits()));          // row_shr:2
        step(dpp_row64<0x114>(bits()));          // row_shr:4
        step(dpp_row64<0x118>(bits()));          // row_shr:8
        step(dpp_rows64<0x142, 0xa>(bits()));    // row_bcast:15 into rows 1 and 3
        step(dpp_rows64<0x143, 0xc>(bits()));    // row_bcast:31 into rows 2 and 3
        return v;
    }
    for (int o = 1; o < width; o <<= 1) {
        const T x = __shfl_up(v, o, width);
        if (l >= o) v += x;
    }
    return v;
}

// Prefix sums over each part's candidates, and what the replay asks of each:
// a wavefront per part (up to four candidates per lane), or several parts per
// wavefront; the f64 work of all candidates in parallel.
template <int TPB, typename Acc>
__device__ __forceinline__ void sub_scan(const SubTree<Acc, TPB> &T, const SubRoot &R, const uint16_t *list, uint32_t nact,
                                         int nb) {
    using Ops = AccOps<Acc>;
    const int width = nb < 64 ? nb : 64, per = nb / width;
    const uint32_t groups = (uint32_t)TPB / (uint32_t)width;
    const int l = (int)(threadIdx.x & (uint32_t)(width - 1));
    for (uint32_t g = threadIdx.x / (uint32_t)width; g < nact; g += groups) {
        const uint32_t s = list[g], e0 = g * (uint32_t)(nb - 1);
        const uint32_t n = T.at(s).n, bc = T.at(s).bc;
        const Acc S = T.at(s).sum, bw = T.at(s).bw;
        const double ideal = Ops::f64(S, R.wrap32) / 2.0;
        uint32_t c[4], lc = 0;
        Acc w[4], lw = (Acc)0;
#pragma unroll
        for (int k = 0; k < 4; k++) {
            c[k] = 0;
            w[k] = (Acc)0;
            const int q = l * per + k;
            if (k < per && q < nb - 1) {
                w[k] = T.binw(e0 + q);
                if constexpr (std::is_same<Acc, uint64_t>::value) {
                    if (R.packed) {
                        c[k] = (uint32_t)(w[k] >> kSubPack);
                        w[k] &= (1ull << kSubPack) - 1;
                    } else {
                        c[k] = T.binc(e0 + q);
                    }
                } else {
                    c[k] = T.binc(e0 + q);
                }
            }
            lc += c[k];
            lw += w[k];
        }
        uint32_t rc = bc + (group_incl_add(lc, width, l) - lc);
        Acc rw = bw + (group_incl_add(lw, width, l) - lw);
#pragma unroll
        for (int k = 0; k < 4; k++) {
            const int q = l * per + k;
            if (k < per && q < nb - 1) {
                rc += c[k];
                rw += w[k];
                uint32_t word = rc | (rc == n ? (uint32_t)kCandFull : 0u);
                if (within(Ops::f64(rw, R.wrap32), ideal, R.tol)) word |= kCandStop;
                if (!Ops::lt(rw, Ops::sub(S, rw), R.wrap32)) word |= kCandLeft;
                T.binc(e0 + q) = word;
                T.binw(e0 + q) = rw;
            }
        }
        if (__builtin_bit_cast(uint32_t, T.at(s).win.w) & kSubMin) {   // suffix minima (the group alike)
            uint32_t m[4], lm = 0xffffffffu;
#pragma unroll
            for (int k = 3; k >= 0; k--) {
                const int q = l * per + k;
                m[k] = k < per && q < nb - 1 ? T.binm(e0 + q) : 0xffffffffu;
                lm = min(lm, m[k]);
            }
            uint32_t im = lm;
            for (int o = 1; o < width; o <<= 1) {
                const uint32_t m2 = __shfl_down(im, o, width);
                if (l + o < width) im = min(im, m2);
            }
            uint32_t rm = __shfl_down(im, 1, width);
            if (l == width - 1) rm = 0xffffffffu;
            rm = min(rm, T.at(s).nhi);
#pragma unroll
            for (int k = 3; k >= 0; k--) {
                const int q = l * per + k;
                if (k < per && q < nb - 1) {
                    rm = min(rm, m[k]);
                    T.binm(e0 + q) = rm;
                }
            }
        }
    }
}

// The decisions of a pass: one lane per part replays the split loop over the
// scanned candidates; the parts still searching go to `next`.
//
// The loop's test hi <= t + d needs d, the distance from t to the smallest
// coordinate m >= t.  A point below a candidate u between t and hi bounds it:
// m < u, so (rounding is monotone) t + d <= t + (u - t), and hi above that
// settles the test without m.  Only a part whose points at or above t all lie
// beyond the last such candidate asks for a pass that takes minima.
template <int TPB, typename Acc>
__device__ __forceinline__ void sub_decide(const SubTree<Acc, TPB> &T, const SubRoot &R, const uint16_t *list,
                                           uint16_t *next, uint32_t nact, int nb, uint32_t *n_next) {
    for (uint32_t g = threadIdx.x; g < nact; g += (uint32_t)TPB) {
        const uint32_t s = list[g], e0 = g * (uint32_t)(nb - 1);
        const float4 v = T.at(s).win;
        float lo = v.x, hi = v.y, split = 0.0f;
        uint32_t prev = T.at(s).prev, f = __builtin_bit_cast(uint32_t, v.w) & ~0xffffu;
        const bool have_min = f & kSubMin;
        f &= ~kSubMin;
        int step = nb >> 1, q = step - 1, below = -1, stop = -1;   // below: the candidate at lo
        bool open = true;
        uint32_t word = T.binc(e0 + q);
        for (;;) {   // selects instead of branches: the parts of a wavefront differ
            const float t = (lo + hi) / 2.0f;
            const uint32_t cnt = word & kCandCount;
            // the candidates either way, looked up ahead of the decision
            const int half = step >> 1;
            const uint32_t wleft = T.binc(e0 + q - half), wright = T.binc(e0 + q + half);
            const bool full = (word & kCandFull) != 0;        // no point at or right of t (:528)
            const bool same = cnt == prev;
            bool end = same | (!full & ((word & kCandStop) != 0));   // :528-539, :552-563
            float u = (t + hi) / 2.0f;
            const bool known = end | full | ((half >= 1) & ((wright & kCandCount) > cnt) & !(hi <= t + (u - t)));
            if (!known) {
                bool bound = false;
                if (have_min) {
                    end = hi <= t + (key_f32(T.binm(e0 + q)) - t);
                    bound = true;
                }
                int qu = q + half;
                for (int r = half >> 1; r >= 1 && !bound; r >>= 1) {
                    u = (u + hi) / 2.0f;
                    qu += r;
                    bound = (T.binc(e0 + qu) & kCandCount) > cnt && !(hi <= t + (u - t));
                }
                if (!bound) {   // this candidate again, with minima when the pass could not get closer
                    if (step > 1) f |= kSubMin;
                    break;
                }
            }
            if (end) {
                split = full ? hi : t;
                stop = full ? -1 : q;
                open = false;
                break;
            }
            const bool left = full | ((word & kCandLeft) != 0);
            prev = cnt;                                       // :540-544, :564
            hi = left ? t : hi;
            lo = left ? lo : t;
            below = left ? below : q;
            f |= left ? (uint32_t)kSubHi : (uint32_t)kSubLo;
            step = half;
            if (step == 0) break;
            q = left ? q - step : q + step;
            word = left ? wleft : wright;
        }
        if (open) {
            if (below >= 0) {
                T.at(s).bc = T.binc(e0 + below) & kCandCount;
                T.at(s).bw = T.binw(e0 + below);
            }
            T.at(s).prev = prev;
            const uint32_t k = atomicAdd(n_next, 1u);
            next[k] = (uint16_t)s;
            T.at(s).win = make_float4(lo, hi, window_scale(lo, hi), __builtin_bit_cast(float, f | k));
        } else {
            T.at(s).bc = stop >= 0 ? T.binc(e0 + stop) & kCandCount : T.at(s).n;
            T.at(s).bw = stop >= 0 ? T.binw(e0 + stop) : T.at(s).sum;
            T.at(s).win = make_float4(split, split, 0.0f, 0.0f);
        }
    }
}

// The windows of the level's parts start at their inherited box on its axis.
template <int TPB, typename Acc>
__device__ __forceinline__ void sub_start(const SubTree<Acc, TPB> &T, uint32_t s, float lo, float hi, uint32_t n, Acc sum,
                                          uint16_t *list, uint32_t *n_list) {
    T.at(s).n = n;
    T.at(s).sum = sum;
    T.at(s).prev = 0xffffffffu;   // no count of a subtree reaches it
    T.at(s).bc = 0;
    T.at(s).bw = (Acc)0;
    T.at(s).nhi = 0xffffffffu;
    uint32_t f = 0;
    if (n) {
        const uint32_t k = atomicAdd(n_list, 1u);
        list[k] = (uint16_t)s;
        f = kSubOpen | k;
    }
    T.at(s).win = make_float4(lo, hi, window_scale(lo, hi), __builtin_bit_cast(float, f));
}

// Splits a subtree of n points of weight `sum` level by level.
// `pass(nb)` bins every point on the level's axis (sub_bin), `descend()`
// moves every point's slot to its child (left of win[slot].x or not), both
// told the axis; `split_out(level, slot, count, left count, split)` sees
// every part.  ctr: three counters in LDS.  false when a search did not end
// (the caller reports it).
template <int D, int TPB, typename Acc, typename Pass, typename Descend, typename Split>
__device__ bool sub_levels(SubTree<Acc, TPB> &T, const SubRoot &R, uint32_t n, Acc sum, uint32_t *ctr, Pass &&pass,
                           Descend &&descend, Split &&split_out) {
    const uint32_t tid = threadIdx.x;
    uint32_t it = 0;
    if (tid < 3) ctr[tid] = 0;
    sub_clear<TPB, Acc>(T, T.bins);
    __syncthreads();
    if (tid == 0 && R.levels) {
        const int a = (int)R.axis;
        sub_start<TPB, Acc>(T, 0, sel3(a, R.lo[0], R.lo[1], R.lo[2]), sel3(a, R.hi[0], R.hi[1], R.hi[2]), n, sum, T.list[0],
                       &ctr[0]);
    }
    __syncthreads();
    uint32_t dirty = 0;   // bins the last pass left
    for (uint32_t level = 0; level < R.levels; level++) {
        const uint32_t slots = 1u << level;
        const int a = (int)((R.axis + level) % D);
        for (int p = 0;; p++) {
            const uint32_t nact = __builtin_amdgcn_readfirstlane(ctr[it % 3]);
            if (nact == 0) break;
            if (p >= kSubPasses) return false;
            int lg = 8;
            while (lg > 1 && nact * ((1u << lg) - 1) > T.bins) lg--;
            const int nb = 1 << lg;
            const uint16_t *list = T.list[it & 1];
            if (tid == 0) ctr[(it + 1) % 3] = 0;
            // few bins cannot bound the distance to the next coordinate
            if (nb <= 4)
                for (uint32_t g = tid; g < nact; g += TPB) {
                    float *w = &T.at(list[g]).win.w;
                    *w = __builtin_bit_cast(float, __builtin_bit_cast(uint32_t, *w) | kSubMin);
                }
            if (dirty || nb <= 4) {
                sub_clear<TPB, Acc>(T, dirty);
                __syncthreads();
            }
            pass(nb, a);
            __syncthreads();
            sub_scan<TPB, Acc>(T, R, list, nact, nb);
            __syncthreads();
            sub_decide<TPB, Acc>(T, R, list, T.list[(it + 1) & 1], nact, nb, &ctr[(it + 1) % 3]);
            dirty = nact * (uint32_t)(nb - 1);
            it++;
            __syncthreads();
        }
        // children: the parts' figures in registers across the barrier
        constexpr int kPer = (1 << (kSubLevels - 1)) / TPB;
        Acc cs[kPer], cw[kPer];
        uint32_t cn[kPer], cl[kPer];
#pragma unroll
        for (int k = 0; k < kPer; k++) {
            const uint32_t s = tid + (uint32_t)k * TPB;
            if (s < slots) {
                cs[k] = T.at(s).sum;
                cw[k] = T.at(s).bw;
                cn[k] = T.at(s).n;
                cl[k] = T.at(s).bc;
                const float split = T.at(s).win.x;
                if (level + 1 < R.levels) T.heap[slots - 1 + s] = split;
                split_out(level, s, cn[k], cl[k], split);
            }
        }
        descend(a);
        if (level + 1 == R.levels) break;
        __syncthreads();
        const int na = (int)((R.axis + level + 1) % D);
#pragma unroll
        for (int k = 0; k < kPer; k++) {
            const uint32_t s = tid + (uint32_t)k * TPB;
            if (s < slots) {
                // the box on the next axis, clipped by the ancestors that
                // split it (the same for both children: D > 1)
                float lo = sel3(na, R.lo[0], R.lo[1], R.lo[2]), hi = sel3(na, R.hi[0], R.hi[1], R.hi[2]);
                for (uint32_t m = (level + 1) % D; m < level; m += D) {
                    const float sp = T.heap[(1u << m) - 1 + (s >> (level - m))];
                    const bool right = (s >> (level - m - 1)) & 1u;
                    lo = right ? sp : lo;
                    hi = right ? hi : sp;
                }
                sub_start<TPB, Acc>(T, 2 * s, lo, hi, cl[k], cw[k], T.list[it & 1], &ctr[it % 3]);
                sub_start<TPB, Acc>(T, 2 * s + 1, lo, hi, cn[k] - cl[k], AccOps<Acc>::sub(cs[k], cw[k]), T.list[it & 1],
                               &ctr[it % 3]);
            }
        }
        sub_clear<TPB, Acc>(T, dirty);
        dirty = 0;
        __syncthreads();
    }
    return true;
}

}  // namespace coupe_hip
