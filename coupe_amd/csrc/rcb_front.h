// rcb_front.h -- the levels of one instance without moving its points, where
// the searches do not end at the boxes' midpoints.
//
// Every point keeps the number of its node in the *frontier*, the parts being
// searched.  A round is two launches: k_front_hist sends each point on to the
// child of a part split in the round before and bins it in its part's window
// (sub_bin, rcb_subtree.h); k_front_decide adds the workgroups' bins, replays
// coupe's loop for every part (sub_scan, sub_decide) and writes the next
// frontier: parts still searching, and the children of the others.  A child
// of few points leaves the frontier for the open nodes that one workgroup
// each searches to the end (k_mid_search).
//
// A round reads the coordinates of the axes it needs (4 or 8 bytes per
// point), the weight and the node number, and writes the number where it
// changed: 8 to 16 bytes per point, against 28 per two levels for the general
// path's moves and 6 to 12 per search pass; it has no tables of tiles, no
// scans and no second run when a search takes long.  Its bins are what limits
// it: the fewer per part, the fewer bisection steps per round.
//
// Measured: 2^24 Gaussian points, 1024 parts: 19 rounds of 57 us (sweep) and 19
// (decision: 256 workgroups' bins read by the few that decide), the call 2.04
// -> 1.83 ms; 2^21 points by Rib, 512 parts: 801 -> 613 us.
#pragma once

#include "rcb_mid.h"

namespace coupe_hip {

constexpr uint32_t kFrontNodes = 1024;        // parts of a frontier: fewer, each holds more than n / 1024 points
constexpr uint32_t kFrontBins = 5376;         // bins of a round: with the parts what the LDS of a CU holds
constexpr int kFrontThreads = 1024;
constexpr uint32_t kFrontCopies = 256;        // workgroups of a round, each with bins of its own
constexpr int kFrontRounds = 256;             // rounds a call may take
constexpr uint64_t kFrontPoints = 1ull << 25; // largest call: see below
// kFrontPoints: Gaussian mixtures 3D, 10 levels, points changing, mean us on the
// frontier and the general path: 2^20 525 and 805, 2^22 905 and 1510, 2^24 1790
// and 2800, 2^25 3320 and 3530, 2^26 6180 and 6390.  Beyond 2^25 what is left
// does not pay for the 28 bytes a point the frontier holds besides.
//
// Calls of more than kFrontEven points that took more than kFrontLong / 2 rounds
// a level go to the general path next time: a round costs a pass over all
// points, the general path's later passes only the parts that still search.  us
// on the frontier and the general path, 3D, 10 levels.  2^23 points: lognormal,
// 28 rounds, 2170 and 1710; fifth powers of normals, 46, 2460 and 2220; Gaussian
// mixture, 19, 1180 and 1400.  2^24: 2890 and 2610, 3780 and 3430, 1820 and 2070.
// From 1 to 12 levels, tolerances 0.001 and 0.02, 5e6 and 2^24 points alike: up
// to 2.3 rounds a level the frontier is faster by 0 to 40%, from 2.6 on slower by
// 0 to 45%.  2^21 points 2D: 24 rounds of 9 levels, 890 and 975, still faster.
// Where the points change, the general path's searches outrun what it queues
// (Cauchy points, 28 rounds, 1840 and 4500): after kFrontReruns such calls the
// frontier keeps the shape.
constexpr uint64_t kFrontEven = 1ull << 22;
constexpr uint32_t kFrontLong = 5;
constexpr uint32_t kFrontReruns = 2;
constexpr uint32_t kFrontDecides = 64;        // workgroups of k_front_decide
constexpr int kDecideThreads = 512;           // (1024 leave too few registers: loads in flight, no spills)

// One part of the frontier.
struct FrontNode {
    uint64_t sum, bw;                 // weight; weight below the window
    uint32_t n, bc, prev, flags;      // points; points below the window; prev_count_left; kSub*
    float lo, hi;                     // search window
    float blo[kMaxDim], bhi[kMaxDim];
    uint32_t heap, levels, axis;      // heap index, levels left, axis of the split
    uint32_t pad[3];
};

// Where the points of a part of the last frontier go.
struct FrontRoute {
    float split;
    uint32_t axis;                    // 3: the part is still searching, and now number `left`
    uint16_t left, right;             // frontier numbers, kFrontSmall + open node, or kFrontNone
};

// What round r works on (zero before the call).
struct FrontRound {
    uint32_t nodes;                   // parts of the frontier
    uint32_t route_axes, bin_axes;    // axes read to send points on, and to bin them
    uint32_t minima;                  // a part asks for smallest coordinates
};

constexpr uint32_t kFrontAxis = 20;           // a window's flags: its axis from this bit on

// Bins per part: as many bisection steps as fit the bins.
__host__ __device__ inline int front_log_bins(uint32_t nodes) {
    int lg = 8;
    while (lg > 1 && nodes * ((1u << lg) - 1) > kFrontBins) lg--;
    return lg;
}

// LDS of k_front_hist, in SubTree's terms (sub_bin).
template <typename Acc>
struct FrontTree {
    static __device__ Acc &binw(uint32_t e) { return ((Acc *)sub_lds_base)[e]; }
    static __device__ uint32_t &binc(uint32_t e) { return ((uint32_t *)(sub_lds_base + kFrontBins * 8))[e]; }
    static __device__ uint32_t &binm(uint32_t e) { return ((uint32_t *)(sub_lds_base + kFrontBins * 12))[e]; }
    static __device__ SubSlot<Acc> &at(uint32_t s) { return ((SubSlot<Acc> *)(sub_lds_base + kFrontBins * 16))[s]; }
    static __device__ FrontRoute &route(uint32_t s) {
        return ((FrontRoute *)(sub_lds_base + kFrontBins * 16 + kFrontNodes * 48))[s];
    }
};
constexpr uint32_t kFrontLds = kFrontBins * 16 + kFrontNodes * (48 + sizeof(FrontRoute));
static_assert(kFrontLds <= kSubLds, "LDS of a CU");
static_assert(kFrontBins >= kFrontNodes, "a bin per part");

// The root as the only part; the call's open nodes and rounds start empty.
template <int D, typename Acc>
__global__ void k_front_init(Instance *__restrict__ insts, const InstReduce *__restrict__ red, FrontNode *nodes,
                             FrontRound *rounds, MidCounters *ctr) {
    const uint32_t tid = threadIdx.x;
    for (uint32_t k = tid; k < (uint32_t)kFrontRounds * sizeof(FrontRound) / 4; k += blockDim.x)
        ((uint32_t *)rounds)[k] = 0;
    for (uint32_t k = tid; k < sizeof(MidCounters) / 4; k += blockDim.x) ((uint32_t *)ctr)[k] = 0;
    __syncthreads();
    if (tid) return;
    Instance &I = insts[0];
    FrontNode N;
    uint64_t su = 0;
    double sf = 0.0;
    for (int c = 0; c < kCopies; c++) {
        su += red[c].sum_u64;
        sf += red[c].sum_f64;
    }
    N.sum = std::is_same<Acc, double>::value ? __builtin_bit_cast(uint64_t, sf) : su;
    N.bw = 0;
    N.n = (uint32_t)I.count;
    N.bc = 0;
    N.prev = 0xffffffffu;
    N.flags = kSubOpen;
    for (int a = 0; a < kMaxDim; a++) {
        N.blo[a] = N.bhi[a] = 0.0f;
        if (a < D) mid_box<D>(red, 1, 0, a, N.blo[a], N.bhi[a]);
    }
    N.lo = N.blo[0];
    N.hi = N.bhi[0];
    N.heap = 0;
    N.levels = I.levels;
    N.axis = 0;
    nodes[0] = N;
    rounds[0] = FrontRound{1u, 0u, 1u, 0u};
    I.min_id = ~0ull;
}

// Round r, first launch.  Workgroups take contiguous shares of the points.
// bins: per workgroup, kFrontBins weights (packed with the counts for 16-bit
// weights), counts, smallest keys, and per part the smallest key beyond.
template <int D, typename WL, typename Acc>
__global__ void __launch_bounds__(kFrontThreads)
k_front_hist(int r, const FrontRound *__restrict__ rounds, const FrontNode *__restrict__ nodes,
             const FrontRoute *__restrict__ routes, uint64_t n, const float *__restrict__ c0,
             const float *__restrict__ c1, const float *__restrict__ c2, const WL *__restrict__ w,
             uint16_t *__restrict__ pid, Acc *__restrict__ gw, uint32_t *__restrict__ gc, uint32_t *__restrict__ gm,
             uint32_t *__restrict__ gh) {
    const FrontRound H = rounds[r];
    const uint32_t before = r ? rounds[r - 1].nodes : 0u;
    if (H.nodes == 0 && before == 0) return;
    constexpr int TPB = kFrontThreads, B = 8;
    constexpr bool packed = packable<WL, Acc>();   // a workgroup's share stays below 2^24 points
    const FrontTree<Acc> T;
    const uint32_t tid = threadIdx.x;
    const int lg = front_log_bins(H.nodes), nb = 1 << lg;
    const bool minima = H.minima || nb <= 4;       // few bins cannot bound the distance to the next coordinate
    const uint32_t used = H.nodes * (uint32_t)(nb - 1);
    for (uint32_t s = tid; s < H.nodes; s += TPB) {
        const FrontNode &N = nodes[s];
        const uint32_t f = N.flags | (nb <= 4 ? (uint32_t)kSubMin : 0u) | s | N.axis << kFrontAxis;
        T.at(s).win = make_float4(N.lo, N.hi, window_scale(N.lo, N.hi), __builtin_bit_cast(float, f));
        T.at(s).nhi = 0xffffffffu;
    }
    for (uint32_t s = tid; s < before; s += TPB) T.route(s) = routes[s];
    for (uint32_t e = tid; e < used; e += TPB) {
        T.binw(e) = (Acc)0;
        T.binc(e) = 0;
        T.binm(e) = 0xffffffffu;
    }
    __syncthreads();
    const uint32_t share = (uint32_t)((n + gridDim.x - 1) / gridDim.x);
    const uint32_t b0 = blockIdx.x * share, b1 = (uint32_t)min((uint64_t)b0 + share, n);
    const uint32_t axes = H.route_axes | H.bin_axes;
    for (uint32_t i0 = b0; i0 < b1; i0 += TPB * B) {
        uint32_t s[B];
        float x0[B], x1[B], x2[B];   // (one array indexed by the lane's axis would live in scratch)
        WL wk[B];
        bool valid[B];
#pragma unroll
        for (int j = 0; j < B; j++) {   // every load of the group first (clamped, unconditional)
            const uint32_t i = i0 + (uint32_t)(j * TPB) + tid, p = i < b1 ? i : b1 - 1;
            valid[j] = i < b1;
            s[j] = r ? (uint32_t)pid[p] : 0u;
            if (H.nodes) wk[j] = w[p];
            x0[j] = x1[j] = x2[j] = 0.0f;
            if (axes & 1u) x0[j] = c0[p];   // uniform
            if (axes & 2u) x1[j] = c1[p];
            if (D == 3 && (axes & 4u)) x2[j] = c2[p];
        }
        if (r) {
            FrontRoute to[B];
#pragma unroll
            for (int j = 0; j < B; j++) to[j] = T.route(s[j] < kFrontSmall ? s[j] : 0u);
#pragma unroll
            for (int j = 0; j < B; j++) {
                const float xr = sel3((int)to[j].axis, x0[j], x1[j], x2[j]);
                const bool right = (to[j].axis < 3) & (xr >= to[j].split);
                uint32_t t = right ? to[j].right : to[j].left;
                t = s[j] < kFrontSmall ? t : s[j];
                if ((t != s[j]) & valid[j]) pid[i0 + (uint32_t)(j * TPB) + tid] = (uint16_t)t;
                s[j] = t;
            }
        } else {
#pragma unroll
            for (int j = 0; j < B; j++)
                if (valid[j]) pid[i0 + (uint32_t)(j * TPB) + tid] = 0;
        }
        if (H.nodes == 0) continue;
#pragma unroll
        for (int h = 0; h < B; h += kAhead) {   // (register arrays: kAhead points' lookups at a time)
            uint32_t sh[kAhead];
            Acc wh[kAhead];
            bool vh[kAhead];
#pragma unroll
            for (int j = 0; j < kAhead; j++) {
                vh[j] = valid[h + j] & (s[h + j] < kFrontSmall);
                sh[j] = vh[j] ? s[h + j] : 0u;
                wh[j] = AccOps<Acc>::of(wk[h + j]);
            }
            sub_bin<kAhead>(T, sh, [&](int j, uint32_t f) {
                return sel3((int)(f >> kFrontAxis & 3u), x0[h + j], x1[h + j], x2[h + j]);
            }, wh, vh, nb, packed);
        }
    }
    __syncthreads();
    const uint64_t g = (uint64_t)blockIdx.x * kFrontBins;
    for (uint32_t e = tid; e < used; e += TPB) {
        gw[g + e] = T.binw(e);
        if constexpr (!packed) gc[g + e] = T.binc(e);
        if (minima) gm[g + e] = T.binm(e);
    }
    if (minima)
        for (uint32_t s = tid; s < H.nodes; s += TPB) gh[(uint64_t)blockIdx.x * kFrontNodes + s] = T.at(s).nhi;
}

// Round r, second launch: a workgroup per 256 bins.  `copies`: workgroups of
// the first.  small: a child of at most so many points leaves the frontier.
template <int D, typename WL, typename Acc>
__global__ void __launch_bounds__(kDecideThreads)
k_front_decide(int r, FrontRound *__restrict__ rounds, const FrontNode *__restrict__ nodes,
               FrontNode *__restrict__ next, FrontRoute *__restrict__ routes, uint32_t copies,
               const Acc *__restrict__ gw, const uint32_t *__restrict__ gc, const uint32_t *__restrict__ gm,
               const uint32_t *__restrict__ gh, Instance *__restrict__ insts, int wrap32, float *__restrict__ heap,
               uint32_t small, MidOpen *__restrict__ open, uint32_t *__restrict__ cursor,
               uint32_t *__restrict__ lists, uint64_t list_stride, MidCounters *ctr) {
    const FrontRound H = rounds[r];
    if (H.nodes == 0) return;
    constexpr int TPB = kDecideThreads, G = TPB / 256;   // G threads share an entry's copies
    constexpr bool packed = packable<WL, Acc>();
    __shared__ Acc pw[G][256];
    __shared__ uint32_t pc[G][256], pm[G][256], s_next;
    const uint32_t tid = threadIdx.x, part = tid >> 8, lane = tid & 255u;
    const int lg = front_log_bins(H.nodes), nb = 1 << lg;
    const bool minima = H.minima || nb <= 4;
    const uint32_t per = 256u >> lg;                    // parts of a workgroup
    Instance &I = insts[0];
    SubRoot R;
    R.tol = I.tol;
    R.wrap32 = wrap32;
    R.packed = false;
    for (uint32_t first = blockIdx.x * per; first < H.nodes; first += gridDim.x * per) {
        const uint32_t mine = min(per, H.nodes - first), entries = mine * (uint32_t)(nb - 1);
        SubTree<Acc, TPB> T(per);
        FrontNode mine_node;   // (loaded beside the bins)
        if (tid < mine) mine_node = nodes[first + tid];
        __syncthreads();   // the last parts' LDS is free
        {
            Acc sw = (Acc)0;
            uint32_t sc = 0, sm = 0xffffffffu;
            if (lane < entries) {
                const uint64_t e = (uint64_t)first * (uint32_t)(nb - 1) + lane;
                // the copies come from other XCDs' memory: as many loads in
                // flight as registers allow
                constexpr uint32_t F = packed ? 64 : 32;
                for (uint32_t c0 = part; c0 < copies; c0 += G * F) {
                    Acc v[F];
                    uint32_t k[F], m[F];
#pragma unroll
                    for (uint32_t u = 0; u < F; u++) {
                        const uint32_t c = c0 + u * G;
                        const uint64_t at = (uint64_t)(c < copies ? c : part) * kFrontBins + e;
                        v[u] = gw[at];
                        if constexpr (!packed) k[u] = gc[at];
                        m[u] = 0xffffffffu;
                        if (minima) m[u] = gm[at];
                    }
#pragma unroll
                    for (uint32_t u = 0; u < F; u++) {
                        if (c0 + u * G >= copies) continue;
                        if constexpr (packed) {
                            sc += (uint32_t)((uint64_t)v[u] >> kSubPack);
                            sw += (Acc)((uint64_t)v[u] & ((1ull << kSubPack) - 1));
                        } else {
                            sw += v[u];
                            sc += k[u];
                        }
                        sm = min(sm, m[u]);
                    }
                }
            }
            pw[part][lane] = sw;
            pc[part][lane] = sc;
            pm[part][lane] = sm;
        }
        if (tid == 0) s_next = 0;
        __syncthreads();
        if (tid < entries) {
            Acc sw = pw[0][tid];
            uint32_t sc = pc[0][tid], sm = pm[0][tid];
#pragma unroll
            for (int v = 1; v < G; v++) {
                sw += pw[v][tid];
                sc += pc[v][tid];
                sm = min(sm, pm[v][tid]);
            }
            T.binw(tid) = sw;
            T.binc(tid) = sc;
            T.binm(tid) = sm;
        }
        if (tid < mine) {
            const FrontNode &N = mine_node;
            SubSlot<Acc> &S = T.at(tid);
            uint32_t nhi = 0xffffffffu;
            if (minima)
                for (uint32_t c = 0; c < copies; c++) nhi = min(nhi, gh[(uint64_t)c * kFrontNodes + first + tid]);
            const uint32_t f = N.flags | (nb <= 4 ? (uint32_t)kSubMin : 0u) | tid;
            S.win = make_float4(N.lo, N.hi, 0.0f, __builtin_bit_cast(float, f));
            S.sum = AccOps<Acc>::from_bits(N.sum);
            S.bw = AccOps<Acc>::from_bits(N.bw);
            S.n = N.n;
            S.prev = N.prev;
            S.bc = N.bc;
            S.nhi = nhi;
            T.list[0][tid] = (uint16_t)tid;
        }
        __syncthreads();
        sub_scan<TPB, Acc>(T, R, T.list[0], mine, nb);
        __syncthreads();
        sub_decide<TPB, Acc>(T, R, T.list[0], T.list[1], mine, nb, &s_next);
        __syncthreads();
        if (tid < mine) {
            const FrontNode &N = mine_node;
            const SubSlot<Acc> &S = T.at(tid);
            const uint32_t f = __builtin_bit_cast(uint32_t, S.win.w);
            FrontRoute to;
            if (f & kSubOpen) {   // still searching, in its new window
                FrontNode M = N;
                M.lo = S.win.x;
                M.hi = S.win.y;
                M.prev = S.prev;
                M.bc = S.bc;
                M.bw = AccOps<Acc>::to_bits(S.bw);
                M.flags = f & ~0xffffu;
                const uint32_t k = atomicAdd(&rounds[r + 1].nodes, 1u);
                next[k] = M;
                atomicOr(&rounds[r + 1].bin_axes, 1u << N.axis);
                if (f & kSubMin) atomicOr(&rounds[r + 1].minima, 1u);
                to.split = 0.0f;
                to.axis = 3;
                to.left = to.right = (uint16_t)k;
            } else {
                const float split = S.win.x;
                const uint32_t cl = S.bc;
                const Acc sum = AccOps<Acc>::from_bits(N.sum), wl = S.bw;
                heap[N.heap] = cl == N.n ? __builtin_nanf("") : split;   // every point left: as the descent walks it
                to.split = cl == N.n ? __builtin_nanf("") : split;
                to.axis = N.axis;
                // places for both children, every atomic issued before any is
                // waited for
                uint32_t cnt[2] = {cl, N.n - cl}, n_front = 0, n_open = 0, n_points = 0;
                bool leaf[2], in_front[2];
#pragma unroll
                for (int side = 0; side < 2; side++) {
                    leaf[side] = cnt[side] > 0 && N.levels == 1;   // (:589-601)
                    in_front[side] = N.levels > 1 && cnt[side] > small;
                    const bool opens = N.levels > 1 && cnt[side] > 0 && cnt[side] <= small;
                    n_front += in_front[side] ? 1u : 0u;
                    n_open += opens ? 1u : 0u;
                    n_points += opens ? cnt[side] : 0u;
                }
                uint32_t k = 0, e = 0, at = 0;
                if (n_front) k = atomicAdd(&rounds[r + 1].nodes, n_front);
                if (n_open) {
                    e = atomicAdd(&ctr->open, n_open);
                    at = atomicAdd(&ctr->points, n_points);
                }
                if (n_front) atomicOr(&rounds[r + 1].bin_axes, 1u << ((N.axis + 1) % D));
                uint16_t code[2];
#pragma unroll
                for (int side = 0; side < 2; side++) {
                    const uint32_t h = 2 * N.heap + 1 + (uint32_t)side;
                    code[side] = (uint16_t)kFrontNone;
                    if (leaf[side]) atomicMin((unsigned long long *)&I.min_id, (unsigned long long)h);
                    if (leaf[side] || cnt[side] == 0) continue;
                    FrontNode C;
                    C.sum = AccOps<Acc>::to_bits(side ? AccOps<Acc>::sub(sum, wl) : wl);   // (:603-641)
                    C.bw = 0;
                    C.n = cnt[side];
                    C.bc = 0;
                    C.prev = 0xffffffffu;
                    C.flags = kSubOpen;
                    for (int a = 0; a < kMaxDim; a++) {
                        C.blo[a] = a == (int)N.axis && side ? split : N.blo[a];
                        C.bhi[a] = a == (int)N.axis && !side ? split : N.bhi[a];
                    }
                    C.heap = h;
                    C.levels = N.levels - 1;
                    C.axis = (N.axis + 1) % D;
                    C.lo = sel3((int)C.axis, C.blo[0], C.blo[1], C.blo[2]);
                    C.hi = sel3((int)C.axis, C.bhi[0], C.bhi[1], C.bhi[2]);
                    if (in_front[side]) {
                        next[k] = C;
                        code[side] = (uint16_t)k++;
                    } else {
                        MidOpen O;
                        O.sum = C.sum;
                        O.count = C.n;
                        O.begin = at;
                        O.node = h;
                        O.inst = 0;
                        O.axis = C.axis;
                        O.levels = C.levels;
                        for (int a = 0; a < kMaxDim; a++) { O.lo[a] = C.blo[a]; O.hi[a] = C.bhi[a]; }
                        open[e] = O;
                        cursor[e] = at;
                        at += C.n;
                        const uint32_t c = C.n <= kMidClass[0] ? 0u : (C.n <= kMidClass[1] ? 1u : 2u);
                        lists[c * list_stride + atomicAdd(&ctr->of_class[c], 1u)] = e;
                        code[side] = (uint16_t)(kFrontSmall + e++);
                    }
                }
                to.left = code[0];
                to.right = code[1];
                atomicOr(&rounds[r + 1].route_axes, 1u << N.axis);
            }
            routes[first + tid] = to;
        }
    }
}

}  // namespace coupe_hip
