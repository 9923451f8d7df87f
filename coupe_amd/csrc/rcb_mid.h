// rcb_mid.h -- all levels of a call from one sweep over its points, where the
// parts split at the middle of their box.
//
// coupe's search starts at the midpoint of a part's box and ends there when
// the halves balance within the tolerance: the usual case on meshes, all the
// way down on regular ones.  The general path finds that out level by level
// and moves the points every two levels.  Here the tree of midpoints is laid
// out ahead (it depends on the root's box alone), one sweep counts and weighs
// the points of each of its 2^L cells, and the sums up the tree settle, node
// by node from the root, whether coupe's loop ends at the midpoint: then that
// node's split is exactly coupe's.  A node whose search goes on is *open*;
// its ancestors are settled, so its box, points and weight are coupe's.  The
// points of the open nodes are gathered and each subtree is searched by one
// workgroup (rcb_subtree.h).  The ids come from each point's cell, or from a
// walk down the searched splits below an open node.
//
// Bound by memory: 4 D + w bytes read and 2 written per point by the sweep,
// 10 by the ids, besides the open points; the levels' moves (2 (4 D + w) per
// two levels) and passes are not made.  2^27 points 3D, 12 levels, 16-bit
// weights: see k_mid_count and k_mid_ids.
#pragma once

#include "rcb_small.h"

namespace coupe_hip {

constexpr uint32_t kMidLevels = 12;            // most levels: 4096 cells, two 16-bit halves of a map entry
constexpr uint32_t kMidDone = 0xffffffffu;     // map: the cell's points are settled
constexpr uint32_t kMidClasses = 3;            // open nodes of at most 2048 and 8192 points, and larger
constexpr uint32_t kMidClass[2] = {512 * 4, 512 * 16};

// An open node: its points are gathered at [begin, begin + count).
struct MidOpen {
    uint64_t sum;            // weight, accumulator bits
    float lo[kMaxDim], hi[kMaxDim];
    uint32_t begin, count;
    uint32_t node;           // heap index in its instance
    uint32_t inst;
    uint32_t axis, levels;   // axis of its split, levels left
};

// A point's place in the frontier (rcb_front.h): a node of it, kFrontSmall + an
// open node's number, or kFrontNone.
constexpr uint32_t kFrontSmall = 0x8000u, kFrontNone = 0xffffu;

// Counters of a call on this path (among the call's counters).
struct MidCounters {
    uint32_t open;                  // open nodes
    uint32_t points;                // their points
    uint32_t of_class[kMidClasses];
    uint32_t big;                   // open nodes too large for a workgroup: the call takes the general path
    uint32_t error;                 // a subtree's search did not end
    uint32_t taken;                 // nodes taken from the queue
};

// An instance's figures on this path: its open nodes are
// [first_open, first_open + n_open) of the table.
struct MidInstance {
    uint32_t first_open, n_open;
};

__device__ __forceinline__ uint64_t mid_cell_base(const Instance &I, uint32_t q) { return I.heap_base + q; }
__device__ __forceinline__ uint32_t mid_axis_levels(uint32_t levels, int a, int dim) {
    return (levels + (uint32_t)(dim - 1 - a)) / (uint32_t)dim;
}

// Box of an instance's root from the prologue's copies, as f32 (:604-605).
template <int D>
__device__ __forceinline__ void mid_box(const InstReduce *__restrict__ red, uint32_t n_inst, uint32_t q, int a,
                                        float &lo, float &hi) {
    uint64_t l = ~0ull, h = 0;
    for (int c = 0; c < kCopies; c++) {
        const InstReduce &r = red[(uint64_t)c * n_inst + q];
        l = r.bmin[a] < l ? r.bmin[a] : l;
        h = r.bmax[a] > h ? r.bmax[a] : h;
    }
    lo = (float)key_f64(l);
    hi = (float)key_f64(h);
}

// ---------------------------------------------------------------------------
// The sweep.  Per axis the midpoints of its levels, sorted; a point's rank
// among them gives its bits of the cell's path, spread to the levels of that
// axis.  Entry r of an axis: midpoint below, midpoint above (NaN past the
// ends), spread bits.
// ---------------------------------------------------------------------------
constexpr int kMidRanks = 1 << (kMidLevels / 2);   // of an axis: 64 in 2D, 16 in 3D

struct MidTables {
    float4 rank[kMaxDim][kMidRanks];
    float lo[kMaxDim], hi[kMaxDim];
};

template <int D>
__device__ __forceinline__ void mid_tables(MidTables &T, uint32_t levels) {
    constexpr float nan = __builtin_nanf("");
    for (int a = 0; a < D; a++) {
        const uint32_t la = mid_axis_levels(levels, a, D), n = 1u << la;
        for (uint32_t r = threadIdx.x; r < n; r += blockDim.x) {
            uint32_t bits = 0;
            for (uint32_t j = 0; j < la; j++)
                bits |= ((r >> (la - 1 - j)) & 1u) << (levels - 1 - (uint32_t)a - j * D);
            T.rank[a][r] = make_float4(r ? candidate(T.lo[a], T.hi[a], (int)r - 1, (int)n) : nan,
                                       r + 1 < n ? candidate(T.lo[a], T.hi[a], (int)r, (int)n) : nan,
                                       __builtin_bit_cast(float, bits), 0.0f);
        }
    }
}

// The spread bits of x on an axis of n ranks: the rank by an estimate, moved
// while the midpoints around it say so (whole wavefronts; seldom at all, at
// most n times).  NaN: rank 0, like !(c >= t).
__device__ __forceinline__ uint32_t mid_rank(const float4 *rank, int n, float x, float lo, float scale) {
    const float e = (x - lo) * scale;
    int r = (int)fminf(fmaxf(e, 0.0f), (float)(n - 1));
    float4 t = rank[r];
    for (int it = 0; it < n; it++) {
        const bool down = x < t.x, up = x >= t.y;
        if (__ballot(down | up) == 0) break;
        r += (up ? 1 : 0) - (down ? 1 : 0);
        t = rank[r];
    }
    return __builtin_bit_cast(uint32_t, t.z);
}

// Whether the shares of a grid stay below 2^24 points, so that the count and
// the weight of a cell (16-bit weights) fit one word.  The host allots the
// LDS by it, for the fewest workgroups the launch may have.
__host__ __device__ constexpr bool mid_one_word(uint64_t tiles, uint64_t grid) {
    return (tiles + grid - 1) / grid * kTile < (1ull << 24);
}
static_assert(mid_one_word(256ull * 8191, 256) && !mid_one_word(256ull * 8191 + 1, 256), "a share of 2^24 points");

// Runs of a wavefront's cells up to which they are added run by run (a random
// cloud has about 60; 2^27 points in mesh order: 553 us without, 505 with).
constexpr int kMidRuns = 14;

// w: the stored weights (w_src 0) or the caller's (w_src 1, 64-bit weights
// are not stored on this path).  cells: per copy (copies of them), the count
// and weight of every instance's cells.  code: each point's cell.
template <int D, int TPB, typename WL, typename Acc>
__global__ void __launch_bounds__(TPB)
k_mid_count(const Tile *__restrict__ tiles, uint32_t n_tiles, const Instance *__restrict__ insts,
            const InstReduce *__restrict__ red, uint32_t n_inst, const float *__restrict__ c0,
            const float *__restrict__ c1, const float *__restrict__ c2, const WL *__restrict__ w, int w_src,
            uint16_t *__restrict__ code, uint32_t *__restrict__ gcnt, Acc *__restrict__ gw, uint64_t cells,
            uint32_t copies) {
    constexpr int IT = kTile / TPB;
    __shared__ MidTables T;
    extern __shared__ __align__(16) char mid_lds[];
    uint32_t t0, t1;
    tile_range(n_tiles, t0, t1);
    if (t0 >= t1) return;
    const bool packed = packable<WL, Acc>() && mid_one_word(n_tiles, gridDim.x);
    Acc *sw = (Acc *)mid_lds;
    uint32_t *sc = nullptr;
    const int tid = threadIdx.x, lane = tid & 63;
    uint32_t cur = 0xffffffffu, levels = 0, n_cells = 0;
    uint64_t gbase = 0, wbase = 0;
    float lo[D], scale[D];
    int ranks[D];
    auto flush = [&]() {
        for (uint32_t c = tid; c < n_cells; c += TPB) {
            uint32_t cnt;
            Acc sum = sw[c];
            if (packed) {
                if constexpr (std::is_same<Acc, uint64_t>::value) {
                    cnt = (uint32_t)(sum >> kPackShift);
                    sum &= (1ull << kPackShift) - 1;
                } else {
                    cnt = sc[c];
                }
            } else {
                cnt = sc[c];
            }
            if (cnt) {
                atomicAdd(&gcnt[gbase + c], cnt);
                atomic_add_acc(&gw[gbase + c], sum);
            }
        }
    };
    for (uint32_t t = t0; t < t1; t++) {
        const Tile U = tiles[t];
        if (U.part != cur) {
            __syncthreads();
            if (cur != 0xffffffffu) flush();
            cur = U.part;
            const Instance &I = insts[cur];
            levels = I.levels;
            n_cells = 1u << levels;
            gbase = (uint64_t)(blockIdx.x % copies) * cells + mid_cell_base(I, cur);
            wbase = w_src ? I.src - I.begin : 0;   // (wraps: added to positions of the instance)
            sc = (uint32_t *)(mid_lds + (uint64_t)n_cells * sizeof(Acc));
            if (tid < D) mid_box<D>(red, n_inst, cur, tid, T.lo[tid], T.hi[tid]);
            __syncthreads();
            mid_tables<D>(T, levels);
            for (uint32_t c = tid; c < n_cells; c += TPB) {
                sw[c] = (Acc)0;
                if (!packed) sc[c] = 0;
            }
#pragma unroll
            for (int a = 0; a < D; a++) {
                ranks[a] = 1 << mid_axis_levels(levels, a, D);
                lo[a] = T.lo[a];
                scale[a] = (float)ranks[a] / (T.hi[a] - T.lo[a]);
            }
            __syncthreads();
        }
        // every load of the tile issued first (clamped, unconditional)
        float x[IT][D];
        WL wk[IT];
#pragma unroll
        for (int k = 0; k < IT; k++) {
            const uint64_t i = U.begin + min((uint32_t)(k * TPB + tid), U.count - 1u);
            x[k][0] = c0[i];
            x[k][1] = c1[i];
            if constexpr (D == 3) x[k][2] = c2[i];
            wk[k] = w[wbase + i];
        }
#pragma unroll
        for (int k = 0; k < IT; k++) {
            uint32_t c = 0;
#pragma unroll
            for (int a = 0; a < D; a++) c |= mid_rank(T.rank[a], ranks[a], x[k][a], lo[a], scale[a]);
            const uint32_t p = (uint32_t)(k * TPB + tid);
            if constexpr (packable<WL, Acc>()) {
                // Points in a mesh's order share cells with their neighbours, and
                // atomics of a wavefront on one address are done one by one: where
                // the lanes' cells form few runs (within rows of 16 lanes), a run
                // adds its prefix at its end and takes off the prefix before it at
                // its start (modulo 2^64: exact)
                const uint64_t heads = __ballot(c != dpp_row<0x111, true>(0u, c) || (tid & 15) == 0);
                if (packed && __popcll(heads) <= kMidRuns && (uint32_t)(k * TPB) + (tid | 63) < U.count) {
                    uint32_t s = (uint32_t)wk[k];
                    s += dpp_row<0x111, true>(0u, s);
                    s += dpp_row<0x112, true>(0u, s);
                    s += dpp_row<0x114, true>(0u, s);
                    s += dpp_row<0x118, true>(0u, s);
                    code[U.begin + p] = (uint16_t)c;
                    const uint64_t tails = heads >> 1 | 1ull << 63;
                    const unsigned long long upto = ((unsigned long long)((tid & 15) + 1) << kPackShift) + s;
                    const unsigned long long own = (1ull << kPackShift) + (uint32_t)wk[k];
                    if (tails >> lane & 1) atomicAdd((unsigned long long *)&sw[c], upto);
                    if ((heads >> lane & 1) && (tid & 15) != 0) atomicAdd((unsigned long long *)&sw[c], own - upto);
                    continue;
                }
            }
            if (p >= U.count) continue;
            code[U.begin + p] = (uint16_t)c;
            if (packed) {
                if constexpr (std::is_same<Acc, uint64_t>::value)
                    atomicAdd((unsigned long long *)&sw[c],
                              (1ull << kPackShift) + (unsigned long long)AccOps<Acc>::of(wk[k]));
            } else {
                atomicAdd(&sc[c], 1u);
                atomic_add_acc(&sw[c], AccOps<Acc>::of(wk[k]));
            }
        }
    }
    __syncthreads();
    flush();
}

// ---------------------------------------------------------------------------
// The tree: one workgroup per instance sums the cells up the tree (the copies
// are left clear), settles the nodes from the root down, and lists the open
// ones.  map: per cell the open node above it (heap index, and its number
// among the instance's open nodes << 16), or kMidDone.
// ---------------------------------------------------------------------------
constexpr uint32_t mid_tree_lds(uint32_t levels) { return (1u << levels) * (2 * 12 + 4); }

template <int D, int TPB, typename Acc>
__global__ void __launch_bounds__(TPB)
k_mid_tree(Instance *__restrict__ insts, const InstReduce *__restrict__ red, uint32_t n_inst, int wrap32,
           uint32_t *__restrict__ gcnt, Acc *__restrict__ gw, uint64_t cells, uint32_t copies,
           float *__restrict__ heap_split, uint32_t *__restrict__ map, MidInstance *__restrict__ minst,
           MidOpen *__restrict__ open, uint32_t *__restrict__ cursor, uint32_t *__restrict__ lists, uint64_t list_stride,
           uint64_t most, MidCounters *ctr) {
    using Ops = AccOps<Acc>;
    extern __shared__ __align__(16) char mid_lds[];
    __shared__ float s_lo[kMaxDim], s_hi[kMaxDim];
    __shared__ uint32_t s_open, s_first, s_min;
    const uint32_t q = blockIdx.x, tid = threadIdx.x;
    Instance &I = insts[q];
    const uint32_t levels = __builtin_amdgcn_readfirstlane(I.levels), n_cells = 1u << levels;
    const uint64_t cbase = mid_cell_base(I, q), hb = I.heap_base;
    Acc *w = (Acc *)mid_lds;                          // by heap index, 2 n_cells - 1 of each
    uint32_t *cnt = (uint32_t *)(w + 2 * n_cells);
    uint32_t *state = cnt + 2 * n_cells;              // 0: no point or above it open, 1: settled, 2 + number: open
    if (tid < (uint32_t)D) mid_box<D>(red, n_inst, q, (int)tid, s_lo[tid], s_hi[tid]);
    if (tid == 0) {
        s_open = 0;
        s_min = 0xffffffffu;
    }
    for (uint32_t c = tid; c < n_cells; c += TPB) {
        uint32_t n = 0;
        Acc s = (Acc)0;
        for (uint32_t k = 0; k < copies; k++) {
            const uint64_t g = (uint64_t)k * cells + cbase + c;
            n += gcnt[g];
            s += gw[g];
            gcnt[g] = 0;
            gw[g] = (Acc)0;
        }
        cnt[n_cells - 1 + c] = n;
        w[n_cells - 1 + c] = s;
    }
    __syncthreads();
    for (int l = (int)levels - 1; l >= 0; l--) {
        for (uint32_t s = tid; s < 1u << l; s += TPB) {
            const uint32_t h = (1u << l) - 1 + s;
            cnt[h] = cnt[2 * h + 1] + cnt[2 * h + 2];
            w[h] = w[2 * h + 1] + w[2 * h + 2];
        }
        __syncthreads();
    }
    if (tid == 0) {   // the root's weight as the general path has it
        uint64_t su = 0;
        double sf = 0.0;
        for (int c = 0; c < kCopies; c++) {
            su += red[(uint64_t)c * n_inst + q].sum_u64;
            sf += red[(uint64_t)c * n_inst + q].sum_f64;
        }
        if constexpr (std::is_same<Acc, double>::value) w[0] = sf;
        else w[0] = su;
    }
    __syncthreads();
    float lo[kMaxDim], hi[kMaxDim];
    bool finite = true;   // and so is every midpoint
#pragma unroll
    for (int a = 0; a < kMaxDim; a++) {
        lo[a] = a < D ? s_lo[a] : 0.0f;
        hi[a] = a < D ? s_hi[a] : 0.0f;
        finite = finite && fabsf(lo[a]) < 1.0e38f && fabsf(hi[a]) < 1.0e38f;
    }
    const double tol = I.tol;
    // the box of node (l, s) on axis a: the bisections of its ancestors there
    auto window = [&](uint32_t l, uint32_t s, int a, float &bl, float &bh) {
        bl = sel3(a, lo[0], lo[1], lo[2]);
        bh = sel3(a, hi[0], hi[1], hi[2]);
        for (uint32_t m = (uint32_t)a; m < l; m += D) {
            const float t = (bl + bh) / 2.0f;
            const bool right = (s >> (l - m - 1)) & 1u;
            bl = right ? t : bl;
            bh = right ? bh : t;
        }
    };
    for (uint32_t l = 0; l < levels; l++) {
        for (uint32_t s = tid; s < 1u << l; s += TPB) {
            const uint32_t h = (1u << l) - 1 + s, n = cnt[h];
            const bool live = n > 0 && (l == 0 || state[(h - 1) / 2] == 1u);
            uint32_t st = 0;
            if (live) {
                const uint32_t cl = cnt[2 * h + 1];
                const Acc S = w[h], wl = w[2 * h + 1];
                if (finite && cl != n && within(Ops::f64(wl, wrap32), Ops::f64(S, wrap32) / 2.0, tol)) {
                    float bl, bh;
                    window(l, s, (int)(l % D), bl, bh);
                    heap_split[hb + h] = (bl + bh) / 2.0f;
                    w[2 * h + 2] = Ops::sub(S, wl);   // the right child's weight (:603-641)
                    st = 1;
                } else {
                    st = 2u + atomicAdd(&s_open, 1u);
                }
            }
            state[h] = st;
        }
        __syncthreads();
    }
    const uint32_t n_open = s_open;
    if (tid == 0) {
        s_first = n_open ? atomicAdd(&ctr->open, n_open) : 0u;
        minst[q] = MidInstance{s_first, n_open};
    }
    __syncthreads();
    const uint32_t first = s_first;
    for (uint32_t h = tid; h < n_cells - 1; h += TPB) {
        const uint32_t st = state[h];
        if (st < 2) continue;
        const uint32_t l = 31u - (uint32_t)__builtin_clz(h + 1), s = h + 1 - (1u << l), e = first + st - 2;
        MidOpen O;
        O.sum = Ops::to_bits(w[h]);
        O.count = cnt[h];
        O.begin = atomicAdd(&ctr->points, O.count);
        O.node = h;
        O.inst = q;
        O.axis = l % D;
        O.levels = levels - l;
        for (int a = 0; a < kMaxDim; a++) {
            O.lo[a] = O.hi[a] = 0.0f;
            if (a < D) window(l, s, a, O.lo[a], O.hi[a]);
        }
        open[e] = O;
        cursor[e] = O.begin;
        const uint32_t k = O.count <= kMidClass[0] ? 0u : (O.count <= kMidClass[1] ? 1u : 2u);
        lists[k * list_stride + atomicAdd(&ctr->of_class[k], 1u)] = e;
        if (O.count > kMidClass[1] && (uint64_t)O.count * O.levels > most) atomicAdd(&ctr->big, 1u);
    }
    uint32_t m = 0xffffffffu;   // smallest settled leaf
    for (uint32_t c = tid; c < n_cells; c += TPB) {
        uint32_t entry = kMidDone;
        for (uint32_t l = 0; l < levels; l++) {
            const uint32_t h = (1u << l) - 1 + (c >> (levels - l)), st = state[h];
            if (st != 1u) {
                if (st >= 2u) entry = h | (st - 2u) << 16;
                break;
            }
        }
        map[cbase + c] = entry;
        if (entry == kMidDone && cnt[n_cells - 1 + c]) m = min(m, n_cells - 1 + c);
    }
    m = wave_min(m);
    if (lane_id() == 0) atomicMin(&s_min, m);
    __syncthreads();
    if (tid == 0) I.min_id = s_min == 0xffffffffu ? ~0ull : (uint64_t)s_min;   // (the subtrees lower it)
}

// One gathered point: a single store per point, whose address no neighbour
// shares when the input is in random order (4096 instances 3D: gather 2.53 -> 1.62 ms
// against one store per coordinate and weight).
template <int D, typename WL>
struct alignas(sizeof(WL) == 8 && D == 3 ? 8 : 16) MidPoint {
    float x[D];
    WL w;
};

// ---------------------------------------------------------------------------
// The open nodes' points, gathered node by node (their order within a node is
// free).  Workgroups take contiguous shares of the tiles: each counts its
// points per open node, takes places for them (one atomic per node) and
// writes them, reading the 2-byte cells twice.
// ---------------------------------------------------------------------------
// FRONT: code holds the points' nodes of the frontier (rcb_front.h) instead of
// cells, and gate the nodes it has left.
template <int D, typename WL, bool FRONT>
__global__ void __launch_bounds__(kBlock)
k_mid_gather(const Tile *__restrict__ tiles, uint32_t n_tiles, const Instance *__restrict__ insts,
             const MidInstance *__restrict__ minst, const float *__restrict__ c0, const float *__restrict__ c1,
             const float *__restrict__ c2, const WL *__restrict__ w, int w_src, const uint16_t *__restrict__ code,
             const uint32_t *__restrict__ map, uint32_t *__restrict__ cursor, MidPoint<D, WL> *__restrict__ gathered,
             const MidCounters *ctr, const uint32_t *gate) {
    if (ctr->open == 0 || ctr->big || (FRONT && *gate)) return;
    __shared__ uint16_t num[FRONT ? 1 : 1 << kMidLevels];   // open node of a cell, 0xffff: settled
    __shared__ uint32_t place[1 << (kMidLevels - 1)];    // at most half as many open nodes as cells
    const int tid = threadIdx.x;
    uint32_t t0, t1;
    tile_range(n_tiles, t0, t1);
    for (uint32_t t = t0; t < t1;) {
        const uint32_t q = tiles[t].part;
        uint32_t e = t;   // [t, e): this share's tiles of instance q
        const Instance &I = insts[q];
        {
            const uint32_t last = I.tile_begin + (uint32_t)((I.count + kTile - 1) / kTile);
            e = last < t1 ? last : t1;
        }
        const MidInstance M = FRONT ? MidInstance{0u, ctr->open} : minst[q];
        if (M.n_open == 0) {
            t = e;
            continue;
        }
        const uint32_t n_cells = 1u << I.levels;
        const uint64_t cbase = mid_cell_base(I, q), wbase = w_src ? I.src - I.begin : 0;
        __syncthreads();
        if constexpr (!FRONT)
            for (uint32_t c = tid; c < n_cells; c += kBlock) {
                const uint32_t m = map[cbase + c];
                num[c] = m == kMidDone ? (uint16_t)0xffffu : (uint16_t)(m >> 16);
            }
        auto open_of = [&](uint16_t c) -> uint16_t {
            if constexpr (FRONT) return c >= kFrontSmall && c != kFrontNone ? (uint16_t)(c - kFrontSmall) : (uint16_t)0xffffu;
            else return num[c];
        };
        for (uint32_t k = tid; k < M.n_open; k += kBlock) place[k] = 0;
        __syncthreads();
        const uint64_t begin = tiles[t].begin, end = tiles[e - 1].begin + tiles[e - 1].count;
        // eight points of a thread at a time: their loads are issued together
        constexpr int G = 8;
        for (uint64_t i0 = begin; i0 < end; i0 += kBlock * G) {
            uint16_t o[G];
#pragma unroll
            for (int k = 0; k < G; k++) {
                const uint64_t i = i0 + (uint32_t)(k * kBlock) + tid;
                o[k] = code[i < end ? i : end - 1];
            }
#pragma unroll
            for (int k = 0; k < G; k++) {
                const uint16_t m = open_of(o[k]);
                if (m != 0xffffu && i0 + (uint32_t)(k * kBlock) + tid < end) atomicAdd(&place[m], 1u);
            }
        }
        __syncthreads();
        for (uint32_t k = tid; k < M.n_open; k += kBlock)
            if (place[k]) place[k] = atomicAdd(&cursor[M.first_open + k], place[k]);
        __syncthreads();
        for (uint64_t i0 = begin; i0 < end; i0 += kBlock * G) {
            uint16_t o[G];
#pragma unroll
            for (int k = 0; k < G; k++) {
                const uint64_t i = i0 + (uint32_t)(k * kBlock) + tid;
                o[k] = code[i < end ? i : end - 1];
            }
            bool any = false;
#pragma unroll
            for (int k = 0; k < G; k++) {
                o[k] = i0 + (uint32_t)(k * kBlock) + tid < end ? open_of(o[k]) : (uint16_t)0xffffu;
                any |= o[k] != 0xffffu;
            }
            if (__ballot(any) == 0) continue;
            MidPoint<D, WL> r[G];
#pragma unroll
            for (int k = 0; k < G; k++) {
                const uint64_t i = i0 + (uint32_t)(k * kBlock) + tid;
                if (o[k] != 0xffffu) {
                    r[k].x[0] = c0[i];
                    r[k].x[1] = c1[i];
                    if constexpr (D == 3) r[k].x[2] = c2[i];
                    r[k].w = w[wbase + i];
                }
            }
#pragma unroll
            for (int k = 0; k < G; k++) {
                if (o[k] == 0xffffu) continue;
                gathered[atomicAdd(&place[o[k]], 1u)] = r[k];
            }
        }
        t = e;
    }
}

// ---------------------------------------------------------------------------
// The open nodes' subtrees, one workgroup each.
// ---------------------------------------------------------------------------
// Root of an open node's subtree, and where its splits go.
template <typename WL>
__device__ __forceinline__ SubRoot mid_root(const MidOpen &O, const Instance &I, int wrap32) {
    SubRoot R;
    for (int a = 0; a < kMaxDim; a++) { R.lo[a] = O.lo[a]; R.hi[a] = O.hi[a]; }
    R.axis = __builtin_amdgcn_readfirstlane(O.axis);
    R.levels = __builtin_amdgcn_readfirstlane(O.levels);
    R.tol = I.tol;
    R.wrap32 = wrap32;
    R.packed = std::is_same<WL, uint16_t>::value && O.count < (1u << 24);
    return R;
}

// split_out of a subtree: the split into the instance's heap (its heap index
// from the subtree's), and at the last level the smallest leaf present.
struct MidSplits {
    float *heap;         // the instance's heap
    uint32_t node;       // heap index of the subtree's root
    uint32_t levels;     // of the subtree
    uint32_t *min_leaf;  // LDS
    __device__ __forceinline__ void operator()(uint32_t level, uint32_t slot, uint32_t n, uint32_t left,
                                               float split) const {
        if (n == 0) return;
        const uint32_t h = ((node + 1) << level) - 1 + slot;
        heap[h] = left == n ? __builtin_nanf("") : split;   // every point left: as the descent walks it
        if (level + 1 == levels) atomicMin(min_leaf, left ? 2 * h + 1 : 2 * h + 2);
    }
};

// A node whose points fit the workgroup's registers.
template <int D, int TPB, int IT, typename WL, typename Acc>
__device__ __forceinline__ bool mid_registers(uint32_t count, const SubRoot &R, Acc sum,
                                              const MidPoint<D, WL> *__restrict__ pts, uint32_t *ctr,
                                              const MidSplits &out) {
    float x[IT][D];
    small_points<D, TPB, IT>(count, x, [&](uint64_t i, float (&p)[D]) {
#pragma unroll
        for (int a = 0; a < D; a++) p[a] = pts[i].x[a];
    });
    RegSlots<IT> slot;
    return reg_levels<D, TPB, IT, kWeightAcc, WL, Acc>(count, x, [&](uint32_t i) { return pts[i].w; }, R, sum, ctr, slot,
                                                       out);
}

// A larger node: its points stay in memory (read again per pass, from the
// caches), their slots beside them.
template <int D, int TPB, typename WL, typename Acc>
__device__ __forceinline__ bool mid_memory(uint32_t count, const SubRoot &R, Acc sum,
                                           const MidPoint<D, WL> *__restrict__ pts, uint16_t *__restrict__ slots,
                                           uint32_t *ctr, const MidSplits &out) {
    // G points of a thread in flight: a CU has this workgroup alone (2^27 jittered
    // points, nodes of up to 131072: 356 us with B in flight, 278 with G)
    constexpr int B = kAhead, G = 16;
    const uint32_t tid = threadIdx.x;
    SubTree<Acc, TPB> T(sub_slots(R.levels));
    bool first = true;   // every point in slot 0: not read
    return sub_levels<D, TPB, Acc>(
        T, R, count, sum, ctr,
        [&](int nb, int a) {
            auto points = [&](uint32_t i0, auto many) {
                constexpr int M = decltype(many)::value;
                uint16_t sg[M];
                float xg[M];
                WL wg[M];
#pragma unroll
                for (int g = 0; g < M; g++) {
                    const uint32_t i = i0 + (uint32_t)(g * TPB) + tid, p = i < count ? i : count - 1;
                    xg[g] = pts[p].x[a];
                    wg[g] = pts[p].w;
                    sg[g] = first ? (uint16_t)0 : slots[p];
                }
#pragma unroll
                for (int g = 0; g < M; g += B) {
                    uint32_t s[B];
                    float xa[B];
                    Acc wk[B];
                    bool valid[B];
#pragma unroll
                    for (int j = 0; j < B; j++) {
                        valid[j] = i0 + (uint32_t)((g + j) * TPB) + tid < count;
                        xa[j] = xg[g + j];
                        wk[j] = AccOps<Acc>::of(wg[g + j]);
                        s[j] = sg[g + j];
                    }
                    sub_bin<B>(T, s, [&](int j, uint32_t) { return xa[j]; }, wk, valid, nb, R.packed);
                }
            };
            uint32_t i0 = 0;
            for (; i0 + TPB * G <= count; i0 += TPB * G) points(i0, std::integral_constant<int, G>{});
            for (; i0 < count; i0 += TPB * B) points(i0, std::integral_constant<int, B>{});
        },
        [&](int a) {
            auto points = [&](uint32_t i0, auto many) {
                constexpr int M = decltype(many)::value;
                uint32_t s[M];
                float xa[M];
#pragma unroll
                for (int j = 0; j < M; j++) {   // (each thread its own points: no other touches their slots)
                    const uint32_t i = i0 + (uint32_t)(j * TPB) + tid, p = i < count ? i : count - 1;
                    xa[j] = pts[p].x[a];
                    s[j] = first ? 0u : (uint32_t)slots[p];
                }
#pragma unroll
                for (int j = 0; j < M; j++) {
                    const uint32_t i = i0 + (uint32_t)(j * TPB) + tid;
                    if (i < count) slots[i] = (uint16_t)(2 * s[j] + (xa[j] >= T.at(s[j]).win.x ? 1u : 0u));
                }
            };
            uint32_t i0 = 0;
            for (; i0 + TPB * G <= count; i0 += TPB * G) points(i0, std::integral_constant<int, G>{});
            for (; i0 < count; i0 += TPB * B) points(i0, std::integral_constant<int, B>{});
            first = false;
        },
        out);
}

// The workgroups take the nodes from a queue, the large ones first.
constexpr int kMidThreads = 512;
template <int D, typename WL, typename Acc>
__global__ void __launch_bounds__(kMidThreads)
k_mid_search(const MidOpen *__restrict__ open, const uint32_t *__restrict__ lists, uint64_t list_stride,
             Instance *__restrict__ insts, const MidPoint<D, WL> *__restrict__ gathered,
             uint16_t *__restrict__ slots, int wrap32, float *__restrict__ heap_split, MidCounters *ctr,
             const uint32_t *gate) {
    if (ctr->big || (gate && *gate)) return;
    constexpr int TPB = kMidThreads;
    SmallShared &sh = *(SmallShared *)sub_lds_base;
    const uint32_t n0 = ctr->of_class[0], n1 = ctr->of_class[1], n2 = ctr->of_class[2], tid = threadIdx.x;
    for (;;) {
        __syncthreads();   // the last node's LDS is free
        if (tid == 0) {
            sh.flags = atomicAdd(&ctr->taken, 1u);
            sh.min_slot = 0xffffffffu;
        }
        __syncthreads();
        uint32_t g = __builtin_amdgcn_readfirstlane(sh.flags);   // every workgroup gets past the end once, and leaves
        if (g >= n0 + n1 + n2) return;
        int k = 2;
        if (g >= n2) { g -= n2; k = 1; }
        if (k == 1 && g >= n1) { g -= n1; k = 0; }
        const MidOpen &O = open[lists[(uint64_t)k * list_stride + g]];
        Instance &I = insts[O.inst];
        const uint32_t count = __builtin_amdgcn_readfirstlane(O.count), begin = __builtin_amdgcn_readfirstlane(O.begin);
        const SubRoot R = mid_root<WL>(O, I, wrap32);
        const MidSplits out{heap_split + I.heap_base, O.node, R.levels, &sh.min_slot};
        const Acc sum = AccOps<Acc>::from_bits(O.sum);
        const MidPoint<D, WL> *pts = gathered + begin;
        bool ok;
        if (k == 0) ok = mid_registers<D, TPB, 4, WL, Acc>(count, R, sum, pts, sh.ctr, out);
        else if (k == 1) ok = mid_registers<D, TPB, 16, WL, Acc>(count, R, sum, pts, sh.ctr, out);
        else ok = mid_memory<D, TPB, WL, Acc>(count, R, sum, pts, slots + begin, sh.ctr, out);
        __syncthreads();
        if (tid == 0) {
            atomicMin((unsigned long long *)&I.min_id, (unsigned long long)sh.min_slot);
            if (!ok) atomicOr(&ctr->error, 1u);
        }
    }
}

// ---------------------------------------------------------------------------
// Ids in input order: a settled cell is its leaf; below an open node the
// point walks the searched splits (the tile's coordinates are read only then).
// ---------------------------------------------------------------------------
template <int D, bool NT>
__global__ void __launch_bounds__(kBlock)
k_mid_ids(const Tile *__restrict__ tiles, uint32_t n_tiles, const Instance *__restrict__ insts,
          const MidInstance *__restrict__ minst, const uint16_t *__restrict__ code, const uint32_t *__restrict__ map,
          const float *__restrict__ heap_split, const float *__restrict__ c0, const float *__restrict__ c1,
          const float *__restrict__ c2, uint64_t *__restrict__ out, const MidCounters *ctr) {
    if (ctr->big) return;
    __shared__ uint16_t node[1 << kMidLevels];   // open node of a cell, 0xffff: settled
    __shared__ float heap[1 << kMidLevels];      // the instance's splits
    const int tid = threadIdx.x;
    uint32_t t0, t1;
    tile_range(n_tiles, t0, t1);
    uint32_t cur = 0xffffffffu, levels = 0, leaf0 = 0;
    uint64_t off = 0, src = 0;
    bool any_open = false;
    for (uint32_t t = t0; t < t1; t++) {
        const Tile U = tiles[t];
        if (U.part != cur) {
            cur = U.part;
            const Instance &I = insts[cur];
            levels = I.levels;
            leaf0 = (1u << levels) - 1;
            off = I.min_id;
            src = I.src - I.begin;
            any_open = minst[cur].n_open != 0;
            if (any_open) {
                const uint64_t cbase = mid_cell_base(I, cur), hb = I.heap_base;
                __syncthreads();
                for (uint32_t c = tid; c <= leaf0; c += kBlock) {
                    node[c] = (uint16_t)map[cbase + c];   // kMidDone: 0xffff
                    if (c < leaf0) heap[c] = heap_split[hb + c];
                }
                __syncthreads();
            }
        }
        uint32_t h[kItems];
        uint64_t at[kItems];
#pragma unroll
        for (int k = 0; k < kItems; k++) {
            at[k] = U.begin + min((uint32_t)(k * kBlock + tid), U.count - 1u);
            if constexpr (NT) h[k] = __builtin_nontemporal_load(&code[at[k]]);
            else h[k] = code[at[k]];
        }
        if (!any_open) {
#pragma unroll
            for (int k = 0; k < kItems; k++) h[k] += leaf0;
        } else {
            bool walk = false;
#pragma unroll
            for (int k = 0; k < kItems; k++) {
                const uint32_t o = node[h[k]];
                h[k] = o != 0xffffu ? o : leaf0 + h[k];
                walk |= h[k] < leaf0;
            }
            if (__ballot(walk)) {
                float x[kItems][D];
#pragma unroll
                for (int k = 0; k < kItems; k++) {
                    if (h[k] < leaf0) {
                        x[k][0] = c0[at[k]];
                        x[k][1] = c1[at[k]];
                        if constexpr (D == 3) x[k][2] = c2[at[k]];
                    }
                }
#pragma unroll
                for (int k = 0; k < kItems; k++) {
                    if (h[k] < leaf0) {
                        int a = (int)((31u - (uint32_t)__builtin_clz(h[k] + 1)) % D);
                        do {
                            const float xa = a == 0 ? x[k][0] : (a == 1 ? x[k][1] : x[k][D - 1]);
                            h[k] = 2 * h[k] + (xa >= heap[h[k]] ? 2u : 1u);
                            a = a + 1 == D ? 0 : a + 1;
                        } while (h[k] < leaf0);
                    }
                }
            }
        }
#pragma unroll
        for (int k = 0; k < kItems; k++) {
            const uint32_t p = (uint32_t)(k * kBlock + tid);
            if (p < U.count) {
                if constexpr (NT) __builtin_nontemporal_store((uint64_t)h[k] - off, &out[src + U.begin + p]);
                else out[src + U.begin + p] = (uint64_t)h[k] - off;
            }
        }
    }
}

}  // namespace coupe_hip
