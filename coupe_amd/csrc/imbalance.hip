// imbalance.hip -- per-part loads and imbalance of a partition, on device
// (coupe/src/imbalance.rs:14-105).  Entry points in include/coupe_hip.h.
#include <hip/hip_runtime.h>

#include <cstring>
#include <new>
#include <type_traits>
#include <vector>

#include "rcb_engine.h"
#include "rcb_device.h"

namespace coupe_hip {

// ---------------------------------------------------------------------------
// Per-part loads (coupe::imbalance::compute_parts_load, imbalance.rs:14-39):
// a weight histogram over part ids, privatised in LDS when the parts fit.
// Integer weights add in 64-bit two's complement (i32 wrapping is recovered
// by truncation); f64 weights add in f64.  Ids >= num_parts are counted as
// errors (coupe's `acc[part]` would panic).
//
// Up to kLoadLds parts a workgroup sums in LDS and adds its sums to its XCD's
// copy of the loads (blockIdx mod kCopies); k_loads_combine adds the copies,
// leaves them clear for the next call and writes the result where the host
// reads it.  Bound by memory (8 + w bytes per point): each thread has eight
// ids and weights in flight, and two workgroups of 1024 per CU flush, not
// five of 256 (2^24 points, f64, 1024 parts: 143 -> 67 us per call, the kernel 50 us).
// ---------------------------------------------------------------------------
constexpr uint32_t kLoadLds = 4096;   // parts privatised in LDS (32 KB)
constexpr int kLoadBlock = 1024;
constexpr int kLoadItems = 8;

template <typename WIN, typename Acc, bool LDS>
__global__ void __launch_bounds__(kLoadBlock)
k_parts_load(const uint64_t *__restrict__ ids, const WIN *__restrict__ w, uint64_t n, uint64_t num_parts,
             Acc *__restrict__ loads, unsigned long long *bad) {
    // LDS: loads holds kCopies copies of num_parts sums; else one
    extern __shared__ __align__(16) char load_lds[];
    Acc *sl = (Acc *)load_lds;
    if constexpr (LDS) {
        for (uint32_t j = threadIdx.x; j < num_parts; j += kLoadBlock) sl[j] = (Acc)0;
        __syncthreads();
    }
    uint32_t nbad = 0;
    const uint64_t stride = (uint64_t)gridDim.x * kLoadBlock * kLoadItems;
    for (uint64_t i0 = (uint64_t)blockIdx.x * kLoadBlock * kLoadItems; i0 < n; i0 += stride) {
        uint64_t p[kLoadItems];
        WIN v[kLoadItems];
#pragma unroll
        for (int k = 0; k < kLoadItems; k++) {   // clamped, unconditional
            const uint64_t i = i0 + (uint32_t)(k * kLoadBlock) + threadIdx.x, c = i < n ? i : n - 1;
            p[k] = __builtin_nontemporal_load(&ids[c]);
            v[k] = __builtin_nontemporal_load(&w[c]);
        }
#pragma unroll
        for (int k = 0; k < kLoadItems; k++) {
            if (i0 + (uint32_t)(k * kLoadBlock) + threadIdx.x >= n) continue;
            if (p[k] >= num_parts) nbad++;
            else if constexpr (LDS) atomic_add_acc(&sl[(uint32_t)p[k]], AccOps<Acc>::of(v[k]));
            else atomic_add_acc(&loads[p[k]], AccOps<Acc>::of(v[k]));
        }
    }
    nbad = wave_sum(nbad);
    if (lane_id() == 0 && nbad) atomicAdd(bad, (unsigned long long)nbad);
    if constexpr (LDS) {
        __syncthreads();
        Acc *mine = loads + (uint64_t)(blockIdx.x % kCopies) * num_parts;
        for (uint32_t j = threadIdx.x; j < num_parts; j += kLoadBlock)
            if (sl[j] != (Acc)0) atomic_add_acc(&mine[j], sl[j]);
    }
}

// out: pinned host memory, the loads and then the count of bad ids.
template <typename Acc>
__global__ void __launch_bounds__(kBlock)
k_loads_combine(Acc *__restrict__ loads, uint32_t num_parts, unsigned long long *bad, Acc *out,
                unsigned long long *out_bad) {
    const uint32_t j = blockIdx.x * kBlock + threadIdx.x;
    if (j == 0) {
        *out_bad = *bad;
        *bad = 0;
    }
    if (j >= num_parts) return;
    Acc s = (Acc)0;
#pragma unroll
    for (int c = 0; c < kCopies; c++) {
        s += loads[(uint64_t)c * num_parts + j];
        loads[(uint64_t)c * num_parts + j] = (Acc)0;
    }
    out[j] = s;
}

namespace {

void ck(hipError_t e) {
    if (e != hipSuccess) throw HipFailure{e};
}

// Loads in the accumulator type, copied to the host.
template <typename WIN, typename Acc>
void loads_typed(Context &cx, hipStream_t st, const uint64_t *ids, uint64_t n, const WIN *w, uint64_t num_parts,
                 std::vector<Acc> &out, uint64_t *bad) {
    const bool lds = num_parts <= kLoadLds;
    const uint64_t sums = lds ? kCopies * kLoadLds : num_parts;   // a fixed place for the count of bad ids
    const size_t need = sums * sizeof(Acc) + sizeof(unsigned long long);
    const bool fresh = cx.loads.bytes < need;
    cx.loads.ensure(need);
    Acc *d = (Acc *)cx.loads.ptr;
    unsigned long long *d_bad = (unsigned long long *)(d + sums);
    if (cx.cu_count <= 0) ck(hipDeviceGetAttribute(&cx.cu_count, hipDeviceAttributeMultiprocessorCount, cx.device));
    if (!cx.host_scratch) ck(hipHostMalloc(&cx.host_scratch, kHostScratch, hipHostMallocDefault));
    static_assert(kHostScratch >= kLoadLds * sizeof(Acc) + 8, "the loads come back through the pinned area");
    // the LDS form leaves the sums clear; anything else clears them first
    if (fresh || !lds || !cx.loads_clean) ck(hipMemsetAsync(cx.loads.ptr, 0, cx.loads.bytes, st));
    cx.loads_clean = false;   // until this call completes
    if (n) {
        const uint64_t per = (uint64_t)kLoadBlock * kLoadItems;
        const unsigned g = (unsigned)std::min<uint64_t>(2ull * (uint64_t)std::max(cx.cu_count, 1), (n + per - 1) / per);
        if (lds)
            k_parts_load<WIN, Acc, true><<<g, kLoadBlock, num_parts * sizeof(Acc), st>>>(ids, w, n, num_parts, d, d_bad);
        else
            k_parts_load<WIN, Acc, false><<<g, kLoadBlock, 0, st>>>(ids, w, n, num_parts, d, d_bad);
        ck(hipGetLastError());
    }
    out.resize(num_parts);
    unsigned long long hb = 0;
    if (lds) {
        volatile unsigned long long *h_bad = (volatile unsigned long long *)cx.host_scratch;
        Acc *h = (Acc *)((char *)cx.host_scratch + 8);
        k_loads_combine<Acc><<<(unsigned)(num_parts / kBlock + 1), kBlock, 0, st>>>(d, (uint32_t)num_parts, d_bad, h,
                                                                                   (unsigned long long *)h_bad);
        ck(hipGetLastError());
        ck(hipStreamSynchronize(st));
        hb = *h_bad;
        if (num_parts) memcpy(out.data(), h, num_parts * sizeof(Acc));
        cx.loads_clean = true;
    } else {
        ck(hipMemcpyAsync(out.data(), d, num_parts * sizeof(Acc), hipMemcpyDeviceToHost, st));
        ck(hipMemcpyAsync(&hb, d_bad, sizeof hb, hipMemcpyDeviceToHost, st));
        ck(hipStreamSynchronize(st));
    }
    *bad = hb;
}

}  // namespace

// Loads converted to the weight type (i32 wraps like Rust's release `+=`).
enum coupe_err parts_load(Context &cx, hipStream_t st, const uint64_t *ids, uint64_t n, int wkind, const void *w,
                          uint64_t num_parts, void *host_loads) {
    if (wkind != COUPE_INT && wkind != COUPE_INT64 && wkind != COUPE_DOUBLE) return COUPE_ERR_BAD_TYPE;
    if (n && (!ids || !w)) return COUPE_ERR_CRASH;
    try {
        ck(hipSetDevice(cx.device));
        uint64_t bad = 0;
        if (wkind == COUPE_DOUBLE) {
            std::vector<double> v;
            loads_typed<double, double>(cx, st, ids, n, (const double *)w, num_parts, v, &bad);
            if (bad) return COUPE_ERR_CRASH;
            memcpy(host_loads, v.data(), num_parts * sizeof(double));
        } else {
            std::vector<uint64_t> v;
            if (wkind == COUPE_INT)
                loads_typed<int32_t, uint64_t>(cx, st, ids, n, (const int32_t *)w, num_parts, v, &bad);
            else
                loads_typed<int64_t, uint64_t>(cx, st, ids, n, (const int64_t *)w, num_parts, v, &bad);
            if (bad) return COUPE_ERR_CRASH;
            for (uint64_t j = 0; j < num_parts; j++) {
                if (wkind == COUPE_INT) ((int32_t *)host_loads)[j] = (int32_t)(uint32_t)v[j];
                else ((int64_t *)host_loads)[j] = (int64_t)v[j];
            }
        }
    } catch (const HipFailure &f) {
        (void)hipGetLastError();
        return map_hip_error(f.err);
    } catch (const std::bad_alloc &) {
        return COUPE_ERR_ALLOC;
    }
    return COUPE_ERR_OK;
}

// imbalance.rs:41-77: max over parts of (load - ideal) / ideal, with
// ideal = (sum of the loads, in W) / num_parts; 0 when num_parts or ideal is 0.
enum coupe_err imbalance(Context &cx, hipStream_t st, const uint64_t *ids, uint64_t n, int wkind, const void *w,
                         uint64_t num_parts, double *out) {
    *out = 0.0;
    if (num_parts == 0) return COUPE_ERR_OK;
    std::vector<unsigned char> buf(num_parts * 8);
    enum coupe_err e = parts_load(cx, st, ids, n, wkind, w, num_parts, buf.data());
    if (e != COUPE_ERR_OK) return e;
    std::vector<double> f(num_parts);
    double total;
    if (wkind == COUPE_DOUBLE) {
        const double *l = (const double *)buf.data();
        double s = 0.0;
        for (uint64_t j = 0; j < num_parts; j++) { s += l[j]; f[j] = l[j]; }
        total = s;
    } else if (wkind == COUPE_INT) {
        const int32_t *l = (const int32_t *)buf.data();
        uint32_t s = 0;
        for (uint64_t j = 0; j < num_parts; j++) { s += (uint32_t)l[j]; f[j] = (double)l[j]; }
        total = (double)(int32_t)s;
    } else {
        const int64_t *l = (const int64_t *)buf.data();
        uint64_t s = 0;
        for (uint64_t j = 0; j < num_parts; j++) { s += (uint64_t)l[j]; f[j] = (double)l[j]; }
        total = (double)(int64_t)s;
    }
    const double ideal = total / (double)num_parts;
    if (ideal == 0.0) return COUPE_ERR_OK;
    double mx = -1.0 / 0.0;
    for (uint64_t j = 0; j < num_parts; j++) {
        const double r = (f[j] - ideal) / ideal;
        if (r > mx) mx = r;
    }
    *out = mx;
    return COUPE_ERR_OK;
}

}  // namespace coupe_hip
