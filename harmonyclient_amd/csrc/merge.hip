// Top-k merge of per-partition results: the final step of a list-sharded
// search, where each partition (a GPU, or a worker in the reference's
// distributed modes) returns its own sorted top-k of every query and the
// merged row is the best k of their union (src/Index.cpp:1327-1343, which
// offers each partition's entries to a k-heap and sorts it).
//
// A row of at most 1024 entries with k <= 256 is one wave's: its keys stay in
// registers, the k-th key is found bit by bit and only the k kept are sorted.
// Larger rows: one 256-thread workgroup per query streams the entries through
// the LDS top-k (threshold filter + bitonic compaction).  Either way the
// result is the exact top-k in the (distance, id) order; entries with a
// negative id (a partial result's sentinel padding) are skipped.
#include <climits>
#include <cstring>
#include <string>

#include "index_impl.hpp"
#include "select.hpp"
#include "wave.hpp"

namespace hivf {
namespace {

constexpr int kMergeNT = 256;

struct MergeArgs {
    const float* Dp;   // [parts][n][k_in]
    const int64_t* Ip;
    int64_t n;
    int parts;
    int k_in;
    int k;
    int metric;
    float* D;          // [n][k]
    int64_t* I;
};

__global__ __launch_bounds__(kMergeNT) void merge_kernel(MergeArgs a) {
    __shared__ LdsTopK<kMergeNT, 2048> tk;
    const int64_t q = blockIdx.x;
    tk.init();
    const int64_t total = (int64_t)a.parts * a.k_in;
    for (int64_t base = 0; base < total; base += kMergeNT) {
        const uint64_t thr = tk.thr;
        const int64_t e = base + threadIdx.x;
        if (e < total) {
            const int64_t p = e / a.k_in, i = e % a.k_in;
            const size_t off = ((size_t)p * a.n + q) * a.k_in + i;
            const int64_t id = a.Ip[off];
            const float v = a.Dp[off];
            const float r = a.metric == kL2 ? v : -v;
            // r < FLT_MAX: the heap's strict admission against its sentinel
            // (never inf or NaN)
            if (id >= 0 && r < FLT_MAX) tk.offer(make_key(r, (uint32_t)id), thr);
        }
        __syncthreads();
        tk.maybe_compact(a.k, kMergeNT);
    }
    tk.finish(a.k);
    const int have = min(tk.cnt, a.k);
    for (int i = threadIdx.x; i < a.k; i += kMergeNT) {
        float dv;
        int64_t iv;
        if (i < have) {
            const uint64_t key = tk.buf[i];
            const float r = key_rank(key);
            dv = dist_of_rank(a.metric, r);
            iv = (int64_t)(uint32_t)key;
        } else {
            dv = a.metric == kL2 ? FLT_MAX : -FLT_MAX;
            iv = -1;
        }
        a.D[(size_t)q * a.k + i] = dv;
        a.I[(size_t)q * a.k + i] = iv;
    }
}

constexpr int kWaveEntries = 1024;  // a wave's row: at most 16 keys a lane,
constexpr int kWaveK = 256;         // and so many kept

// Of the wave's values v (~0u: none), counted from the highest bit that
// differs down, one count per bit: a limit with exactly kth values below it
// (true), or the kth smallest (1-based), when values equal to it lie on both
// sides.  Distinct values part after about log2 of their number of bits.
template <int SLOTS>
__device__ inline bool kth_of(const uint32_t (&v)[SLOTS], int kth, uint32_t& lim) {
    uint32_t all_or = 0, all_and = ~0u;
#pragma unroll
    for (int t = 0; t < SLOTS; ++t) {
        all_or |= v[t] != ~0u ? v[t] : 0u;
        all_and &= v[t];
    }
    for (int off = 32; off > 0; off >>= 1) {
        all_or |= __shfl_xor(all_or, off);
        all_and &= __shfl_xor(all_and, off);
    }
    const uint32_t diff = all_or ^ all_and;
    lim = all_and;
    if (diff == 0) return false;
    const int top = 31 - __builtin_clz(diff);
    uint32_t res = top < 31 ? all_and & ~((2u << top) - 1u) : 0u;
    for (int b = top; b >= 0; --b) {
        lim = res | (1u << b);
        int c = 0;
#pragma unroll
        for (int t = 0; t < SLOTS; ++t) c += __popcll(__ballot(v[t] < lim));
        if (c == kth) return true;
        if (c < kth) res = lim;
    }
    lim = res;
    return false;
}

// One wave per query, all its keys in registers (SLOTS x 64 >= parts x k_in).
// Bound by the counts and the sort of k keys, not by its bytes: 10,000 rows
// of 8 x 100 entries at k = 100 take 41 us (108 MB: 21 us at the rate of
// a copy) against 163 for the workgroup form, whose LDS top-k sorts all 800.
template <int SLOTS>
__global__ __launch_bounds__(kMergeNT) void merge_wave_kernel(MergeArgs a, uint32_t inv_k_in) {
    __shared__ __align__(16) uint64_t keys[kMergeNT / 64][kWaveK];
    const int lane = threadIdx.x & 63;
    uint64_t* kk = keys[threadIdx.x / 64];
    const int64_t q = (int64_t)blockIdx.x * (kMergeNT / 64) + threadIdx.x / 64;
    if (q >= a.n) return;  // whole wave; no workgroup barrier below
    const uint32_t total = (uint32_t)(a.parts * a.k_in);
    uint32_t rank[SLOTS], id[SLOTS];
    bool on[SLOTS];
    {
        int64_t iv[SLOTS];
        float dv[SLOTS];
#pragma unroll
        for (int t = 0; t < SLOTS; ++t) {
            const uint32_t e = min((uint32_t)(t * 64 + lane), total - 1);
            const uint32_t p = (e * inv_k_in) >> 20;  // e / k_in: both are at most 1024
            const size_t off = ((size_t)p * a.n + q) * a.k_in + (e - p * a.k_in);
            iv[t] = a.Ip[off];
            dv[t] = a.Dp[off];
        }
#pragma unroll
        for (int t = 0; t < SLOTS; ++t) {
            const float r = a.metric == kL2 ? dv[t] : -dv[t];
            // r < FLT_MAX: the heap's strict admission against its sentinel
            // (never inf or NaN)
            on[t] = (uint32_t)(t * 64 + lane) < total && iv[t] >= 0 && r < FLT_MAX;
            rank[t] = on[t] ? (uint32_t)(make_key(r, 0u) >> 32) : ~0u;
            id[t] = (uint32_t)iv[t];
        }
    }
    int have = 0;
#pragma unroll
    for (int t = 0; t < SLOTS; ++t) have += __popcll(__ballot(on[t]));
    const int keep = min(have, a.k);
    if (have > a.k) {  // leave exactly k keys on
        uint32_t lim;
        const bool apart = kth_of(rank, a.k, lim);
        if (apart) {
#pragma unroll
            for (int t = 0; t < SLOTS; ++t) on[t] = rank[t] < lim;
        } else {  // the k-th distance is lim: of the rows at it, those of the smallest ids
            uint32_t tie[SLOTS];
            int room = a.k;
#pragma unroll
            for (int t = 0; t < SLOTS; ++t) {
                on[t] = rank[t] < lim;
                tie[t] = rank[t] == lim ? id[t] : ~0u;
                room -= __popcll(__ballot(on[t]));
            }
            uint32_t ki;
            const bool split = kth_of(tie, room, ki);
#pragma unroll
            for (int t = 0; t < SLOTS; ++t) {
                const bool less = tie[t] < ki;
                on[t] = on[t] || less;
                room -= __popcll(__ballot(less));
            }
            if (!split) {  // equal entries: any of them
#pragma unroll
                for (int t = 0; t < SLOTS; ++t) {
                    const bool same = tie[t] == ki;
                    const uint64_t mk = __ballot(same);
                    on[t] = on[t] || (same && (int)lanes_below(mk) < room);
                    room = max(0, room - (int)__popcll(mk));
                }
            }
        }
    }
    uint32_t pos = 0;
#pragma unroll
    for (int t = 0; t < SLOTS; ++t) {
        const uint64_t mk = __ballot(on[t]);
        if (on[t]) kk[pos + lanes_below(mk)] = (uint64_t)rank[t] << 32 | id[t];
        pos += (uint32_t)__popcll(mk);
    }
    uint32_t n2 = 64;
    while (n2 < (uint32_t)keep) n2 <<= 1;
    for (uint32_t i = (uint32_t)keep + lane; i < n2; i += 64) kk[i] = ~0ull;
    __builtin_amdgcn_wave_barrier();
    wave_sort(kk, n2, lane);
    for (int i = lane; i < a.k; i += 64) {
        const bool ok = i < keep;
        a.D[(size_t)q * a.k + i] = ok ? dist_of_rank(a.metric, key_rank(kk[i])) : a.metric == kL2 ? FLT_MAX : -FLT_MAX;
        a.I[(size_t)q * a.k + i] = ok ? (int64_t)(uint32_t)kk[i] : -1;
    }
}

int check_merge(int metric, int64_t n, int64_t parts, int64_t k_in, int64_t k) {
    if (metric != HIVF_METRIC_L2 && metric != HIVF_METRIC_IP) return HIVF_EINVAL;
    if (n < 0 || parts < 1 || k_in < 1 || k < 1) return HIVF_EINVAL;
    if (k > kMaxK) return HIVF_EUNSUPPORTED;
    if (n > INT32_MAX || parts * k_in > INT32_MAX) return HIVF_EUNSUPPORTED;
    return HIVF_OK;
}

hipError_t launch_merge(int metric, int64_t n, int64_t parts, int64_t k_in, const float* Dp, const int64_t* Ip,
                        int64_t k, float* D, int64_t* I, hipStream_t s) {
    if (n == 0) return hipSuccess;
    MergeArgs a{Dp, Ip, n, (int)parts, (int)k_in, (int)k, metric, D, I};
    const int64_t total = parts * k_in;
    if (total <= kWaveEntries && k <= kWaveK) {
        const uint32_t inv = (uint32_t)((1 << 20) + k_in - 1) / (uint32_t)k_in;
        const dim3 grid((unsigned)((n + kMergeNT / 64 - 1) / (kMergeNT / 64)));
        if (total <= 256)
            hipLaunchKernelGGL(merge_wave_kernel<4>, grid, dim3(kMergeNT), 0, s, a, inv);
        else if (total <= 512)
            hipLaunchKernelGGL(merge_wave_kernel<8>, grid, dim3(kMergeNT), 0, s, a, inv);
        else
            hipLaunchKernelGGL(merge_wave_kernel<16>, grid, dim3(kMergeNT), 0, s, a, inv);
    } else {
        hipLaunchKernelGGL(merge_kernel, dim3((unsigned)n), dim3(kMergeNT), 0, s, a);
    }
    return hipGetLastError();
}

}  // namespace
}  // namespace hivf

using namespace hivf;

extern "C" {

int hivf_merge_topk_device(int metric, int64_t n, int64_t parts, int64_t k_in, const float* D_parts,
                           const int64_t* I_parts, int64_t k, float* D, int64_t* I, void* stream) {
    HIVF_API_BEGIN
    int rc = check_merge(metric, n, parts, k_in, k);
    if (rc) {
        set_global_error("hivf_merge_topk_device: bad metric, n, parts, k_in or k (k <= 1024)");
        return rc;
    }
    if (n == 0) return HIVF_OK;
    if (!D_parts || !I_parts || !D || !I) {
        set_global_error("hivf_merge_topk_device: null buffer");
        return HIVF_EINVAL;
    }
    hipError_t e = launch_merge(metric, n, parts, k_in, D_parts, I_parts, k, D, I, static_cast<hipStream_t>(stream));
    if (e != hipSuccess) {
        set_global_error(std::string("hivf_merge_topk_device: ") + hipGetErrorString(e));
        return HIVF_EHIP;
    }
    return HIVF_OK;
    HIVF_API_END(nullptr)
}

int hivf_merge_topk(int metric, int64_t n, int64_t parts, int64_t k_in, const float* D_parts,
                    const int64_t* I_parts, int64_t k, float* D, int64_t* I) {
    HIVF_API_BEGIN
    int rc = check_merge(metric, n, parts, k_in, k);
    if (rc) {
        set_global_error("hivf_merge_topk: bad metric, n, parts, k_in or k (k <= 1024)");
        return rc;
    }
    if (n == 0) return HIVF_OK;
    if (!D_parts || !I_parts || !D || !I) {
        set_global_error("hivf_merge_topk: null buffer");
        return HIVF_EINVAL;
    }
    const size_t in_el = (size_t)parts * n * k_in, out_el = (size_t)n * k;
    for (size_t i = 0; i < in_el; ++i)
        if (I_parts[i] >= (int64_t)kNoId) {
            set_global_error("hivf_merge_topk: ids must be below 2^32 - 1");
            return HIVF_EUNSUPPORTED;
        }
    DevBuf<float> dp, d;
    DevBuf<int64_t> ip, i;
    hipStream_t s = nullptr;
    hipError_t e = hipStreamCreateWithFlags(&s, hipStreamNonBlocking);
    if (e == hipSuccess) e = dp.ensure(in_el);
    if (e == hipSuccess) e = ip.ensure(in_el);
    if (e == hipSuccess) e = d.ensure(out_el);
    if (e == hipSuccess) e = i.ensure(out_el);
    if (e == hipSuccess) e = hipMemcpyAsync(dp.p, D_parts, in_el * sizeof(float), hipMemcpyHostToDevice, s);
    if (e == hipSuccess) e = hipMemcpyAsync(ip.p, I_parts, in_el * sizeof(int64_t), hipMemcpyHostToDevice, s);
    if (e == hipSuccess) e = launch_merge(metric, n, parts, k_in, dp.p, ip.p, k, d.p, i.p, s);
    if (e == hipSuccess) e = hipMemcpyAsync(D, d.p, out_el * sizeof(float), hipMemcpyDeviceToHost, s);
    if (e == hipSuccess) e = hipMemcpyAsync(I, i.p, out_el * sizeof(int64_t), hipMemcpyDeviceToHost, s);
    if (e == hipSuccess) e = hipStreamSynchronize(s);
    if (s) (void)hipStreamDestroy(s);
    if (e != hipSuccess) {
        set_global_error(std::string("hivf_merge_topk: ") + hipGetErrorString(e));
        return e == hipErrorOutOfMemory ? HIVF_ENOMEM : HIVF_EHIP;
    }
    return HIVF_OK;
    HIVF_API_END(nullptr)
}

}  // extern "C"
