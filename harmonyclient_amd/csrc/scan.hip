// Per-query kernels of the IVF-Flat query path on CDNA4:
//   coarse_kernel : query x centroid distances + top-nprobe
//                   (src/Index.cpp:967-995, src/IVFScan.hpp:108-138)
//   scan_kernel   : inverted-list scan with top-k, three modes
//       plain   : full distances (src/Index.cpp:1420-1554,
//                 src/IVFScan.hpp:247-272)
//       pruned  : dimension-block partial distances, a row is dropped once
//                 its running distance exceeds min(tau_q, running k-th)
//                 (src/node.cpp:606-678, 1056-1174)
//       warm-up : k-th distance over the first W rows of the first L probed
//                 lists (src/Index.cpp:999-1051)
//
// One workgroup of 256 threads per query.  Each wavefront owns one tile of
// 64 list rows per round, one row per lane, and streams it with coalesced
// 1 KiB loads (tile layout in kernels.hpp); the query sits in LDS and is
// read with broadcast loads.  A distance is one sequential FMA chain over
// the dims, the same arithmetic as the oracle, so results are bit-identical.
#include <algorithm>
#include <type_traits>

#include "common.hpp"
#include "kernels.hpp"
#include "select.hpp"

namespace hivf {

namespace {

constexpr int kNT = 256;
constexpr int kNW = kNT / kWave;
constexpr int kBuf = 2048;


__device__ inline void load_query(float4* qs, const float4* q, int nquad) {
    for (int j = threadIdx.x; j < nquad; j += kNT) qs[j] = q[j];
}

__device__ inline float quad_comp(float4 v, int c) {
    return c == 0 ? v.x : c == 1 ? v.y : c == 2 ? v.z : v.w;
}

// Quads [j, je) of the canonical chain of one row, 8 loads in flight.  (Loaded
// into registers first, and fenced: from an unrolled loop of load and FMA the
// compiler waits for each load in some inlined copies.  The rescan of 1988 listed
// queries, 32 lists of 488 rows x 128 dims each: 1.97 ms so, 1.25 now.)  The last 1 to
// 7 quads likewise, four and up to three (the last one's address again where there
// are fewer), not each after the other: 200 queries of 4 lists of 1500 rows, 60 dims,
// plain 137 us and pruned 138, now 108 and 124; pruned blocks of 24 dims, 96 dims 158
// and 122.
template <int METRIC>
__device__ inline float accum_quads(float acc, const float4* qs, const float4* tp, int j, int je) {
    for (; j + 8 <= je; j += 8) {
        float4 x[8];
#pragma unroll
        for (int u = 0; u < 8; ++u) x[u] = tp[(size_t)(j + u) * kWave];
        __builtin_amdgcn_sched_barrier(0x104);  // (scalar operations and LDS reads may cross)
#pragma unroll
        for (int u = 0; u < 8; ++u) acc = accum<METRIC>(acc, qs[j + u], x[u]);
    }
    if (j + 4 <= je) {
        float4 x[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) x[u] = tp[(size_t)(j + u) * kWave];
        __builtin_amdgcn_sched_barrier(0x104);
#pragma unroll
        for (int u = 0; u < 4; ++u) acc = accum<METRIC>(acc, qs[j + u], x[u]);
        j += 4;
    }
    if (j < je) {
        float4 x[3];
#pragma unroll
        for (int u = 0; u < 3; ++u) x[u] = tp[(size_t)min(j + u, je - 1) * kWave];
        __builtin_amdgcn_sched_barrier(0x104);
#pragma unroll
        for (int u = 0; u < 3; ++u)
            if (j + u < je) acc = accum<METRIC>(acc, qs[j + u], x[u]);
    }
    return acc;
}

// Dims [d0, d1) of the canonical chain of one row: a partial first quad,
// whole quads, a partial last quad (the partial steps only where a block
// boundary falls inside a quad).
template <int METRIC>
__device__ inline float accum_dims(float acc, const float4* qs, const float4* tp, int d0, int d1) {
    int j = d0 >> 2;
    const int c0 = d0 & 3;
    if (c0) {
        const float4 q = qs[j], x = tp[(size_t)j * kWave];
        const int c1 = min(4, d1 - 4 * j);
        for (int c = c0; c < c1; ++c) {
            const float qv = quad_comp(q, c), xv = quad_comp(x, c);
            if constexpr (METRIC == kL2) {
                const float t = qv - xv;
                acc = __builtin_fmaf(t, t, acc);
            } else {
                acc = __builtin_fmaf(qv, xv, acc);
            }
        }
        ++j;
    }
    const int jend = d1 >> 2;
    if (j < jend) {
        acc = accum_quads<METRIC>(acc, qs, tp, j, jend);
        j = jend;
    }
    const int r = d1 & 3;
    if (r && 4 * j >= d0 && 4 * j < d1) {
        const float4 q = qs[j], x = tp[(size_t)j * kWave];
        for (int c = 0; c < r; ++c) {
            const float qv = quad_comp(q, c), xv = quad_comp(x, c);
            if constexpr (METRIC == kL2) {
                const float t = qv - xv;
                acc = __builtin_fmaf(t, t, acc);
            } else {
                acc = __builtin_fmaf(qv, xv, acc);
            }
        }
    }
    return acc;
}

// The probes' lists, kProbeChunk at a time, staged in LDS: first arena tile,
// rows (capped at row_limit) and tiles before each.
constexpr int kProbeChunk = kNT;
struct ProbeMap {
    int tile0[kProbeChunk];
    int rows[kProbeChunk];
    int before[kProbeChunk + 1];
    int wsum[kNW];
};

// Stages probes [j0, j0 + m) (m <= kProbeChunk); all threads, ends with a
// barrier.  Their tiles number pm.before[m].
__device__ inline void stage_probes(const ScanArgs& a, const int32_t* probes, int j0, int m, ProbeMap& pm) {
    const int tid = threadIdx.x, lane = tid % kWave, wave = tid / kWave;
    int rows = 0, tile0 = 0;
    if (tid < m) {
        const int l = probes[j0 + tid];
        if (l >= 0) {
            rows = min(a.lists.list_size[l], a.row_limit);
            tile0 = a.lists.list_tile_off[l];
        }
    }
    const int nt = (rows + kTileRows - 1) / kTileRows;
    int incl = nt;
    for (int off = 1; off < kWave; off <<= 1) {
        const int v = __shfl_up(incl, off);
        if (lane >= off) incl += v;
    }
    if (lane == kWave - 1) pm.wsum[wave] = incl;
    pm.tile0[tid] = tile0;
    pm.rows[tid] = rows;
    __syncthreads();
    int base = 0;
    for (int w = 0; w < wave; ++w) base += pm.wsum[w];
    pm.before[tid + 1] = base + incl;
    if (tid == 0) pm.before[0] = 0;
    __syncthreads();
}

// The kth smallest (1-based) of n <= 64 kSlots keys' ranks, by one wave: the keys
// stay in registers and the rank's bits are fixed from the highest that
// differs down, one count per bit.  (A bitonic sort of the 1000-odd rows of a
// warm-up scan is 55 stages with a barrier each.)
template <int kSlots>
__device__ inline uint32_t wave_kth_rank(const uint64_t* keys, int n, int kth, int lane) {
    uint32_t v[kSlots];
    uint32_t all_or = 0, all_and = ~0u;
#pragma unroll
    for (int t = 0; t < kSlots; ++t) {
        const int i = t * kWave + lane;
        v[t] = i < n ? (uint32_t)(keys[i] >> 32) : ~0u;
        if (i < n) {
            all_or |= v[t];
            all_and &= v[t];
        }
    }
    for (int off = 32; off > 0; off >>= 1) {
        all_or |= __shfl_xor(all_or, off);
        all_and &= __shfl_xor(all_and, off);
    }
    const uint32_t diff = all_or ^ all_and;
    // res: the bits fixed so far (those above the highest difference are common)
    const int top = diff ? 31 - __builtin_clz(diff) : -1;
    uint32_t res = top < 31 ? all_and & ~((2u << max(top, 0)) - 1u) : 0u;
    if (top < 0) return all_and;
    for (int b = top; b >= 0; --b) {
        const uint32_t test = res | (1u << b);  // ranks below it: the b-th bit clear under the prefix, or smaller
        int c = 0;
#pragma unroll
        for (int t = 0; t < kSlots; ++t) c += __popcll(__ballot(v[t] < test));
        if (c < kth) res = test;
    }
    return res;
}

// Tiles a wave takes between two barriers of the workgroup: the top-k's
// buffer holds k <= 1024 kept keys and 4 x 256 more.  (The pruned scan takes
// one: its bound follows the running k-th.)
// Past k = 512, two: with four the kept keys leave no room for a second round,
// and the buffer is sorted after nearly every one (64 queries of 32 lists, k =
// 1000, four, two and one: 635, 397 and 379 us; the warm-up of 10 lists 322, 260
// and 278; k = 512: 316, 325 and 342).
constexpr int kRoundTiles = 4;
static_assert(kMaxK + kRoundTiles * kNT <= kBuf, "a round's keys fit beside the kept ones");

// One query, by the whole workgroup.  The probes' sizes come from LDS (a chain
// of two dependent loads per list otherwise), a warm-up scan ends in a bit
// search for its k-th rank instead of a sort: warm-up of 2000 queries over 10
// lists x 100 rows of 128 dims 103 -> 65 us, of 4096 on skewed lists 221 -> 172, of
// 2000 with 420 dims 190 -> 163 (the rows come from L2 at 17 to 21 TB/s).  More
// than 8 row loads in flight per wave is slower (16: 305 us at 420 dims).
//
// With nparts > 1 the workgroup takes every nparts-th round of the query's
// tiles (each part starts at the near lists, so its running k-th is as tight
// as one workgroup's after the same number of rounds) and leaves its top k in
// slot's part of part_keys; the last part to end merges them.
template <int MODE, int METRIC>
__device__ void scan_one(const ScanArgs& a, const int qi, const int part = 0, const int nparts = 1,
                         const uint32_t slot = 0) {
    __shared__ LdsTopK<kNT, kBuf> top;
    __shared__ ProbeMap pm;
    __shared__ unsigned long long s_stats[3];
    extern __shared__ float4 qs[];

    const int tid = threadIdx.x;
    const int wave = tid / kWave;
    const int lane = tid % kWave;
    const int nquad = a.lists.nquad;
    const int32_t* probes = a.probes + (size_t)qi * a.probe_stride;
    int P = a.nprobe_q ? a.nprobe_q[qi] : a.nprobe;
    if (P > a.probe_stride) P = a.probe_stride;
    if (MODE == kScanWarmup && P > a.warm_lists) P = a.warm_lists;  // src/Index.cpp:1008-1011

    top.init();
    if (tid == 0) s_stats[0] = s_stats[1] = s_stats[2] = 0;
    load_query(qs, a.q + (size_t)qi * nquad, nquad);

    const float tau_q = (MODE == kScanPruned && a.tau) ? a.tau[qi] : FLT_MAX;
    const int nblocks = MODE == kScanPruned ? a.nblocks : 1;
    unsigned long long my_cand = 0, my_skip = 0;
    uint64_t thr = top.thr;

    const int round = MODE == kScanPruned ? 1 : a.k <= kBuf / 4 ? kRoundTiles : 2;
    for (int j0 = 0; j0 < P; j0 += kProbeChunk) {
        stage_probes(a, probes, j0, min(kProbeChunk, P - j0), pm);
        const int m = min(kProbeChunk, P - j0);
        const int total = pm.before[m];
        int j = 0;  // this wave's probe: before[j] <= its tile < before[j + 1]
        for (int g0 = part * kNW * round; g0 < total; g0 += nparts * kNW * round) {
            for (int u = 0; u < round; ++u) {
                const int g = g0 + u * kNW + wave;
                if (g >= total) break;
                while (pm.before[j + 1] <= g) ++j;
                const int t = __builtin_amdgcn_readfirstlane(g - pm.before[j]);
                const int tile = __builtin_amdgcn_readfirstlane(pm.tile0[j]) + t;
                const bool valid = lane < pm.rows[j] - t * kTileRows;
                const float4* tp = a.lists.codes + (size_t)tile * nquad * kWave + lane;
                const uint32_t id = a.lists.ids[(size_t)tile * kWave + lane];
                float acc = 0.0f;
                bool keep = valid;
                if constexpr (MODE == kScanPruned) {
                    const float bound = fminf(tau_q, key_rank(thr));
                    for (int b = 0; b < nblocks; ++b) {
                        if (__ballot(keep) == 0) break;
                        if (keep) {
                            const int d0 = b * a.block_dims;
                            const int d1 = b < nblocks - 1 ? d0 + a.block_dims : 4 * nquad;
                            acc = accum_dims<METRIC>(acc, qs, tp, d0, d1);
                            if (b < nblocks - 1 && acc > bound) {
                                keep = false;
                                my_skip += nblocks - 1 - b;
                            }
                        }
                    }
                } else {
                    if (valid) acc = accum_quads<METRIC>(acc, qs, tp, 0, nquad);
                }
                if (valid) my_cand++;
                if (keep) top.offer(make_key(rank_of<METRIC>(acc), id), thr);
            }
            __syncthreads();
            top.maybe_compact(a.k, kNT * round);
            thr = top.thr;
        }
        __syncthreads();  // the map's last reads are done
    }

    if (a.stats) {
        if (my_cand) atomicAdd(&s_stats[0], my_cand);
        if (my_skip) atomicAdd(&s_stats[2], my_skip);
        __syncthreads();
        if (tid == 0) {
            atomicAdd(&a.stats[0], s_stats[0]);
            atomicAdd(&a.stats[1], s_stats[0] * (unsigned long long)nblocks);
            atomicAdd(&a.stats[2], s_stats[2]);
        }
    }

    if constexpr (MODE == kScanWarmup) {
        // only the k-th rank is wanted, of the keys kept so far
        if (top.cnt > 1024) top.finish(a.k);
        if (wave == 0) {
            const int cnt = top.cnt;
            float v = sentinel<METRIC>();
            // (16 slots' counts per bit are longer than the sort was where the rows are
            // few: a pruned query of one list of 16 x 128 rows 38.6 us, 36.0 with the
            // sort, now 34.5)
            if (cnt >= a.k)
                v = dist_of_rank(METRIC, ord2f(cnt <= 64 ? wave_kth_rank<1>(top.buf, cnt, a.k, lane)
                                               : cnt <= 256 ? wave_kth_rank<4>(top.buf, cnt, a.k, lane)
                                                            : wave_kth_rank<16>(top.buf, cnt, a.k, lane)));
            if (lane == 0) a.out_tau[qi] = v;
        }
    } else {
        top.finish(a.k);
        if (nparts > 1) {
            __shared__ uint32_t s_before;
            uint64_t* mine = a.part_keys + ((size_t)slot * nparts + part) * a.k;
            for (int i = tid; i < a.k; i += kNT) mine[i] = i < top.cnt ? top.buf[i] : ~0ull;
            __threadfence();
            __syncthreads();
            if (tid == 0) s_before = atomicAdd(&a.part_cnt[slot], 1u);
            __syncthreads();
            if (s_before + 1 != (uint32_t)nparts) return;
            __threadfence();
            top.init();
            thr = top.thr;
            const uint64_t* all = a.part_keys + (size_t)slot * nparts * a.k;
            const int nk = nparts * a.k;
            for (int i0 = 0; i0 < nk; i0 += kRoundTiles * kNT) {
                uint64_t key[kRoundTiles];
#pragma unroll
                for (int u = 0; u < kRoundTiles; ++u) {
                    const int i = i0 + u * kNT + tid;
                    key[u] = i < nk ? all[i] : ~0ull;
                }
#pragma unroll
                for (int u = 0; u < kRoundTiles; ++u) top.offer(key[u], thr);
                __syncthreads();
                top.maybe_compact(a.k, kRoundTiles * kNT);
                thr = top.thr;
            }
            top.finish(a.k);
        }
        const int cnt = top.cnt;
        for (int i = tid; i < a.k; i += kNT) {
            float dv = sentinel<METRIC>();
            int64_t iv = -1;
            if (i < cnt) {
                uint64_t key = top.buf[i];
                float rk = key_rank(key);
                dv = dist_of_rank(METRIC, rk);
                iv = (int64_t)(uint32_t)key;
            }
            a.out_d[(size_t)qi * a.k + i] = dv;
            a.out_i[(size_t)qi * a.k + i] = iv;
        }
    }
}

// One workgroup per query, or (LIST) a grid that walks the query list.  A list
// too short for the grid has its queries split: one query's 62k rows of 128 dims
// on one workgroup hold a search for 0.9 ms, 43 such queries for 1.9 ms, against
// 0.42 ms split.  (A kernel of its own with one call of scan_one: with several
// in one kernel the compiler waited for each row load of some of them.)
template <int MODE, int METRIC, bool LIST>
__global__ __launch_bounds__(kNT) void scan_kernel(ScanArgs a) {
    if constexpr (!LIST) {
        scan_one<MODE, METRIC>(a, blockIdx.x);
    } else {
        const uint32_t nl = *a.qcount;
        const uint32_t np = MODE != kScanWarmup && a.part_keys && nl ? max(1u, min(gridDim.x / nl, (uint32_t)kListParts)) : 1u;
        // (of a split list each workgroup takes one query: the step ends the loop)
        for (uint32_t i = blockIdx.x / np; i < nl; i += gridDim.x) {
            __syncthreads();  // the previous query's LDS reads are done
            scan_one<MODE, METRIC>(a, __builtin_amdgcn_readfirstlane(a.qlist[i]), (int)(blockIdx.x % np), (int)np, i);
        }
    }
}

template <int METRIC>
__device__ void coarse_one(const CoarseArgs& a, const int qi) {
    __shared__ LdsTopK<kNT, kBuf> top;
    extern __shared__ float4 qs[];
    const int tid = threadIdx.x;
    const int wave = tid / kWave;
    const int lane = tid % kWave;
    top.init();
    load_query(qs, a.q + (size_t)qi * a.nquad, a.nquad);
    __syncthreads();
    const int tiles = (a.nlist + kTileRows - 1) / kTileRows;
    const int rounds = (tiles + kNW - 1) / kNW;
    uint64_t thr = top.thr;
    for (int r = 0; r < rounds; ++r) {
        const int tile = r * kNW + wave;
        const int c = tile * kTileRows + lane;
        if (tile < tiles && c < a.nlist) {
            const float4* tp = a.cent + (size_t)tile * a.nquad * kWave + lane;
            float acc = 0.0f;
#pragma unroll 8
            for (int jj = 0; jj < a.nquad; ++jj)
                acc = accum<METRIC>(acc, qs[jj], tp[(size_t)jj * kWave]);
            top.offer(make_key(rank_of<METRIC>(acc), (uint32_t)c), thr);
        }
        __syncthreads();
        top.maybe_compact(a.P, kNT);
        thr = top.thr;
    }
    top.finish(a.P);
    const int cnt = top.cnt;
    for (int i = tid; i < a.P; i += kNT) {
        float dv = sentinel<METRIC>();
        int32_t lv = -1;
        if (i < cnt) {
            uint64_t key = top.buf[i];
            float rk = key_rank(key);
            dv = dist_of_rank(METRIC, rk);
            lv = (int32_t)(uint32_t)key;
        }
        a.out_d[(size_t)qi * a.P + i] = dv;
        a.out_l[(size_t)qi * a.P + i] = lv;
    }
}

// One workgroup per query, or, with a query list, a grid that walks the list.
template <int METRIC>
__global__ __launch_bounds__(kNT) void coarse_kernel(CoarseArgs a) {
    if (a.qlist) {
        const uint32_t nl = *a.qcount;
        for (uint32_t i = blockIdx.x; i < nl; i += gridDim.x) {
            __syncthreads();  // the previous query's LDS reads are done
            coarse_one<METRIC>(a, a.qlist[i]);
        }
        return;
    }
    coarse_one<METRIC>(a, blockIdx.x);
}

template <int MODE>
hipError_t launch_scan_mode(const ScanArgs& a, int metric, hipStream_t s) {
    size_t lds = (size_t)a.lists.nquad * sizeof(float4);
    // (a list of few queries gets workgroups to split them over)
    const int64_t want = a.part_keys ? (int64_t)a.nq * 16 : a.nq;
    const dim3 grid((unsigned)(a.qlist ? std::min<int64_t>(want, kListGrid) : a.nq));
    auto go = [&](auto list) {
        constexpr bool L = decltype(list)::value;
        if (metric == kL2)
            hipLaunchKernelGGL((scan_kernel<MODE, kL2, L>), grid, dim3(kNT), lds, s, a);
        else
            hipLaunchKernelGGL((scan_kernel<MODE, kIP, L>), grid, dim3(kNT), lds, s, a);
    };
    if (a.qlist)
        go(std::true_type{});
    else
        go(std::false_type{});
    return hipGetLastError();
}

}  // namespace

hipError_t launch_scan(const ScanArgs& a, int mode, int metric, hipStream_t s) {
    if (a.nq <= 0) return hipSuccess;
    switch (mode) {
        case kScanPlain: return launch_scan_mode<kScanPlain>(a, metric, s);
        case kScanPruned: return launch_scan_mode<kScanPruned>(a, metric, s);
        default: return launch_scan_mode<kScanWarmup>(a, metric, s);
    }
}

hipError_t launch_coarse(const CoarseArgs& a, int metric, hipStream_t s) {
    if (a.nq <= 0) return hipSuccess;
    size_t lds = (size_t)a.nquad * sizeof(float4);
    const dim3 grid((unsigned)(a.qlist ? std::min(a.nq, kListGrid) : a.nq));
    if (metric == kL2)
        hipLaunchKernelGGL((coarse_kernel<kL2>), grid, dim3(kNT), lds, s, a);
    else
        hipLaunchKernelGGL((coarse_kernel<kIP>), grid, dim3(kNT), lds, s, a);
    return hipGetLastError();
}

}  // namespace hivf
