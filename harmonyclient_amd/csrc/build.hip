// Index build on the GPU: the Lloyd update of k-means and the list fill of
// Index::add.
//
//   k-means (src/Clustering.cpp:93-152, src/Index.cpp:381-425): every round
//     assigns each training row to its nearest centroid (the coarse kernel
//     with one probe, lowest id on exact ties), groups the rows by centroid
//     in row order, and sets each centroid to the mean of its rows,
//     accumulated in FP64 in row order and rounded once to FP32 (a centroid
//     without rows keeps its value).  The fixed order makes the result
//     independent of scheduling, unlike the reference's `omp critical`
//     accumulation.
//   add (src/Index.cpp:581-698): assigns every row, orders each list by
//     distance to its centroid (ascending for L2, descending for IP; equal
//     distances by row id -- the canonical form of the reference's unstable
//     std::sort, src/Index.cpp:643-651), and writes the tiled list arena,
//     the ids and the FP64-accumulated squared norms.
//
// Grouping and ordering are stable least-significant-digit radix passes of
// 8 bits: each pass counts digits per 1024-element chunk (one wave per
// chunk, an LDS histogram), scans the counts of every digit over the chunks,
// and places each element at its digit's base + its chunk's offset + its
// rank among the chunk's earlier elements with the same digit.  Elements
// start in row order, so every pass keeps equal keys in row order.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <climits>
#include <cmath>
#include <cstring>
#include <vector>

#include "index_impl.hpp"
#include "wave.hpp"

namespace hivf {

namespace {

constexpr int kChunk = 1024;  // elements per chunk of a radix pass
constexpr int kDigits = 256;  // 8-bit digits

// Digit counts of every chunk: counts[digit * nchunks + chunk].
__global__ __launch_bounds__(64) void rp_count_kernel(const uint32_t* __restrict__ key,
                                                      const int32_t* __restrict__ perm_in, int shift, int64_t n,
                                                      int nchunks, uint32_t* __restrict__ counts) {
    __shared__ uint32_t hist[kDigits];
    const int c = blockIdx.x, lane = threadIdx.x;
    for (int b = lane; b < kDigits; b += 64) hist[b] = 0;
    __syncthreads();
    const int64_t i0 = (int64_t)c * kChunk;
    const int64_t i1 = std::min<int64_t>(n, i0 + kChunk);
    // (every load in flight together; positions past the end count nothing)
    int32_t el[kChunk / 64];
    uint32_t kv[kChunk / 64];
#pragma unroll
    for (int t = 0; t < kChunk / 64; ++t) {
        const int64_t i = std::min<int64_t>(i0 + t * 64 + lane, n - 1);
        el[t] = perm_in ? perm_in[i] : (int32_t)i;
    }
#pragma unroll
    for (int t = 0; t < kChunk / 64; ++t) kv[t] = key[el[t]];
#pragma unroll
    for (int t = 0; t < kChunk / 64; ++t)
        if (i0 + t * 64 + lane < i1) atomicAdd(&hist[(kv[t] >> shift) & (kDigits - 1)], 1u);
    __syncthreads();
    for (int b = lane; b < kDigits; b += 64) counts[(size_t)b * nchunks + c] = hist[b];
}

// Per digit (one workgroup each): exclusive scan of its chunk counts, in
// place, and the digit's total.
__global__ __launch_bounds__(256) void rp_scan_kernel(uint32_t* __restrict__ counts, int nchunks,
                                                      uint32_t* __restrict__ total) {
    __shared__ uint32_t part[256];
    uint32_t* col = counts + (size_t)blockIdx.x * nchunks;
    const int t = threadIdx.x;
    const int per = (nchunks + 255) / 256;
    const int c0 = t * per, c1 = std::min(nchunks, c0 + per);
    uint32_t s = 0;
    for (int c = c0; c < c1; ++c) s += col[c];
    part[t] = s;
    __syncthreads();
    if (t == 0) {
        uint32_t run = 0;
        for (int i = 0; i < 256; ++i) {
            const uint32_t v = part[i];
            part[i] = run;
            run += v;
        }
        total[blockIdx.x] = run;
    }
    __syncthreads();
    uint32_t run = part[t];
    for (int c = c0; c < c1; ++c) {
        const uint32_t v = col[c];
        col[c] = run;
        run += v;
    }
}

// Stable placement: one wave per chunk walks its elements 64 at a time in
// order; lanes with equal digits take consecutive positions by lane.  What
// bounded it was latency, not bytes: the digits' starts were summed by one
// lane (512 dependent loads, 100 us of the 140 a pass over 500k keys took), and
// the lanes of a digit were matched one digit at a time.  Now each lane loads
// four digits' counts and totals and a wave scan gives the starts, the keys of
// all 1024 elements are loaded together, and eight
// ballots (one per digit bit) give every lane its digit's lanes at once: 9.6 us
// per pass over 500k keys (12 of them in an add and its first search).
__global__ __launch_bounds__(64) void rp_fill_kernel(const uint32_t* __restrict__ key,
                                                     const int32_t* __restrict__ perm_in, int shift, int64_t n,
                                                     int nchunks, const uint32_t* __restrict__ counts,
                                                     const uint32_t* __restrict__ total,
                                                     int32_t* __restrict__ perm_out) {
    constexpr int kSteps = kChunk / 64;
    __shared__ uint32_t next[kDigits];
    const int c = blockIdx.x, lane = threadIdx.x;
    const int64_t i0 = (int64_t)c * kChunk;
    const int64_t i1 = std::min<int64_t>(n, i0 + kChunk);
    // this chunk's elements and digits, every load in flight together
    // (positions past the end read the last element and place nothing)
    int32_t el[kSteps];
    uint32_t kv[kSteps];
#pragma unroll
    for (int t = 0; t < kSteps; ++t) {
        const int64_t i = std::min<int64_t>(i0 + t * 64 + lane, n - 1);
        el[t] = perm_in ? perm_in[i] : (int32_t)i;
    }
    {
        uint32_t cnt[4], tot[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            cnt[u] = counts[(size_t)(lane * 4 + u) * nchunks + c];
            tot[u] = total[lane * 4 + u];
        }
#pragma unroll
        for (int t = 0; t < kSteps; ++t) kv[t] = key[el[t]];
        uint32_t run = wave_incl_scan(tot[0] + tot[1] + tot[2] + tot[3], lane) - (tot[0] + tot[1] + tot[2] + tot[3]);
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            next[lane * 4 + u] = run + cnt[u];
            run += tot[u];
        }
    }
    __builtin_amdgcn_wave_barrier();
#pragma unroll
    for (int t = 0; t < kSteps; ++t) {
        if (i0 + t * 64 >= i1) break;
        const bool valid = i0 + t * 64 + lane < i1;
        const uint32_t dg = (kv[t] >> shift) & (kDigits - 1);
        uint64_t same = __ballot(valid);
#pragma unroll
        for (int b = 0; b < 8; ++b) {
            const bool bit = (dg >> b) & 1u;
            const uint64_t m = __ballot(bit);
            same &= bit ? m : ~m;
        }
        const uint32_t start = next[dg];
        __builtin_amdgcn_wave_barrier();  // (one wave: its LDS operations stay in order)
        if (valid) {
            perm_out[start + lanes_below(same)] = el[t];
            // the digit's last lane moves its start past these
            if ((same >> lane) == 1ull) next[dg] = start + (uint32_t)__popcll(same);
        }
        __builtin_amdgcn_wave_barrier();
    }
}

// Sort key of a row's distance to its centroid: ascending for L2,
// descending for IP; -0 and +0 equal.
__global__ void dist_key_kernel(const float* __restrict__ dist, int64_t n, int l2, uint32_t* __restrict__ key) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const uint32_t o = f2ord(dist[i]);
    key[i] = l2 ? o : ~o;
}

// Sort key of a row's label: the label, or nlist for a row the assignment
// left without a centroid (non-finite values), which then sorts after every
// list.
__global__ void label_key_kernel(const int32_t* __restrict__ label, int64_t n, int nlist,
                                 uint32_t* __restrict__ key) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const int32_t l = label[i];
    key[i] = (l >= 0 && l < nlist) ? (uint32_t)l : (uint32_t)nlist;
}

// off[l] (l = 0 .. nlist) = the first position of the sorted rows whose label
// is l or more: every position where the label changes writes the labels it
// passes.  (Counting rows per label with global atomics took 0.1 to 1.5 ms,
// most when neighbouring rows share a label; this reads each label once.)
__global__ void label_off_kernel(const uint32_t* __restrict__ key, const int32_t* __restrict__ order, int64_t n,
                                 int nlist, int64_t* __restrict__ off) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i > n) return;
    const int64_t a = i == 0 ? -1 : (int64_t)key[order[i - 1]];
    const int64_t b = i == n ? (int64_t)nlist : (int64_t)key[order[i]];
    for (int64_t l = a + 1; l <= b; ++l) off[l] = i;
}

__global__ void zero_u32_kernel(uint32_t* p, int64_t n) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) p[i] = 0u;
}

// FP64 sums of a centroid's rows (members in row order) per dimension, then
// the mean rounded to FP32.  One 64-thread workgroup per centroid and 64
// dims, a thread per dim.  The additions stay in row order (the result does
// not depend on the schedule), so a long list is a serial chain; what bounded
// it was a load waited for per row, then per 32 rows.  Now kMeanRows x kMeanBufs
// rows are in flight, their numbers loaded 64 at a time a round ahead: 131k x 96
// rows over 512 centroids, a load per row 479 us, 32 rows ahead 105, now 58.
constexpr int kMeanRows = 32, kMeanBufs = 4, kMeanRound = kMeanRows * kMeanBufs;

__global__ __launch_bounds__(64) void centroid_mean_kernel(const float* __restrict__ x, int64_t ldx, int d,
                                                           const int32_t* __restrict__ members,
                                                           const int64_t* __restrict__ off,
                                                           float* __restrict__ cent) {
    const int l = blockIdx.x, lane = threadIdx.x;
    const int64_t m0 = off[l], m1 = off[l + 1];
    if (m1 == m0) return;  // keeps its value
    const int j = blockIdx.y * 64 + lane, jc = min(j, d - 1);
    float v[kMeanBufs][kMeanRows];
    int32_t row[kMeanRound / 64], next[kMeanRound / 64];
    // the rows of round m (past the end: the last one again, not added)
    auto rows = [&](int32_t (&r)[kMeanRound / 64], int64_t m) {
#pragma unroll
        for (int i = 0; i < kMeanRound / 64; ++i) r[i] = members[min(m + i * 64 + lane, m1 - 1)];
    };
    auto load = [&](int u) {
#pragma unroll
        for (int t = 0; t < kMeanRows; ++t) {
            const int at = u * kMeanRows + t;
            v[u][t] = x[(int64_t)__builtin_amdgcn_readlane(row[at / 64], at % 64) * ldx + jc];
        }
    };
    double acc = 0.0;
    rows(row, m0);
    rows(next, m0 + kMeanRound);
#pragma unroll
    for (int u = 0; u < kMeanBufs; ++u) load(u);
    for (int64_t m = m0; m < m1; m += kMeanRound) {
#pragma unroll
        for (int i = 0; i < kMeanRound / 64; ++i) row[i] = next[i];
        rows(next, m + 2 * kMeanRound);
#pragma unroll
        for (int u = 0; u < kMeanBufs; ++u) {
            const int64_t mu = m + u * kMeanRows;
            if (mu + kMeanRows <= m1) {
#pragma unroll
                for (int t = 0; t < kMeanRows; ++t) acc += (double)v[u][t];
            } else {
#pragma unroll
                for (int t = 0; t < kMeanRows; ++t)
                    if (mu + t < m1) acc += (double)v[u][t];
            }
            __builtin_amdgcn_sched_barrier(0);  // (the loads stay ahead of the next additions)
            load(u);
            __builtin_amdgcn_sched_barrier(0);
        }
    }
    if (j < d) cent[(size_t)l * d + j] = (float)(acc / (double)(m1 - m0));
}

// The search's forms of the centroids, one thread per (row, quad): tiles (as
// the list arena) and padded rows; clears the largest norm.
__global__ void cent_layout_kernel(const float* __restrict__ raw, int64_t nlist, int d, int nquad, int64_t tiles,
                                   float4* __restrict__ cent, float4* __restrict__ rows,
                                   uint32_t* __restrict__ cmax) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i == 0) *cmax = 0u;
    if (i >= tiles * kTileRows * nquad) return;
    const int64_t r = i / nquad;
    const int j = (int)(i % nquad);
    float v[4] = {0.f, 0.f, 0.f, 0.f};
    if (r < nlist)
        for (int c = 0; c < 4; ++c)
            if (j * 4 + c < d) v[c] = raw[r * d + j * 4 + c];
    const float4 q = make_float4(v[0], v[1], v[2], v[3]);
    cent[((r / kTileRows) * nquad + j) * kTileRows + r % kTileRows] = q;
    if (r < nlist) rows[r * nquad + j] = q;
}

// Squared norms, FP64 sums in dim order rounded once (0 on padding rows), and
// the bits of the largest (those of inf when one is not finite).
__global__ __launch_bounds__(64) void cent_norm_kernel(const float* __restrict__ raw, int64_t nlist, int d,
                                                       float* __restrict__ norm, uint32_t* __restrict__ cmax) {
    const int64_t r = (int64_t)blockIdx.x * 64 + threadIdx.x;
    double s = 0.0;
    if (r < nlist) {
        const float* p = raw + r * d;
        int j = 0;
        for (; j + 16 <= d; j += 16) {
            float v[16];
#pragma unroll
            for (int t = 0; t < 16; ++t) v[t] = p[j + t];
#pragma unroll
            for (int t = 0; t < 16; ++t) s += (double)v[t] * (double)v[t];
        }
        for (; j < d; ++j) s += (double)p[j] * (double)p[j];
    }
    const float f = (float)s;
    norm[r] = f;
    atomicMax(cmax, f <= FLT_MAX ? __float_as_uint(f) : 0x7F800000u);
}

// The tiled list arena from rows in list order: one thread per (tile, lane).
__global__ __launch_bounds__(256) void fill_arena_kernel(const float4* __restrict__ x, int nquad, int d,
                                                         const int32_t* __restrict__ order,
                                                         const int64_t* __restrict__ list_off,
                                                         const int32_t* __restrict__ tile_off,
                                                         const int32_t* __restrict__ tile_list, int64_t tiles,
                                                         float4* __restrict__ codes, uint32_t* __restrict__ ids,
                                                         float* __restrict__ norms, uint32_t* __restrict__ flags) {
    const int64_t g = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    const int64_t T = g / kTileRows;  // (a tile is one wave: its lanes stay together)
    if (T >= tiles) return;
    const int r = (int)(g % kTileRows);
    const int l = tile_list[T];
    const int64_t rr = (T - tile_off[l]) * kTileRows + r;
    const int64_t n_l = list_off[l + 1] - list_off[l];
    float4* dst = codes + (size_t)T * nquad * kTileRows + r;
    uint32_t f = 0;
    float mx = 0.0f;
    if (rr >= n_l) {
        for (int j = 0; j < nquad; ++j) dst[(size_t)j * kTileRows] = make_float4(0.f, 0.f, 0.f, 0.f);
        ids[g] = kNoId;
        norms[g] = 0.0f;
    } else {
        const int32_t row = order[list_off[l] + rr];
        const float4* src = x + (size_t)row * nquad;
        double s = 0.0;
        bool u8 = true;
#pragma unroll 4
        for (int j = 0; j < nquad; ++j) {
            const float4 v = src[j];
            dst[(size_t)j * kTileRows] = v;
            const float c[4] = {v.x, v.y, v.z, v.w};
            for (int i = 0; i < 4; ++i) {
                if (4 * j + i >= d) break;
                s += (double)c[i] * (double)c[i];
                mx = fmaxf(mx, fabsf(c[i]));
                u8 = u8 && c[i] >= 0.0f && c[i] <= 255.0f && c[i] == rintf(c[i]);
            }
        }
        ids[g] = (uint32_t)row;
        const float nr = (float)s;
        norms[g] = nr;
        f = (u8 ? 0u : 1u) | (nr < 1e37f ? 0u : 2u);
    }
    // bit 0: a value that is no integer in [0, 255]; bit 1: a norm past 1e37;
    // flags[1]: bits of the largest magnitude.  One atomic per wave, and none
    // where it would change nothing (one per row queued up on the line).
    const uint32_t fw = (__ballot(f & 1u) ? 1u : 0u) | (__ballot(f & 2u) ? 2u : 0u);
    mx = wave_max(mx);
    if (r == 0) {
        if (fw & ~flags[0]) atomicOr(flags, fw);
        if (__float_as_uint(mx) > flags[1]) atomicMax(flags + 1, __float_as_uint(mx));
    }
}

// Row i divided by its norm (the FP32 FMA chain over the d dims, then a
// correctly rounded square root and quotient); a zero row stays zero.
__global__ void normalize_rows_kernel(const float* __restrict__ x, int64_t n, int d, int ld,
                                      float* __restrict__ y) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const float* r = x + i * ld;
    float s = 0.0f;
    for (int j = 0; j < d; ++j) s = __builtin_fmaf(r[j], r[j], s);
    const float nr = __builtin_sqrtf(s);
    float* o = y + i * ld;
    for (int j = 0; j < ld; ++j) o[j] = nr > 0.0f ? r[j] / nr : r[j];
}

unsigned grid_of(int64_t n, int bs) { return (unsigned)((n + bs - 1) / bs); }

// Stable radix passes over 8-bit digits [shift0, shift0 + 8 * passes) of
// key[], starting from the order perm (nullptr = row order); the result
// is left in *out (one of a, b).
hipError_t radix_passes(const uint32_t* key, int64_t n, int shift0, int passes, const int32_t* perm, int32_t* a,
                        int32_t* b, uint32_t* counts, uint32_t* total, hipStream_t s, const int32_t** out) {
    const int nchunks = (int)((n + kChunk - 1) / kChunk);
    const int32_t* in = perm;
    int32_t* bufs[2] = {a, b};
    for (int p = 0; p < passes; ++p) {
        int32_t* o = bufs[p & 1];
        if (o == in) o = bufs[(p + 1) & 1];
        const int shift = shift0 + 8 * p;
        hipLaunchKernelGGL(rp_count_kernel, dim3(nchunks), dim3(64), 0, s, key, in, shift, n, nchunks, counts);
        hipLaunchKernelGGL(rp_scan_kernel, dim3(kDigits), dim3(256), 0, s, counts, nchunks, total);
        hipLaunchKernelGGL(rp_fill_kernel, dim3(nchunks), dim3(64), 0, s, key, in, shift, n, nchunks, counts, total,
                           o);
        hipError_t e = hipGetLastError();
        if (e != hipSuccess) return e;
        in = o;
    }
    *out = in;
    return hipSuccess;
}

// 8-bit passes covering the label keys 0 .. nlist
int label_passes(int64_t nlist) { return nlist < 256 ? 1 : nlist < 65536 ? 2 : 3; }

}  // namespace

// Rows grouped by label (stable: row order inside a label) and the label
// offsets, for n labels already on the device.  `key` may hold a second
// key (sorted first, inside each label) or be null.
struct Grouping {
    DevBuf<int32_t> pa, pb;
    DevBuf<uint32_t> counts, total, lkey;
    DevBuf<int64_t> off;
    const int32_t* order = nullptr;
};

static int group_rows(hivf_index* h, const int32_t* label, const uint32_t* key2, int64_t n, Grouping& G,
                      hipStream_t s) {
    const int nchunks = (int)((n + kChunk - 1) / kChunk);
    HIP_TRY(h, G.pa.ensure((size_t)n));
    HIP_TRY(h, G.pb.ensure((size_t)n));
    HIP_TRY(h, G.counts.ensure((size_t)nchunks * kDigits));
    HIP_TRY(h, G.total.ensure(kDigits));
    HIP_TRY(h, G.lkey.ensure((size_t)n));
    HIP_TRY(h, G.off.ensure((size_t)h->nlist + 1));
    hipLaunchKernelGGL(label_key_kernel, dim3(grid_of(n, 256)), dim3(256), 0, s, label, n, (int)h->nlist, G.lkey.p);
    const int32_t* order = nullptr;
    if (key2) HIP_TRY(h, radix_passes(key2, n, 0, 4, nullptr, G.pa.p, G.pb.p, G.counts.p, G.total.p, s, &order));
    // labels are the final (most significant) key
    HIP_TRY(h, radix_passes(G.lkey.p, n, 0, label_passes(h->nlist), order, G.pa.p, G.pb.p, G.counts.p, G.total.p, s,
                            &order));
    hipLaunchKernelGGL(label_off_kernel, dim3(grid_of(n + 1, 256)), dim3(256), 0, s, G.lkey.p, order, n,
                       (int)h->nlist, G.off.p);
    HIP_TRY(h, hipGetLastError());
    G.order = order;
    return HIVF_OK;
}

int layout_centroids(hivf_index* h, hipStream_t s) {
    const int64_t tiles = (h->nlist + kTileRows - 1) / kTileRows;
    HIP_TRY(h, h->d_cent.ensure((size_t)tiles * h->nquad * kTileRows));
    HIP_TRY(h, h->d_cent_rows.ensure((size_t)h->nlist * h->nquad));
    HIP_TRY(h, h->d_cent_norm.ensure((size_t)tiles * kTileRows));
    HIP_TRY(h, h->d_cent_max.ensure(1));
    hipLaunchKernelGGL(cent_layout_kernel, dim3(grid_of(tiles * kTileRows * h->nquad, 256)), dim3(256), 0, s,
                       h->d_cent_raw.p, h->nlist, (int)h->d, h->nquad, tiles, h->d_cent.p, h->d_cent_rows.p,
                       h->d_cent_max.p);
    hipLaunchKernelGGL(cent_norm_kernel, dim3((unsigned)tiles), dim3(kTileRows), 0, s, h->d_cent_raw.p, h->nlist,
                       (int)h->d, h->d_cent_norm.p, h->d_cent_max.p);
    HIP_TRY(h, hipGetLastError());
    h->coarse.valid = false;
    return HIVF_OK;
}

int gpu_lloyd(hivf_index* h, const float4* xa, const float* xsum, int64_t ldx, int64_t n, int niter,
              float* cent_host) {
    hipStream_t s = h->stream;
    Grouping G;
    for (int it = 0; it < niter; ++it) {
        int rc = run_assign(h, xa, n, false, s);
        if (rc) return rc;
        rc = group_rows(h, h->d_probes.p, nullptr, n, G, s);
        if (rc) return rc;
        hipLaunchKernelGGL(centroid_mean_kernel, dim3((unsigned)h->nlist, (unsigned)((h->d + 63) / 64)), dim3(64), 0, s,
                           xsum, ldx, (int)h->d, G.order, G.off.p, h->d_cent_raw.p);
        HIP_TRY(h, hipGetLastError());
        rc = layout_centroids(h, s);
        if (rc) return rc;
    }
    HIP_TRY(h, hipMemcpyAsync(cent_host, h->d_cent_raw.p, (size_t)h->nlist * h->d * sizeof(float),
                              hipMemcpyDeviceToHost, s));
    HIP_TRY(h, hipStreamSynchronize(s));
    return HIVF_OK;
}

namespace {

// Element e of the CSR order (row r of list l) -> its arena row, its list
// and the order key of its radius.
__global__ void shadow_elems_kernel(const int32_t* __restrict__ tile_list, const int32_t* __restrict__ tile_off,
                                    const int32_t* __restrict__ size, const int64_t* __restrict__ list_off,
                                    const float* __restrict__ radius, int64_t arena_rows,
                                    int32_t* __restrict__ elem_row, int32_t* __restrict__ elem_list,
                                    uint32_t* __restrict__ key) {
    const int64_t g = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (g >= arena_rows) return;
    const int l = tile_list[g / kTileRows];
    const int64_t r = g - (int64_t)tile_off[l] * kTileRows;
    if (r >= size[l]) return;  // padding
    const int64_t e = list_off[l] + r;
    elem_row[e] = (int32_t)g;
    elem_list[e] = l;
    key[e] = f2ord(radius[g]);
}

// perm[arena position] = arena row shown there: every list's real rows by
// (radius, arena row), padding rows in place.
__global__ void shadow_perm_kernel(const int32_t* __restrict__ tile_list, const int32_t* __restrict__ tile_off,
                                   const int32_t* __restrict__ size, const int64_t* __restrict__ list_off,
                                   const int32_t* __restrict__ order, const int32_t* __restrict__ elem_row,
                                   int64_t arena_rows, int32_t* __restrict__ perm) {
    const int64_t g = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (g >= arena_rows) return;
    const int l = tile_list[g / kTileRows];
    const int64_t r = g - (int64_t)tile_off[l] * kTileRows;
    perm[g] = r < size[l] ? elem_row[order[list_off[l] + r]] : (int32_t)g;
}

// Radius interval of every 32-row tile in shadow order, widened by 10^-4
// (empty tiles: an empty interval).
__global__ void shadow_bounds_kernel(const int32_t* __restrict__ tile_list, const int32_t* __restrict__ tile_off,
                                     const int32_t* __restrict__ size, const int32_t* __restrict__ perm,
                                     const float* __restrict__ radius, int64_t tiles32, float2* __restrict__ rb) {
    const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= tiles32) return;
    const int l = tile_list[t / 2];
    const int64_t r0 = (t - 2 * (int64_t)tile_off[l]) * 32;
    float lo = INFINITY, hi = -INFINITY;
    for (int i = 0; i < 32; ++i) {
        if (r0 + i >= size[l]) break;
        const float x = radius[perm[t * 32 + i]];
        lo = fminf(lo, x * (1.0f - 1e-4f));
        hi = fmaxf(hi, x * (1.0f + 1e-4f) + 1e-30f);
    }
    rb[t] = make_float2(lo, hi);
}

}  // namespace

int shadow_order(hivf_index* h, const float* radius, int32_t* perm, float2* rb8, hipStream_t s) {
    const int64_t nlist = h->nlist, tiles = h->tiles, arena_rows = tiles * kTileRows, n = h->ntotal;
    if (tiles == 0) return HIVF_OK;
    std::vector<int32_t> tile_list((size_t)tiles);
    for (int64_t l = 0; l < nlist; ++l)
        for (int32_t t = h->tile_off[l]; t < h->tile_off[l + 1]; ++t) tile_list[t] = (int32_t)l;
    DevBuf<int32_t> dtl, erow, elist;
    DevBuf<uint32_t> key;
    DevBuf<int64_t> loff;
    HIP_TRY(h, dtl.ensure((size_t)tiles));
    HIP_TRY(h, loff.ensure((size_t)nlist + 1));
    HIP_TRY(h, erow.ensure((size_t)std::max<int64_t>(n, 1)));
    HIP_TRY(h, elist.ensure((size_t)std::max<int64_t>(n, 1)));
    HIP_TRY(h, key.ensure((size_t)std::max<int64_t>(n, 1)));
    HIP_TRY(h, hipMemcpyAsync(dtl.p, tile_list.data(), tiles * sizeof(int32_t), hipMemcpyHostToDevice, s));
    HIP_TRY(h, hipMemcpyAsync(loff.p, h->list_off.data(), (nlist + 1) * sizeof(int64_t), hipMemcpyHostToDevice, s));
    hipLaunchKernelGGL(shadow_elems_kernel, dim3(grid_of(arena_rows, 256)), dim3(256), 0, s, dtl.p, h->d_tile_off.p,
                       h->d_size.p, loff.p, radius, arena_rows, erow.p, elist.p, key.p);
    HIP_TRY(h, hipGetLastError());
    Grouping G;
    if (n > 0) {
        int rc = group_rows(h, elist.p, key.p, n, G, s);
        if (rc) return rc;
    }
    hipLaunchKernelGGL(shadow_perm_kernel, dim3(grid_of(arena_rows, 256)), dim3(256), 0, s, dtl.p, h->d_tile_off.p,
                       h->d_size.p, loff.p, n > 0 ? G.order : erow.p, erow.p, arena_rows, perm);
    hipLaunchKernelGGL(shadow_bounds_kernel, dim3(grid_of(2 * tiles, 256)), dim3(256), 0, s, dtl.p, h->d_tile_off.p,
                       h->d_size.p, perm, radius, 2 * tiles, rb8);
    HIP_TRY(h, hipGetLastError());
    HIP_TRY(h, hipStreamSynchronize(s));  // locals
    return HIVF_OK;
}

int normalize_rows(hivf_index* h, const float4* x, int64_t n, float4* y) {
    hipLaunchKernelGGL(normalize_rows_kernel, dim3(grid_of(n, 256)), dim3(256), 0, h->stream,
                       reinterpret_cast<const float*>(x), n, (int)h->d, (int)h->d_pad, reinterpret_cast<float*>(y));
    HIP_TRY(h, hipGetLastError());
    return HIVF_OK;
}

int gpu_add(hivf_index* h, int64_t n) {
    // rows are staged in h->d_q (padded float4 rows)
    hipStream_t s = h->stream;
    const int64_t nlist = h->nlist;
    HIP_TRY(h, h->d_cd.ensure((size_t)std::max<int64_t>(n, 1)));
    HIP_TRY(h, h->d_probes.ensure((size_t)std::max<int64_t>(n, 1)));
    Grouping G;
    DevBuf<uint32_t> key;
    if (n > 0) {
        int rc = run_assign(h, h->d_q.p, n, true, s);
        if (rc) return rc;
        HIP_TRY(h, key.ensure((size_t)n));
        hipLaunchKernelGGL(dist_key_kernel, dim3(grid_of(n, 256)), dim3(256), 0, s, h->d_cd.p, n,
                           h->metric == HIVF_METRIC_L2 ? 1 : 0, key.p);
        rc = group_rows(h, h->d_probes.p, key.p, n, G, s);
        if (rc) return rc;
    }
    std::vector<int64_t> list_off(nlist + 1, 0);
    if (n > 0) {
        HIP_TRY(h, hipMemcpyAsync(list_off.data(), G.off.p, (nlist + 1) * sizeof(int64_t), hipMemcpyDeviceToHost, s));
        HIP_TRY(h, hipStreamSynchronize(s));
        // (rows past the last list's end have no centroid)
        if (list_off[nlist] != n) return h->fail(HIVF_EINVAL, "rows without a nearest centroid (non-finite values)");
    }
    std::vector<int32_t> tile_off(nlist + 1, 0), size(nlist, 0);
    int64_t tiles = 0;
    for (int64_t l = 0; l < nlist; ++l) {
        const int64_t n_l = list_off[l + 1] - list_off[l];
        if (n_l > INT32_MAX) return h->fail(HIVF_EINVAL, "list too long");
        size[l] = (int32_t)n_l;
        tile_off[l] = (int32_t)tiles;
        tiles += (n_l + kTileRows - 1) / kTileRows;
        if (tiles > INT32_MAX / kTileRows) return h->fail(HIVF_EINVAL, "index too large");
    }
    tile_off[nlist] = (int32_t)tiles;
    std::vector<int32_t> tile_list((size_t)std::max<int64_t>(tiles, 1), 0);
    for (int64_t l = 0; l < nlist; ++l)
        for (int32_t t = tile_off[l]; t < tile_off[l + 1]; ++t) tile_list[t] = (int32_t)l;
    const int nquad = h->nquad;
    HIP_TRY(h, h->d_codes.ensure((size_t)std::max<int64_t>(tiles, 1) * nquad * kTileRows + kArenaTail));
    HIP_TRY(h, h->d_ids.ensure((size_t)std::max<int64_t>(tiles, 1) * kTileRows));
    HIP_TRY(h, h->d_norms.ensure((size_t)std::max<int64_t>(tiles, 1) * kTileRows));
    HIP_TRY(h, h->d_tile_off.ensure(nlist + 1));
    HIP_TRY(h, h->d_size.ensure(nlist));
    HIP_TRY(h, hipMemcpyAsync(h->d_tile_off.p, tile_off.data(), (nlist + 1) * sizeof(int32_t), hipMemcpyHostToDevice,
                              s));
    HIP_TRY(h, hipMemcpyAsync(h->d_size.p, size.data(), nlist * sizeof(int32_t), hipMemcpyHostToDevice, s));
    uint32_t flags[2] = {0, 0};
    if (tiles > 0) {
        DevBuf<int32_t> dtl;
        DevBuf<uint32_t> flag;
        HIP_TRY(h, dtl.ensure((size_t)tiles));
        HIP_TRY(h, flag.ensure(2));
        HIP_TRY(h, hipMemcpyAsync(dtl.p, tile_list.data(), tiles * sizeof(int32_t), hipMemcpyHostToDevice, s));
        hipLaunchKernelGGL(zero_u32_kernel, dim3(1), dim3(64), 0, s, flag.p, 2);
        hipLaunchKernelGGL(zero_u32_kernel, dim3(grid_of(kArenaTail * 4, 256)), dim3(256), 0, s,
                           reinterpret_cast<uint32_t*>(h->d_codes.p + (size_t)tiles * nquad * kTileRows),
                           kArenaTail * 4);
        hipLaunchKernelGGL(fill_arena_kernel, dim3(grid_of(tiles * kTileRows, 256)), dim3(256), 0, s, h->d_q.p,
                           nquad, (int)h->d, G.order, G.off.p, h->d_tile_off.p, dtl.p, tiles, h->d_codes.p,
                           h->d_ids.p, h->d_norms.p, flag.p);
        HIP_TRY(h, hipGetLastError());
        HIP_TRY(h, hipMemcpyAsync(flags, flag.p, sizeof(flags), hipMemcpyDeviceToHost, s));
    }
    HIP_TRY(h, hipStreamSynchronize(s));  // host vectors and local buffers
    h->lists_uint8 = (flags[0] & 1u) == 0;
    h->lists_sane = (flags[0] & 2u) == 0;
    std::memcpy(&h->lists_absmax, flags + 1, sizeof(float));
    h->list_off = list_off;
    h->tile_off = tile_off;
    h->ntotal = list_off[nlist];
    h->tiles = tiles;
    h->have_lists = true;
    h->batched.invalidate();
    h->drop_graph();
    return HIVF_OK;
}

}  // namespace hivf
