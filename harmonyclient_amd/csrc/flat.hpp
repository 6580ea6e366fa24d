// Exact FP32 scans of a batch of plain or pruned searches (included by
// batched.hip): every row whose distance lies within its query's bound goes
// to the query's survivor buffer, and the selection takes the top-k.
//
// The distance is the canonical FMA chain, so keys are final.  The bound (the
// warm-up scan's k-th distance over some of the query's own rows) is >= the
// k-th distance, so every row of the top-k survives.  For L2 a chain only
// grows: once a row's partial distance exceeds the bound its distance does
// too, and the remaining dims of a group are skipped when that holds for
// every row and query of it.
#pragma once

namespace hivf {
namespace {

struct FlatArgs {
    DevLists lists;
    const float4* q;       // [nq x nquad]
    const float* tau;      // [nq] bounds (inner products for IP)
    uint32_t* scnt;        // [nq] survivors per query
    uint64_t* sbuf;        // [nq x cap] (rank, arena row)
    uint32_t cap;
    int block_dims;        // dims between two bound checks (made on whole quads)
    int nblocks;
    unsigned long long* rows_scanned;  // optional: rows of the scanned lists (pair form)
    unsigned long long* skips;         // optional: (row, block) pairs skipped
    // list-major form
    const BatchItem* items;
    uint32_t* meta;
    const int32_t* lq;     // query ids per list
    uint32_t max_items;
    // pair form
    const int32_t* probes; // [nq x P]
    const int32_t* npq;    // per-query probe counts (null: P)
    int P;
    int parts;             // workgroups per (query, probe)
};

typedef const __attribute__((address_space(4))) float4* UniformQuads;

// R tiles of 64 rows (a row per lane) from `tile` on against QB queries whose
// ids and rank bounds are wave-uniform.  The queries' components come through
// the scalar cache as SGPR operands, so a quad of R tiles costs R vector loads
// for 8 R QB vector operations.  left: the list's rows from the first tile on.
template <int METRIC, int R, int QB>
__device__ __forceinline__ void flat_tiles(const FlatArgs& a, int tile, int left, const int (&qid)[QB],
                                           const float (&rtau)[QB], int lane, unsigned long long& skipped) {
    const int nquad = a.lists.nquad;
    const float4* tp = a.lists.codes + (size_t)tile * nquad * 64 + lane;
    const UniformQuads qb = (UniformQuads)a.q;
    UniformQuads qp[QB];
#pragma unroll
    for (int i = 0; i < QB; ++i) qp[i] = qb + (size_t)qid[i] * nquad;
    float acc[QB][R];
#pragma unroll
    for (int i = 0; i < QB; ++i)
#pragma unroll
        for (int r = 0; r < R; ++r) acc[i][r] = 0.0f;
    int j = 0;
    const int nb = METRIC == kL2 ? a.nblocks : 1;
    for (int b = 0; b < nb; ++b) {
        const int je = b < nb - 1 ? ((b + 1) * a.block_dims) >> 2 : nquad;
#pragma unroll(QB == 1 ? 4 : 2)
        for (; j < je; ++j) {
            float4 x[R];
#pragma unroll
            for (int r = 0; r < R; ++r) x[r] = tp[((size_t)r * nquad + j) * 64];
#pragma unroll
            for (int i = 0; i < QB; ++i) {
                const float4 qv = {qp[i][j].x, qp[i][j].y, qp[i][j].z, qp[i][j].w};
#pragma unroll
                for (int r = 0; r < R; ++r) acc[i][r] = accum<METRIC>(acc[i][r], qv, x[r]);
            }
        }
        if (METRIC == kL2 && b < nb - 1) {
            uint64_t any = 0;
#pragma unroll
            for (int i = 0; i < QB; ++i)
#pragma unroll
                for (int r = 0; r < R; ++r) {
                    // (a padding row's chain is finite too; it only costs a round more)
                    const uint64_t m = __ballot(acc[i][r] <= rtau[i]);
                    any |= m;
                    if (a.skips && rtau[i] >= 0.0f) {  // (not an absent query's)
                        const int rows = min(64, left - r * 64);
                        const uint64_t live = rows >= 64 ? ~0ull : (1ull << rows) - 1ull;
                        skipped += (unsigned)__popcll(live & ~m);
                    }
                }
            if (any == 0) {
                if (a.skips) {  // every later check of these rows as well
#pragma unroll
                    for (int i = 0; i < QB; ++i)
                        if (rtau[i] >= 0.0f) skipped += (unsigned long long)min(64 * R, left) * (nb - 2 - b);
                }
                return;
            }
        }
    }
    uint64_t m[QB][R];
    uint64_t any = 0;
    uint32_t cnt = 0;
#pragma unroll
    for (int i = 0; i < QB; ++i) {
        uint32_t c = 0;
#pragma unroll
        for (int r = 0; r < R; ++r) {
            m[i][r] = __ballot(lane < left - r * 64 && rank_of<METRIC>(acc[i][r]) <= rtau[i]);
            c += (uint32_t)__popcll(m[i][r]);
            any |= m[i][r];
        }
        cnt = lane == i ? c : cnt;
    }
    if (any == 0) return;
    // lane i reserves query i's run: one round trip for all of them
    uint32_t base = 0;
    int myq = qid[0];
#pragma unroll
    for (int i = 1; i < QB; ++i) myq = lane == i ? qid[i] : myq;
    if (lane < QB && cnt) base = atomicAdd(&a.scnt[myq], cnt);
#pragma unroll
    for (int i = 0; i < QB; ++i) {
        uint32_t at = __builtin_amdgcn_readlane(base, i);
        uint64_t* out = a.sbuf + (size_t)qid[i] * a.cap;
#pragma unroll
        for (int r = 0; r < R; ++r) {
            if ((m[i][r] >> lane) & 1ull) {
                const uint32_t pos = at + lanes_below(m[i][r]);
                if (pos < a.cap)
                    out[pos] = make_key(rank_of<METRIC>(acc[i][r]), (uint32_t)((tile + r) * 64 + lane));
            }
            at += (uint32_t)__popcll(m[i][r]);
        }
    }
}

// Rank bound of a query: the warm-up bound, or for an absent one NaN, which no
// rank is within (an inner product of +inf ranks at -inf).
template <int METRIC>
__device__ inline float flat_rank_bound(const FlatArgs& a, int qi) {
    return qi < 0 ? __builtin_nanf("") : METRIC == kL2 ? a.tau[qi] : -a.tau[qi];
}

// Queries of a list-major item, and how many of them share a pass over its
// tiles (the rest of an item with few takes half as many).
constexpr int kFlatItem = 16;
constexpr int kFlatQB = 8;
constexpr int kFlatTiles = 8;  // 32-row tiles per item (a near-query item: half)

template <int METRIC, int QB>
__device__ __forceinline__ void flat_item_group(const FlatArgs& a, int t0, int te, int rows, int tile0, int myq,
                                                float mytau, int g, int lane, unsigned long long& skipped) {
    int qid[QB];
    float rtau[QB];
#pragma unroll
    for (int i = 0; i < QB; ++i) {
        qid[i] = max(__builtin_amdgcn_readlane(myq, g + i), 0);
        rtau[i] = __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(mytau), g + i));
    }
    int t = t0;
    for (; t + 2 <= te; t += 2) flat_tiles<METRIC, 2, QB>(a, tile0 + t, rows - t * 64, qid, rtau, lane, skipped);
    if (t < te) flat_tiles<METRIC, 1, QB>(a, tile0 + t, rows - t * 64, qid, rtau, lane, skipped);
}

// List-major form: persistent waves take (list, up to 16 queries, tiles) items
// from the plan's per-XCD queues, as the batched scans do.  What bounds it is
// vector arithmetic (8 operations per row, query and quad, 4 for IP), where
// the per-query kernel is bound by the caches: it reads every probed list
// once per query, 20 GB through L2 and the Infinity Cache for 1000 queries of
// 32 lists (500k x 128).  That search: 2.75 -> 0.71 ms (this kernel 0.34); 2000
// pruned queries of 48 lists 1.82 -> 0.99 ms (0.76); 500 inner-product queries
// of 20 lists of 201 dims 0.61 -> 0.29 ms (0.15).
template <int METRIC>
__global__ __launch_bounds__(kNT) void flat_scan_kernel(FlatArgs a) {
    const int lane = threadIdx.x & 63;
    unsigned long long skipped = 0;
    int grp = blockIdx.x % kXcds, switches = 0;
    uint32_t start = a.meta[kMetaOff + grp];
    uint32_t end = min(a.meta[kMetaOff + grp + 1], a.max_items);
    for (;;) {
        uint32_t it = 0;
        if (lane == 0) it = start + atomicAdd(&a.meta[kMetaHead + grp * kHeadStride], 1u);
        it = __builtin_amdgcn_readfirstlane(it);
        if (it >= end) {
            if (++switches == kXcds) break;
            grp = (grp + 1) % kXcds;
            start = a.meta[kMetaOff + grp];
            end = min(a.meta[kMetaOff + grp + 1], a.max_items);
            continue;
        }
        const BatchItem w = a.items[it];
        const int nq = __builtin_amdgcn_readfirstlane(w.nq & 0xFFFF);
        const int list = __builtin_amdgcn_readfirstlane(w.list);
        const int rows = a.lists.list_size[list];
        const int tile0 = a.lists.list_tile_off[list];
        // (items start and end on whole 64-row tiles: their tile counts are even)
        const int t0 = __builtin_amdgcn_readfirstlane(w.t0) >> 1;
        const int te = min((rows + 63) >> 6, t0 + (__builtin_amdgcn_readfirstlane(w.nq >> 16) >> 1));
        const int myq = lane < nq ? a.lq[w.q0 + lane] : -1;
        const float mytau = flat_rank_bound<METRIC>(a, myq);
        for (int g = 0; g < nq; g += kFlatQB) {
            if (nq - g > kFlatQB / 2)
                flat_item_group<METRIC, kFlatQB>(a, t0, te, rows, tile0, myq, mytau, g, lane, skipped);
            else
                flat_item_group<METRIC, kFlatQB / 2>(a, t0, te, rows, tile0, myq, mytau, g, lane, skipped);
        }
    }
    if (a.skips && lane == 0 && skipped) atomicAdd(a.skips, skipped);
}

// Pair form, for batches whose queries share few lists: `parts` workgroups per
// (query, probed list), their waves striding the list's tile pairs.
template <int METRIC>
__global__ __launch_bounds__(kNT) void flat_pair_kernel(FlatArgs a) {
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / 64);
    const int part = blockIdx.x % a.parts;
    const int e = blockIdx.x / a.parts;
    const int qi = e / a.P, jp = e % a.P;
    const int Pq = a.npq ? min(a.npq[qi], a.P) : a.P;
    const int l = jp < Pq ? a.probes[(size_t)qi * a.P + jp] : -1;
    if (l < 0) return;
    const int rows = a.lists.list_size[l];
    const int tile0 = a.lists.list_tile_off[l];
    const int nt = (rows + 63) >> 6;
    const int qid[1] = {qi};
    const float rtau[1] = {flat_rank_bound<METRIC>(a, qi)};
    unsigned long long skipped = 0;
    for (int t = (part * (kNT / 64) + wave) * 2; t < nt; t += a.parts * (kNT / 64) * 2) {
        if (t + 2 <= nt)
            flat_tiles<METRIC, 2, 1>(a, tile0 + t, rows - t * 64, qid, rtau, lane, skipped);
        else
            flat_tiles<METRIC, 1, 1>(a, tile0 + t, rows - t * 64, qid, rtau, lane, skipped);
    }
    if (a.skips && lane == 0 && skipped) atomicAdd(a.skips, skipped);
    if (a.rows_scanned && part == 0 && threadIdx.x == 0) atomicAdd(a.rows_scanned, (unsigned long long)rows);
}

// Counters of one chunk of queries, cleared before it.
__global__ void flat_clear_kernel(uint32_t* scnt, int n, uint32_t* lcnt, int nlist, uint32_t* fbc,
                                  int fbc_words, uint32_t* all_int) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) scnt[i] = 0;
    if (i < nlist) lcnt[i] = 0;
    if (i < fbc_words) fbc[i] = 0;
    if (i == 0) *all_int = 0;
}

}  // namespace
}  // namespace hivf
