// List-major scan of a batch on MFMA at nearly FP32 precision (included by
// batched.hip): rows and queries as two BF16 pieces each (v = hi + lo + r,
// |r| <= 2^-16 |v|), three products per 16 dims, straight from the FP32 list
// arena.  A row survives when its approximate rank - E is within the query's
// bound, E = split_coef (||q||^2 + ||x||^2) + kSplitAbs bounding the error
// against the FP32 chain; the selection rescores the few rows near the k-th
// with that chain, so results are the chain's.
//
// What bounds it: the products are 3 v_mfma_f32_32x32x16_bf16 (96 cycles) per 16
// dims of 32 rows x 32 queries, and splitting the rows about as many vector
// cycles, where the FP32 chain needs 2048 vector cycles for the same.  1000 plain
// queries of 32 lists (500k x 128): 98 us against 336 for the FP32 scan, their host
// search 0.70 -> 0.49 ms with it (0.35 now); 2000 pruned queries of 48 lists 173 us,
// the search without statistics 0.96 -> 0.43 ms (0.26 now); 500 inner-product
// queries of 201 dims 46 us against 152.
#pragma once

namespace hivf {
namespace {

struct SplitArgs {
    DevLists lists;
    const float* norms;    // [rows] squared row norms
    const uint16_t* qh;    // [nq x dpad16] the queries' pieces
    const uint16_t* ql;
    const float* qn;       // [nq] squared norms
    const float* tau;      // [nq] bounds (inner products for IP)
    const BatchItem* items;
    uint32_t* meta;
    const int32_t* lq;
    uint32_t max_items;
    uint32_t* scnt;
    uint64_t* sbuf;
    uint32_t cap;          // even
    int nkc, dpad16;
    float coef;
};

// absolute part of E: BF16 / FP32 values below the normal range may be
// flushed to zero by the matrix cores
constexpr float kSplitAbs = 1e-30f;

// Eight consecutive dims as their two BF16 pieces (RNE).
template <bool LO>
__device__ __forceinline__ void split8(const float4& u, const float4& v, bf16x8& h, bf16x8& l) {
    typedef __attribute__((ext_vector_type(2))) __bf16 bf16x2;
    typedef __attribute__((ext_vector_type(4))) uint32_t u32x4;
    const float e[8] = {u.x, u.y, u.z, u.w, v.x, v.y, v.z, v.w};
    u32x4 hp, lp;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const bf16x2 p = {(__bf16)e[2 * i], (__bf16)e[2 * i + 1]};
        const uint32_t w = __builtin_bit_cast(uint32_t, p);
        hp[i] = w;
        if constexpr (LO) {
            const bf16x2 r = {(__bf16)(e[2 * i] - __uint_as_float(w << 16)),
                              (__bf16)(e[2 * i + 1] - __uint_as_float(w & 0xFFFF0000u))};
            lp[i] = __builtin_bit_cast(uint32_t, r);
        }
    }
    h = __builtin_bit_cast(bf16x8, hp);
    if constexpr (LO) l = __builtin_bit_cast(bf16x8, lp);
}

// One tile's accumulators against the bound of this lane's query: rank - E =
// fma(-2, acc, (1 - coef)(qn + xn) - abs) for L2, -acc - E for IP.  (The two
// roundings are far below the 1 % that coef is widened by.)  Returns the mask
// of passing rows ((r / 4) * 8 + half * 4 + r % 4) and their ranks.
template <int METRIC>
__device__ __forceinline__ uint32_t split_pass(const floatx16& acc, const float (&xn)[16], float qn, float rtau,
                                               float coef, uint32_t rows_ok) {
    float t[16];
#pragma unroll
    for (int r = 0; r < 16; ++r) {
        const float s = qn + xn[r];
        t[r] = METRIC == kL2 ? __builtin_fmaf(-2.0f, acc[r], __builtin_fmaf(1.0f - coef, s, -kSplitAbs))
                             : -acc[r] - __builtin_fmaf(coef, s, kSplitAbs);
    }
    float mn = fminf(fminf(t[0], t[1]), t[2]);
#pragma unroll
    for (int r = 3; r < 15; r += 2) mn = fminf(fminf(mn, t[r]), t[r + 1]);
    mn = fminf(mn, t[15]);
    if (__ballot(mn <= rtau) == 0) return 0u;
    uint32_t m = 0;
#pragma unroll
    for (int r = 0; r < 16; ++r) m |= (t[r] <= rtau ? 1u : 0u) << r;
    return m & rows_ok;
}

template <int METRIC>
__device__ __forceinline__ float split_rank(float acc, float qn, float xn) {
    return METRIC == kL2 ? __builtin_fmaf(-2.0f, acc, qn + xn) : -acc;
}

// d <= 128: a wave per item of up to 32 queries.  The queries' pieces stay in
// registers (B operands), a tile's FP32 rows are loaded a tile ahead and split
// in registers.  XLO: the rows' second piece exists (integer rows in [0, 255]
// are exact in the first).
constexpr int kSplitItem = 32;

template <int METRIC, int NKC, bool XLO>
__global__ __launch_bounds__(kNT) __attribute__((amdgpu_waves_per_eu(2))) void split_wave_kernel(SplitArgs a) {
    __shared__ uint64_t st_key[kNT / 64][32][kStage + 1];
    const int wv = threadIdx.x / 64, lane = threadIdx.x & 63, half = lane >> 5, slot = lane & 31;
    const int nquad = a.lists.nquad, nkc = a.nkc;
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
        const int nq = w.nq & 0xFFFF;
        const int list = __builtin_amdgcn_readfirstlane(w.list);
        const int rows = a.lists.list_size[list];
        const int T0 = a.lists.list_tile_off[list] * 2;  // 32-row tiles
        const int te = min((rows + 31) >> 5, w.t0 + (w.nq >> 16));
        const bool live = slot < nq;
        const int qid = a.lq[w.q0 + min(slot, nq - 1)];
        float4 raw[NKC][2];
        // a tile's rows (lane: row slot, quads 4 kc + 2 half and the next) and
        // norms; quads past the row's end are the next tile's (or the arena's
        // zeroed tail), finite values that meet zeros of the queries' pieces
        // (No branch around a load: with one, every product waits for all loads
        // in flight.  Past nkc the last chunk meets zeros.  A chunk's next rows
        // are loaded once it is split: with the whole tile's after the products,
        // 40 registers spilled, and 2000 pruned queries took 379 us, now 334; 1000
        // plain 406, now 392.)
        const uint32_t lo = half * 128 + slot;
        auto tile = [&](int T) {
            const int g = __builtin_amdgcn_readfirstlane(T0 + T);
            return a.lists.codes + (size_t)(g >> 1) * nquad * 64 + (g & 1) * 32;
        };
        auto load = [&](const float4* p, int kc) {
            const float4* c = p + min(kc, nkc - 1) * 256;
            raw[kc][0] = c[lo];
            raw[kc][1] = (c + 64)[lo];
        };
        {
            const float4* p = tile(w.t0);
#pragma unroll
            for (int kc = 0; kc < NKC; ++kc) load(p, kc);
        }
        bf16x8 bh[NKC], bl[NKC];
        {
            const bf16x8* hp = reinterpret_cast<const bf16x8*>(a.qh + (size_t)qid * a.dpad16 + half * 8);
            const bf16x8* lp = reinterpret_cast<const bf16x8*>(a.ql + (size_t)qid * a.dpad16 + half * 8);
            const bf16x8 z = {};
#pragma unroll
            for (int kc = 0; kc < NKC; ++kc) {
                bh[kc] = kc < nkc ? hp[kc * 2] : z;
                bl[kc] = kc < nkc ? lp[kc * 2] : z;
            }
        }
        const float qn = a.qn[qid];
        const float tq = a.tau[qid];
        const float rtau = !live ? -INFINITY : METRIC == kL2 ? (tq < FLT_MAX ? tq : INFINITY) : (tq > -FLT_MAX ? -tq : INFINITY);
        uint32_t mycnt = 0;  // keys staged for the lane's slot (the same in both halves)
        auto flush = [&]() {  // (runs of even length, as the int8 scan's)
            const uint32_t take = (mycnt + 1u) & ~1u;
            uint32_t b0 = 0;
            if (half == 0 && mycnt > 0) {
                b0 = atomicAdd(&a.scnt[qid], take);
                if (take != mycnt) st_key[wv][slot][mycnt] = kNoKey;
            }
            b0 = __shfl(b0, slot);
            __builtin_amdgcn_wave_barrier();
            for (uint32_t j = 2 * half; j < take; j += 4) {
                const uint32_t dst = b0 + j;
                const uint64_t k0 = st_key[wv][slot][j], k1 = st_key[wv][slot][j + 1];
                uint64_t* out = a.sbuf + (size_t)qid * a.cap + dst;
                if (dst + 1 < a.cap)
                    *reinterpret_cast<ulonglong2*>(out) = make_ulonglong2(k0, k1);
                else if (dst < a.cap)
                    *out = k0;
            }
            mycnt = 0;
            __builtin_amdgcn_wave_barrier();
        };
        for (int T = w.t0; T < te; ++T) {
            floatx16 acc = {};
            float4 xv[4];
            const float* np = a.norms + (size_t)__builtin_amdgcn_readfirstlane(T0 + T) * 32;
#pragma unroll
            for (int r4 = 0; r4 < 4; ++r4) xv[r4] = *reinterpret_cast<const float4*>(np + r4 * 8 + half * 4);
            const float4* next = tile(min(T + 1, te - 1));
#pragma unroll
            for (int kc = 0; kc < NKC; ++kc) {
                bf16x8 h, l;
                split8<XLO>(raw[kc][0], raw[kc][1], h, l);
                load(next, kc);
                if constexpr (XLO) acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(l, bh[kc], acc, 0, 0, 0);
                acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(h, bl[kc], acc, 0, 0, 0);
                acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(h, bh[kc], acc, 0, 0, 0);
            }
            float xn[16];
#pragma unroll
            for (int r4 = 0; r4 < 4; ++r4) {
                xn[r4 * 4 + 0] = xv[r4].x;
                xn[r4 * 4 + 1] = xv[r4].y;
                xn[r4 * 4 + 2] = xv[r4].z;
                xn[r4 * 4 + 3] = xv[r4].w;
            }
            const uint32_t m = split_pass<METRIC>(acc, xn, qn, rtau, a.coef, tile_rows_ok(rows - T * 32, half));
            if (__ballot(m != 0) == 0) continue;
            const uint32_t cg = (uint32_t)__builtin_popcount(m);
            const uint32_t oc = __shfl_xor(cg, 32);
            if (__ballot(mycnt + cg + oc > (uint32_t)kStage) != 0) flush();
            uint64_t* sk = &st_key[wv][slot][mycnt + (half ? oc : 0u)];
            mycnt += cg + oc;
#pragma unroll
            for (int r = 0; r < 16; ++r)
                if ((m >> r) & 1u) {
                    const int row = (r >> 2) * 8 + half * 4 + (r & 3);
                    sk[__builtin_popcount(m & ((1u << r) - 1u))] =
                        make_key(split_rank<METRIC>(acc[r], qn, xn[r]), (uint32_t)((T0 + T) * 32 + row));
                }
        }
        if (__ballot(mycnt != 0) != 0) flush();
    }
}

// d <= 512: a workgroup of 8 waves per item.  The queries' pieces of all dim
// chunks are staged in LDS once per item (2 KB per 16 dims, up to 64 KB) and
// read by every wave; the waves stride the item's tiles, 2 chunks of rows
// loaded while the 2 before are split and multiplied (4: registers spill, 500 inner
// products of 201 dims 183 us against 181, 1000 of 150 dims 291 against 276).
constexpr int kSplitWgNT = 512, kSplitChunks = 2;

template <int METRIC, bool XLO>
__global__ __launch_bounds__(kSplitWgNT) __attribute__((amdgpu_waves_per_eu(4))) void split_wg_kernel(SplitArgs a) {
    extern __shared__ bf16x8 sb[];  // [hi, lo][kC nch][64 lanes], zeros past nkc
    __shared__ uint32_t s_it;
    constexpr int kW = kSplitWgNT / 64, kC = kSplitChunks;
    const int tid = threadIdx.x, lane = tid & 63, half = lane >> 5, slot = lane & 31;
    const int wv = __builtin_amdgcn_readfirstlane(tid / 64);
    const int nquad = a.lists.nquad, nkc = a.nkc;
    const int nch = (nkc + 2 * kC - 1) / (2 * kC) * 2;  // (an even number of chunk groups)
    int grp = blockIdx.x % kXcds, switches = 0;  // (thread 0's)
    for (;;) {
        __syncthreads();  // every wave is done with the item's queries
        if (tid == 0) {
            uint32_t it = ~0u;
            while (switches < kXcds) {
                const uint32_t end = min(a.meta[kMetaOff + grp + 1], a.max_items);
                it = a.meta[kMetaOff + grp] + atomicAdd(&a.meta[kMetaHead + grp * kHeadStride], 1u);
                if (it < end) break;
                it = ~0u;
                grp = (grp + 1) % kXcds;
                ++switches;
            }
            s_it = it;
        }
        __syncthreads();
        const uint32_t it = __builtin_amdgcn_readfirstlane(s_it);
        if (it == ~0u) break;
        const BatchItem w = a.items[it];
        const int nq = w.nq & 0xFFFF;
        const int list = __builtin_amdgcn_readfirstlane(w.list);
        const int rows = a.lists.list_size[list];
        const int T0 = a.lists.list_tile_off[list] * 2;
        const int te = min((rows + 31) >> 5, w.t0 + (w.nq >> 16));
        for (int e = tid; e < 2 * nch * kC * 64; e += kSplitWgNT) {
            const int l = e & 63, lo = (e >> 6) >= nch * kC, kc = (e >> 6) - lo * nch * kC;
            const int q = a.lq[w.q0 + min(l & 31, nq - 1)];
            const bf16x8 z = {};
            sb[e] = kc < nkc ? *reinterpret_cast<const bf16x8*>((lo ? a.ql : a.qh) + (size_t)q * a.dpad16 + kc * 16 + (l >> 5) * 8) : z;
        }
        const int qid = a.lq[w.q0 + min(slot, nq - 1)];
        const float qn = a.qn[qid];
        const float tq = a.tau[qid];
        const float rtau = slot >= nq ? -INFINITY
                           : METRIC == kL2 ? (tq < FLT_MAX ? tq : INFINITY) : (tq > -FLT_MAX ? -tq : INFINITY);
        __syncthreads();
        float4 ra[kC][2], rb[kC][2];
        auto load = [&](float4 (&raw)[kC][2], int T, int ch) {  // chunk group ch of tile T (or of the next tile)
            if (ch >= nch) {
                ch -= nch;
                T += kW;
            }
            const int g = __builtin_amdgcn_readfirstlane(T0 + min(T, te - 1));
            const float4* p = a.lists.codes + (size_t)(g >> 1) * nquad * 64 + (g & 1) * 32;
            const uint32_t lo = half * 128 + slot;
#pragma unroll
            for (int c = 0; c < kC; ++c) {
                const int kc = min(ch * kC + c, nkc - 1);  // (no branch, as above)
                raw[c][0] = (p + kc * 256)[lo];
                raw[c][1] = (p + kc * 256 + 64)[lo];
            }
        };
        if (w.t0 + wv < te) load(ra, w.t0 + wv, 0);
        for (int T = w.t0 + wv; T < te; T += kW) {
            floatx16 acc = {};
            float4 xv[4];
#pragma unroll
            for (int r4 = 0; r4 < 4; ++r4)
                xv[r4] = *reinterpret_cast<const float4*>(a.norms + (size_t)(T0 + T) * 32 + r4 * 8 + half * 4);
            auto step = [&](const float4 (&raw)[kC][2], int ch) {
#pragma unroll
                for (int c = 0; c < kC; ++c) {
                    const int kc = ch * kC + c;
                    const bf16x8 bh = sb[(size_t)kc * 64 + lane], bl = sb[(size_t)(nch * kC + kc) * 64 + lane];
                    bf16x8 h, l;
                    split8<XLO>(raw[c][0], raw[c][1], h, l);
                    if constexpr (XLO) acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(l, bh, acc, 0, 0, 0);
                    acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(h, bl, acc, 0, 0, 0);
                    acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(h, bh, acc, 0, 0, 0);
                }
            };
            for (int ch = 0; ch < nch; ch += 2) {
                load(rb, T, ch + 1);
                step(ra, ch);
                load(ra, T, ch + 2);
                step(rb, ch + 1);
            }
            float xn[16];
#pragma unroll
            for (int r4 = 0; r4 < 4; ++r4) {
                xn[r4 * 4 + 0] = xv[r4].x;
                xn[r4 * 4 + 1] = xv[r4].y;
                xn[r4 * 4 + 2] = xv[r4].z;
                xn[r4 * 4 + 3] = xv[r4].w;
            }
            const uint32_t m = split_pass<METRIC>(acc, xn, qn, rtau, a.coef, tile_rows_ok(rows - T * 32, half));
            if (__ballot(m != 0) == 0) continue;
            const uint32_t cg = (uint32_t)__builtin_popcount(m);
            if (cg) {
                uint32_t at = atomicAdd(&a.scnt[qid], cg);
                uint64_t* out = a.sbuf + (size_t)qid * a.cap;
#pragma unroll
                for (int r = 0; r < 16; ++r)
                    if ((m >> r) & 1u) {
                        const int row = (r >> 2) * 8 + half * 4 + (r & 3);
                        if (at < a.cap)
                            out[at] = make_key(split_rank<METRIC>(acc[r], qn, xn[r]), (uint32_t)((T0 + T) * 32 + row));
                        ++at;
                    }
            }
        }
    }
}

// Bound on |approximate rank - exact chain rank| per unit of ||q||^2 +
// ||x||^2 (u = 2^-8, gamma_m = m 2^-24 / (1 - m 2^-24)), as coarse_coef:
//   the pieces' residuals and the dropped lo.lo product: 3 2^-16 (1 + u)^2
//   ||q|| ||x||; FP32 accumulation of 3 d products, whose magnitudes sum to at
//   most (1 + 2u)^2 ||q|| ||x||: gamma_{3d} of it, taken twice (any rounding
//   inside the matrix core's sums); norms and epilogue 8 2^-24 (||q||^2 +
//   ||x||^2); the chain's own error 2 gamma_{d+2} of it.
// Doubled for -2 q.x, halved by ||q|| ||x|| <= (||q||^2 + ||x||^2) / 2; the IP
// rank is within the same bound.  Scaled by 1.01 for the check's rounding.
float split_coef(int64_t d) {
    const double u = 1.0 / 256.0, e = 1.0 / 16777216.0;
    auto gamma = [&](double m) { return m * e / (1.0 - m * e); };
    return (float)(1.01 * (3 * std::ldexp(1.0, -16) * (1 + u) * (1 + u) + 2 * gamma(3.0 * d) * (1 + 2 * u) * (1 + 2 * u) +
                           8 * e + 2 * gamma(d + 2.0)));
}

// Every step-th tile (a wave each, a row per lane): the workgroup's rows with
// w ||x||^2 above their squared distance to the list's centroid, and (high word) all
// rows asked, into its word of out (those on their centroid tell nothing).
// At most kWideTiles tiles: a list's first search waits for them (1024 of 128 dims with
// an atomic per tile 44 us).
constexpr int kWideTiles = 256;
__global__ __launch_bounds__(256) void wide_rows_kernel(DevLists lists, const float* __restrict__ norms,
                                                        const float4* __restrict__ cent, int nlist, int64_t tiles,
                                                        int64_t step, float w, unsigned long long* __restrict__ out) {
    __shared__ unsigned long long votes[4];
    const int lane = threadIdx.x & 63, wave = threadIdx.x / 64;
    const int64_t T = ((int64_t)blockIdx.x * 4 + wave) * step;
    unsigned long long v = 0;
    if (T < tiles) {            // whole wave
        int l = 0, hi = nlist;  // the last list that starts at T or before
        while (hi - l > 1) {
            const int mid = (l + hi) / 2;
            if (lists.list_tile_off[mid] <= T) l = mid;
            else hi = mid;
        }
        const int rows = lists.list_size[l] - (int)(T - lists.list_tile_off[l]) * 64;
        float dist = 0.0f;
        const float4 *c = cent + (size_t)l * lists.nquad, *x = lists.codes + (size_t)T * lists.nquad * 64 + lane;
#pragma unroll 8
        for (int j = 0; j < lists.nquad; ++j) dist = accum<kL2>(dist, c[j], x[(size_t)j * 64]);
        const bool on = lane < rows && dist > 0.0f && dist < FLT_MAX;
        v = (unsigned long long)__popcll(__ballot(on)) << 32 |
            (unsigned)__popcll(__ballot(on && w * norms[T * 64 + lane] > dist));
    }
    if (lane == 0) votes[wave] = v;
    __syncthreads();
    if (threadIdx.x == 0) out[blockIdx.x] = votes[0] + votes[1] + votes[2] + votes[3];
}

// 32-row tiles per item (near-query items: half) of the two forms.
constexpr int kSplitTiles = 8;
constexpr int kSplitWgTiles = 32;

void launch_split(const SplitArgs& a, bool l2, bool xlo, int cus, hipStream_t s) {
    auto go = [&](auto metric, auto lo) {
        constexpr int M = decltype(metric)::value;
        constexpr bool X = decltype(lo)::value;
        if (a.nkc <= 4)
            hipLaunchKernelGGL((split_wave_kernel<M, 4, X>), dim3(cus * 4), dim3(kNT), 0, s, a);
        else if (a.nkc <= 8)
            hipLaunchKernelGGL((split_wave_kernel<M, 8, X>), dim3(cus * 2), dim3(kNT), 0, s, a);
        else
            hipLaunchKernelGGL((split_wg_kernel<M, X>), dim3(cus * 2), dim3(kSplitWgNT), (size_t)((a.nkc + 2 * kSplitChunks - 1) / (2 * kSplitChunks) * 2 * kSplitChunks) * 2048, s, a);
    };
    using std::integral_constant;
    if (l2 && xlo) go(integral_constant<int, kL2>{}, integral_constant<bool, true>{});
    else if (l2) go(integral_constant<int, kL2>{}, integral_constant<bool, false>{});
    else if (xlo) go(integral_constant<int, kIP>{}, integral_constant<bool, true>{});
    else go(integral_constant<int, kIP>{}, integral_constant<bool, false>{});
}

}  // namespace
}  // namespace hivf
