// Scan of the FP16 shadow past 128 dims (included by batched.hip): a workgroup
// per item of up to 64 queries, whose fragments of all dim chunks are staged in
// LDS once per item (2 KB per 16 dims, up to 64 KB).  A wave takes 64 rows at a
// time, straight from the shadow, against all of them: four products per pair
// of LDS reads and pair of row loads.
//
// What bounds it: the shadow's bytes through L2 and the latency of an item's
// set-up.  With a wave per 32 queries, all of whose fragments and a tile's rows
// sit in registers (256, one wave per SIMD), each tile is read for 32 queries and
// nothing hides its loads: 2000 queries of 420 dims at nprobe 50 830 us, now 711;
// 1200 of 300 dims 424 and 391, 1500 of 150 dims 329 and 302, 40 of 200 dims 164
// and 165.  (MFMA 21 % busy, 9 TB/s from L2.)
#pragma once

namespace hivf {
namespace {

constexpr int kShadowItem = 64;

// Chunks that an item's loop runs over: two groups of four at a time.
__host__ __device__ inline int shadow_chunks(int nkc) { return (nkc + 7) / 8 * 8; }

__global__ __launch_bounds__(kNT) __attribute__((amdgpu_waves_per_eu(2))) void shadow_wg_kernel(BatchArgs a) {
    extern __shared__ bf16x8 sb[];  // [group][kC nch][64 lanes], zeros past nkc
    __shared__ uint32_t s_it;
    __shared__ int s_q[kShadowItem];
    constexpr int kW = kNT / 64, kC = 4;
    const int tid = threadIdx.x, lane = tid & 63, half = lane >> 5, slot = lane & 31;
    const int wv = __builtin_amdgcn_readfirstlane(tid / 64);
    const int nkc = a.nkc;
    const int nch = shadow_chunks(nkc) / kC;
    int grp = blockIdx.x % kXcds, switches = 0;         // (thread 0's)
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
        const int nq = __builtin_amdgcn_readfirstlane(w.nq & 0xFFFF);
        const int ng = nq > 32 ? 2 : 1;
        const int list = __builtin_amdgcn_readfirstlane(w.list);
        const int nrows = a.list_size[list];
        const int64_t G0 = (int64_t)a.list_tile_off[list] * 2;
        const int t0 = __builtin_amdgcn_readfirstlane(w.t0);
        const int te = min((nrows + 31) >> 5, t0 + __builtin_amdgcn_readfirstlane(w.nq >> 16));
        if (tid < kShadowItem) s_q[tid] = tid < nq ? a.lq[w.q0 + tid] : -1;
        bf16x8 ra[2][kC], rb[2][kC];
        // chunk group ch of tiles T and T + 1 (past the last: of the wave's next pair)
        auto load = [&](bf16x8 (&raw)[2][kC], int T, int ch) {
            if (ch >= nch) {
                ch -= nch;
                T += 2 * kW;
            }
#pragma unroll
            for (int t = 0; t < 2; ++t) {
                const int64_t G = G0 + min(T + t, te - 1);
                const bf16x8* xa = reinterpret_cast<const bf16x8*>(a.xbf) + G * nkc * 64 + lane;
                // (no branch: with one, every product waits for all loads in
                // flight.  Past nkc the last chunk meets zeros.)
#pragma unroll
                for (int c = 0; c < kC; ++c) raw[t][c] = xa[min(ch * kC + c, nkc - 1) * 64];
            }
        };
        if (t0 + 2 * wv < te) load(ra, t0 + 2 * wv, 0);
        __syncthreads();
        for (int e = tid; e < ng * nch * kC * 64; e += kNT) {
            const int l = e & 63, g = (e >> 6) >= nch * kC, kc = (e >> 6) - g * nch * kC;
            const int q = max(s_q[g * 32 + (l & 31)], 0);
            const bf16x8 z = {};
            sb[e] = kc < nkc ? *reinterpret_cast<const bf16x8*>(a.qbf + (size_t)q * a.dpad16 + kc * 16 + (l >> 5) * 8) : z;
        }
        int qid[2];
        float qn[2], tau[2];
#pragma unroll
        for (int g = 0; g < 2; ++g) {
            qid[g] = s_q[g * 32 + slot];
            qn[g] = a.qnorm[max(qid[g], 0)];
            tau[g] = qid[g] >= 0 ? a.tau[qid[g]] + a.mabs : -FLT_MAX;
        }
        __syncthreads();
        for (int T = t0 + 2 * wv; T < te; T += 2 * kW) {
            floatx16 acc[2][2];
#pragma unroll
            for (int t = 0; t < 2; ++t)
#pragma unroll
                for (int g = 0; g < 2; ++g) acc[t][g] = floatx16{};
            float4 xv[2][4];
#pragma unroll
            for (int t = 0; t < 2; ++t)
#pragma unroll
                for (int r4 = 0; r4 < 4; ++r4)
                    xv[t][r4] = *reinterpret_cast<const float4*>(a.norms + (G0 + min(T + t, te - 1)) * 32 + r4 * 8 + half * 4);
            auto step = [&](const bf16x8 (&raw)[2][kC], int ch) {
#pragma unroll
                for (int c = 0; c < kC; ++c) {
                    const bf16x8 b0 = sb[(ch * kC + c) * 64 + lane];
                    acc[0][0] = mfma16<true>(raw[0][c], b0, acc[0][0]);
                    acc[1][0] = mfma16<true>(raw[1][c], b0, acc[1][0]);
                    if (ng == 2) {
                        const bf16x8 b1 = sb[((nch + ch) * kC + c) * 64 + lane];
                        acc[0][1] = mfma16<true>(raw[0][c], b1, acc[0][1]);
                        acc[1][1] = mfma16<true>(raw[1][c], b1, acc[1][1]);
                    }
                }
            };
            for (int ch = 0; ch < nch; ch += 2) {
                load(rb, T, ch + 1);
                step(ra, ch);
                load(ra, T, ch + 2);
                step(rb, ch + 1);
            }
#pragma unroll
            for (int g = 0; g < 2; ++g) {
                if (g >= ng) break;
                uint32_t m[2];
#pragma unroll
                for (int t = 0; t < 2; ++t) {
                    m[t] = 0;
#pragma unroll
                    for (int r = 0; r < 16; ++r) {
                        const float4 x4 = xv[t][r >> 2];
                        const float sn = qn[g] + ((r & 3) == 0 ? x4.x : (r & 3) == 1 ? x4.y : (r & 3) == 2 ? x4.z : x4.w);
                        const float dist = __builtin_fmaf(a.dot_scale, acc[t][g][r], sn);
                        acc[t][g][r] = dist;
                        m[t] |= (__builtin_fmaf(-a.mcoef, sn, dist) <= tau[g] ? 1u : 0u) << r;
                    }
                    // (an absent query's slot holds another's fragments, not finite perhaps)
                    m[t] &= qid[g] >= 0 && T + t < te ? tile_rows_ok(nrows - (T + t) * 32, half) : 0u;
                }
                const uint32_t cnt = (uint32_t)__builtin_popcount(m[0]) + (uint32_t)__builtin_popcount(m[1]);
                if (cnt == 0) continue;
                uint32_t at = atomicAdd(&a.scnt[qid[g]], cnt);
                uint64_t* out = a.sbuf + (size_t)qid[g] * a.cap;
#pragma unroll
                for (int t = 0; t < 2; ++t)
#pragma unroll
                    for (int r = 0; r < 16; ++r)
                        if ((m[t] >> r) & 1u) {
                            const int row = (r >> 2) * 8 + half * 4 + (r & 3);
                            if (at < a.cap) out[at] = make_key(acc[t][g][r], (uint32_t)((G0 + T + t) * 32 + row));
                            ++at;
                        }
            }
        }
    }
}

}  // namespace
}  // namespace hivf
