// Warm-up bound of a batched search from its 16- or 8-bit shadow (included by
// batched.hip): a value >= the k-th distance over the first rows of a query's
// nearest lists, hence >= its k-th distance.  Int8 shadow: exact integer
// distances (the rows nearest to their centroids come first); a query of such
// a batch that is not integer runs the FP32 chain.  FP16 shadow: the
// approximate distance plus its error bound.
//
// What bounds it: the rows' bytes through L2 and the vector instructions of the
// FP32 chain (256 per 64 rows and 128 dims), a quarter of both with v_dot4 on
// int8, a half and a quarter with v_dot2 on FP16.  Against the FP32 scan: 4096
// queries on skewed integer lists 170 -> 43 us (that search 456 -> 313), 2000 of
// 420 dims 160 -> 101 (902 -> 832), 1200 of 300 dims and k 150 560 -> 426, 8000
// of an integer list 390 -> 333.
#pragma once

namespace hivf {
namespace {

constexpr int kWarmSlots = 4096;  // rows of one query (whole 32-row tiles)
constexpr int kWarmLists = 128;

struct WarmArgs {
    DevLists lists;
    const float4* q;        // [nq x nquad]
    const int32_t* probes;  // [nq x P]
    int P;
    const int32_t* npq;
    int L, W, k;            // rows: the first W of each of the first L lists
    const int32_t* qint;    // int8: the query holds integers in [0, 255]
    const i32x4* x8;
    const int32_t* xn8;     // negated row norms
    const int8_t* q8;
    const int32_t* qn8;
    int dpad32;
    const uint16_t* xbf;    // FP16
    const uint16_t* qbf;
    const float* norms;
    const float* qnorm;
    int nkc, dpad16;
    float dot_scale, mcoef, mabs;
    float* out;             // [nq]
};

// One workgroup per query.  NKC8: 32-dim chunks of the int8 shadow, 0: FP16.
template <int NKC8>
__global__ __launch_bounds__(kNT) void warm_kernel(WarmArgs a) {
    constexpr int kW = kNT / 64;
    __shared__ float v[kWarmSlots];
    __shared__ __align__(16) uint32_t hist[256];
    __shared__ int s_tile[kWarmLists], s_rows[kWarmLists], s_before[kWarmLists + 1];
    __shared__ float s_red[2][kW];
    __shared__ uint32_t s_fin[kW];
    __shared__ __align__(16) uint16_t sq[NKC8 == 0 ? 512 : 1];
    const int tid = threadIdx.x, lane = tid & 63, half = lane >> 5, row = lane & 31;
    const int wv = __builtin_amdgcn_readfirstlane(tid / 64);
    const int qi = blockIdx.x;
    const int L = min(a.L, a.npq ? min(a.npq[qi], a.P) : a.P);
    if (tid < L) {
        const int l = a.probes[(size_t)qi * a.P + tid];
        s_rows[tid] = l >= 0 ? min(a.lists.list_size[l], a.W) : 0;
        s_tile[tid] = l >= 0 ? a.lists.list_tile_off[l] * 2 : 0;
    }
    if constexpr (NKC8 == 0) {
        for (int c = tid; c < a.dpad16 / 8; c += kNT)
            reinterpret_cast<uint4*>(sq)[c] = reinterpret_cast<const uint4*>(a.qbf + (size_t)qi * a.dpad16)[c];
    }
    __syncthreads();
    if (tid <= L) {
        int b = 0;
        for (int u = 0; u < tid; ++u) b += (s_rows[u] + 31) >> 5;
        s_before[tid] = b;
    }
    for (int i = tid; i < 256; i += kNT) hist[i] = 0;
    __syncthreads();
    const int total = L > 0 ? s_before[L] : 0;
    // tile g (of all lists'): its place in the arena and the rows it holds
    auto place = [&](int g, int& j, int& rows) {
        while (s_before[j + 1] <= g) ++j;
        rows = __builtin_amdgcn_readfirstlane(s_rows[j] - (g - s_before[j]) * 32);
        return __builtin_amdgcn_readfirstlane(s_tile[j] + g - s_before[j]);
    };
    // (lanes past a tile's rows read its last row again: no bytes for them; 2000
    // queries of 420 dims, 100 rows of each list, 661 us, now 652)
    auto lane_of = [&](int rows) { return half * 32 + min(row, rows - 1); };
    if (NKC8 > 0 && a.qint[qi]) {
        constexpr int K = NKC8 > 0 ? NKC8 : 1;
        const i32x4* qa = reinterpret_cast<const i32x4*>(a.q8 + (size_t)qi * a.dpad32 + half * 16);
        i32x4 y[K];
#pragma unroll
        for (int c = 0; c < K; ++c) y[c] = qa[c * 2];
        const int qn = a.qn8[qi];
        int j = 0, rows[2];
        for (int g = wv; g < total; g += 2 * kW) {  // two tiles' loads in flight
            i32x4 x[2][K];
            int xn[2];
#pragma unroll
            for (int u = 0; u < 2; ++u) {
                const int G = place(min(g + u * kW, total - 1), j, rows[u]);
#pragma unroll
                for (int c = 0; c < K; ++c) x[u][c] = a.x8[((int64_t)G * K + c) * 64 + lane_of(rows[u])];
                xn[u] = a.xn8[(int64_t)G * 32 + row];
            }
#pragma unroll
            for (int u = 0; u < 2; ++u) {
                int dot = 0;
#pragma unroll
                for (int c = 0; c < K; ++c)
#pragma unroll
                    for (int w = 0; w < 4; ++w) dot = __builtin_amdgcn_sdot4(x[u][c][w], y[c][w], dot, false);
                dot += __shfl_xor(dot, 32);
                // (exact, below 2^24)
                if (half == 0 && g + u * kW < total)
                    v[(g + u * kW) * 32 + row] = row < rows[u] ? (float)(qn - (2 * dot + xn[u])) : INFINITY;
            }
        }
    } else if constexpr (NKC8 > 0) {
        int j = 0, rows;
        for (int g = wv; g < total; g += kW) {
            const int G = place(g, j, rows);
            const float4* tp = a.lists.codes + (size_t)(G >> 1) * a.lists.nquad * 64 + (G & 1) * 32 + min(row, rows - 1);
            const float4* q = a.q + (size_t)qi * a.lists.nquad;
            float acc = 0.0f;
#pragma unroll 8
            for (int c = 0; c < a.lists.nquad; ++c) acc = accum<kL2>(acc, q[c], tp[(size_t)c * 64]);
            if (half == 0) v[g * 32 + row] = row < rows && acc < FLT_MAX ? acc : INFINITY;
        }
    } else {
        typedef __attribute__((ext_vector_type(2))) _Float16 f16x2;
        const float qn = a.qnorm[qi];
        int j = 0, rows;
        for (int g = wv; g < total; g += kW) {
            const int G = place(g, j, rows);
            const uint4* xa = reinterpret_cast<const uint4*>(a.xbf) + (int64_t)G * a.nkc * 64 + lane_of(rows);
            const uint4* qa = reinterpret_cast<const uint4*>(sq) + half;
            const float sn = qn + a.norms[(int64_t)G * 32 + row];
            float dot = 0.0f;
#pragma unroll 8
            for (int c = 0; c < a.nkc; ++c) {
                const uint4 x = xa[c * 64], y = qa[c * 2];
                dot = __builtin_amdgcn_fdot2(__builtin_bit_cast(f16x2, x.x), __builtin_bit_cast(f16x2, y.x), dot, false);
                dot = __builtin_amdgcn_fdot2(__builtin_bit_cast(f16x2, x.y), __builtin_bit_cast(f16x2, y.y), dot, false);
                dot = __builtin_amdgcn_fdot2(__builtin_bit_cast(f16x2, x.z), __builtin_bit_cast(f16x2, y.z), dot, false);
                dot = __builtin_amdgcn_fdot2(__builtin_bit_cast(f16x2, x.w), __builtin_bit_cast(f16x2, y.w), dot, false);
            }
            dot += __shfl_xor(dot, 32);
            const float u = __builtin_fmaf(a.dot_scale, dot, sn) + __builtin_fmaf(a.mcoef, sn, a.mabs);
            if (half == 0) v[g * 32 + row] = row < rows && u < FLT_MAX ? u : INFINITY;
        }
    }
    __syncthreads();
    // the k-th smallest, from above: the largest value of the bins up to its
    // own in a 256-bin histogram whose k-th's bin is split by a second one
    const int slots = total * 32;
    float mn = INFINITY, mx = -INFINITY;
    uint32_t fin = 0;
    for (int i = tid; i < slots; i += kNT)
        if (v[i] < FLT_MAX) {
            mn = fminf(mn, v[i]);
            mx = fmaxf(mx, v[i]);
            ++fin;
        }
    mn = wave_min(mn);
    mx = wave_max(mx);
    for (int off = 32; off > 0; off >>= 1) fin += __shfl_xor(fin, off);
    if (lane == 0) {
        s_red[0][wv] = mn;
        s_red[1][wv] = mx;
        s_fin[wv] = fin;
    }
    __syncthreads();
    fin = 0;
#pragma unroll
    for (int w = 0; w < kW; ++w) {
        mn = fminf(mn, s_red[0][w]);
        mx = fmaxf(mx, s_red[1][w]);
        fin += s_fin[w];
    }
    if (fin < (uint32_t)a.k) {  // (uniform) fewer rows than k: no bound
        if (tid == 0) a.out[qi] = FLT_MAX;
        return;
    }
    const float w1 = (mx - mn) * (1.0f / 256.0f);
    const float inv1 = w1 > 0.0f ? 1.0f / w1 : 0.0f;
    for (int i = tid; i < slots; i += kNT)
        if (v[i] < FLT_MAX) atomicAdd(&hist[lin_bin(v[i], mn, inv1)], 1u);
    __syncthreads();
    uint32_t need = (uint32_t)a.k;
    const int b1 = wave_find_bin(hist, &need, lane);
    __syncthreads();
    for (int i = tid; i < 256; i += kNT) hist[i] = 0;
    __syncthreads();
    const float lo2 = mn + (float)b1 * w1, inv2 = w1 > 0.0f ? 256.0f / w1 : 0.0f;
    for (int i = tid; i < slots; i += kNT)
        if (v[i] < FLT_MAX && lin_bin(v[i], mn, inv1) == b1) atomicAdd(&hist[lin_bin(v[i], lo2, inv2)], 1u);
    __syncthreads();
    const int b2 = wave_find_bin(hist, &need, lane);
    float top = -INFINITY;
    for (int i = tid; i < slots; i += kNT)
        if (v[i] < FLT_MAX) {
            const int b = lin_bin(v[i], mn, inv1);
            if (b < b1 || (b == b1 && lin_bin(v[i], lo2, inv2) <= b2)) top = fmaxf(top, v[i]);
        }
    top = wave_max(top);
    if (lane == 0) s_red[0][wv] = top;  // (mn, mx: read before the barriers above)
    __syncthreads();
    if (tid == 0) {
        for (int w = 1; w < kW; ++w) top = fmaxf(top, s_red[0][w]);
        a.out[qi] = fmaxf(top, 0.0f);
    }
}

// Whether the L lists' first W rows fit the kernel.
bool warm_fits(int64_t L, int64_t W) { return L <= kWarmLists && L * ((W + 31) / 32) * 32 <= kWarmSlots; }

}  // namespace
}  // namespace hivf
