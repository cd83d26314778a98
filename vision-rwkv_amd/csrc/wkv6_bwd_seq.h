// wkv6 backward, sequential sweeps (exact for any decay; what the chunked kernel leaves a sequence to when a chunk decays
// beyond its range).  Three sweeps per pass, each a sequential 64x64-state scan like the forward's exact kernel: one
// 256-thread workgroup per (b,h); a lane owns one "own" index and a 16-wide slice of the other index, quads finish the
// contractions with two quad-permute adds; each wave stages the rows of a token in its own LDS slot, so the token loop has
// no workgroup barrier.
//   sweep S (ascending)   own = key j:    S  -> gr, a (workspace), gu partial
//   sweep G (descending)  own = key j:    G  -> gk, gw
//   sweep V (descending)  own = value i:  G^T -> gv
// DIR 1 (descending pass) writes its results, DIR 0 (ascending, with the bonus) adds.  Every sweep maps (token, channel) to
// the same thread as the sweep it depends on, so program order is enough between them.
#pragma once
#include "wkv6_chunk_common.h"

namespace vrwkv {
namespace wkv6_detail {

constexpr int SEQ_STAGE_FLOATS = 4 * 3 * HN;         // LDS: three rows per wave in every sweep (the waves run on unsynchronised)

template <typename T> __device__ __forceinline__ float ldf(const T* p, size_t o) { return to_f32(p[o]); }
__device__ __forceinline__ float quad_sum(float x) {
    x += __shfl_xor(x, 1);
    x += __shfl_xor(x, 2);
    return x;
}
__device__ __forceinline__ void lds_order() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}
template <typename WT, bool W_IS_EW>
__device__ __forceinline__ float log_decay(const WT* w_, size_t o) {
    const float w = to_f32(w_[o]);
    return W_IS_EW ? w : -__expf(w);
}

// ---- sweep S: state S, own = j ----------------------------------------------------------------
template <typename IO, typename WT, int DIR, bool W_IS_EW>
__device__ __forceinline__
void seq_sweep_s(int bh, const IO* __restrict__ r_, const IO* __restrict__ k_, const IO* __restrict__ v_,
                      const WT* __restrict__ w_, const float* __restrict__ u_, const float* __restrict__ gy_,
                      float* __restrict__ gr_, float* __restrict__ a_, float* __restrict__ gu_part,
                      float* __restrict__ stage, int T, int C, int H)
{
    float (*s_row)[3][HN] = reinterpret_cast<float (*)[3][HN]>(stage);   // [wave][v, gy][i]
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6) & 3;
    const int b = bh / H, h = bh % H;
    const int sq = lane & 3, j = wave * 16 + (lane >> 2);
    const size_t base = (size_t)b * T * C + (size_t)h * HN;
    const float uj = DIR == 0 ? u_[h * HN + j] : 0.f;
    float S[16];
#pragma unroll
    for (int e = 0; e < 16; ++e) S[e] = 0.f;
    float gu = 0.f;
    for (int n = 0; n < T; ++n) {
        const int t = DIR == 0 ? n : T - 1 - n;
        const size_t o = base + (size_t)t * C;
        s_row[wave][0][lane] = ldf(v_, o + lane);
        s_row[wave][1][lane] = gy_[o + lane];
        const float rj = ldf(r_, o + j), kj = ldf(k_, o + j), dj = __expf(log_decay<WT, W_IS_EW>(w_, o + j));
        lds_order();
        float dot = 0.f, sg = 0.f;
#pragma unroll
        for (int q4 = 0; q4 < 4; ++q4) {
            const float4 v4 = *reinterpret_cast<const float4*>(&s_row[wave][0][sq * 16 + q4 * 4]);
            const float4 g4 = *reinterpret_cast<const float4*>(&s_row[wave][1][sq * 16 + q4 * 4]);
            const float vv[4] = {v4.x, v4.y, v4.z, v4.w}, gg[4] = {g4.x, g4.y, g4.z, g4.w};
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                float& s = S[q4 * 4 + e];
                dot = fmaf(vv[e], gg[e], dot);
                sg = fmaf(s, gg[e], sg);
                s = fmaf(s, dj, kj * vv[e]);
            }
        }
        dot = quad_sum(dot);
        sg = quad_sum(sg);
        if (sq == 0) {
            const float gr = uj * kj * dot + sg;
            if (DIR == 0) gr_[o + j] += gr; else gr_[o + j] = gr;
            a_[o + j] = rj * sg;
        }
        gu = fmaf(rj * kj, dot, gu);
        lds_order();
    }
    if (DIR == 0 && sq == 0) gu_part[j] = gu;
}

// ---- sweep G: adjoint G, own = j, descending in pass order ---------------------------------------
template <typename IO, typename WT, int DIR, bool W_IS_EW>
__device__ __forceinline__
void seq_sweep_g(int bh, const IO* __restrict__ r_, const IO* __restrict__ k_, const IO* __restrict__ v_,
                      const WT* __restrict__ w_, const float* __restrict__ u_, const float* __restrict__ gy_,
                      const float* __restrict__ a_, float* __restrict__ gk_, float* __restrict__ gw_,
                      float* __restrict__ stage, int T, int C, int H)
{
    float (*s_row)[3][HN] = reinterpret_cast<float (*)[3][HN]>(stage);
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6) & 3;
    const int b = bh / H, h = bh % H;
    const int sq = lane & 3, j = wave * 16 + (lane >> 2);
    const size_t base = (size_t)b * T * C + (size_t)h * HN;
    const float uj = DIR == 0 ? u_[h * HN + j] : 0.f;
    float G[16];
#pragma unroll
    for (int e = 0; e < 16; ++e) G[e] = 0.f;
    float X = 0.f;                                        // sum over later tokens of (a - b)
    for (int n = T - 1; n >= 0; --n) {
        const int t = DIR == 0 ? n : T - 1 - n;
        const size_t o = base + (size_t)t * C;
        s_row[wave][0][lane] = ldf(v_, o + lane);
        s_row[wave][1][lane] = gy_[o + lane];
        const float rj = ldf(r_, o + j), kj = ldf(k_, o + j), ew = log_decay<WT, W_IS_EW>(w_, o + j);
        const float dj = __expf(ew), an = a_[o + j];
        lds_order();
        float dot = 0.f, gvv = 0.f;
#pragma unroll
        for (int q4 = 0; q4 < 4; ++q4) {
            const float4 v4 = *reinterpret_cast<const float4*>(&s_row[wave][0][sq * 16 + q4 * 4]);
            const float4 g4 = *reinterpret_cast<const float4*>(&s_row[wave][1][sq * 16 + q4 * 4]);
            const float vv[4] = {v4.x, v4.y, v4.z, v4.w}, gg[4] = {g4.x, g4.y, g4.z, g4.w};
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                float& gq = G[q4 * 4 + e];
                dot = fmaf(vv[e], gg[e], dot);
                gvv = fmaf(gq, vv[e], gvv);
                gq = fmaf(gq, dj, rj * gg[e]);
            }
        }
        dot = quad_sum(dot);
        gvv = quad_sum(gvv);
        const float bn = kj * gvv;
        if (sq == 0) {
            const float gk = uj * rj * dot + gvv;
            const float gw = ew * (X - bn);
            if (DIR == 0) { gk_[o + j] += gk; gw_[o + j] += gw; } else { gk_[o + j] = gk; gw_[o + j] = gw; }
        }
        X += an - bn;
        lds_order();
    }
}

// ---- sweep V: adjoint G^T, own = i, descending in pass order --------------------------------------
template <typename IO, typename WT, int DIR, bool W_IS_EW>
__device__ __forceinline__
void seq_sweep_v(int bh, const IO* __restrict__ r_, const IO* __restrict__ k_,
                      const WT* __restrict__ w_, const float* __restrict__ u_, const float* __restrict__ gy_,
                      float* __restrict__ gv_, float* __restrict__ stage, int T, int C, int H)
{
    float (*s_row)[3][HN] = reinterpret_cast<float (*)[3][HN]>(stage);   // [wave][r, k, d][j]
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6) & 3;
    const int b = bh / H, h = bh % H;
    const int sq = lane & 3, i = wave * 16 + (lane >> 2);
    const size_t base = (size_t)b * T * C + (size_t)h * HN;
    float uu[16];
#pragma unroll
    for (int e = 0; e < 16; ++e) uu[e] = DIR == 0 ? u_[h * HN + sq * 16 + e] : 0.f;
    float G[16];
#pragma unroll
    for (int e = 0; e < 16; ++e) G[e] = 0.f;
    for (int n = T - 1; n >= 0; --n) {
        const int t = DIR == 0 ? n : T - 1 - n;
        const size_t o = base + (size_t)t * C;
        s_row[wave][0][lane] = ldf(r_, o + lane);
        s_row[wave][1][lane] = ldf(k_, o + lane);
        s_row[wave][2][lane] = __expf(log_decay<WT, W_IS_EW>(w_, o + lane));
        const float gyi = gy_[o + i];
        lds_order();
        float gv = 0.f;
#pragma unroll
        for (int q4 = 0; q4 < 4; ++q4) {
            const float4 r4 = *reinterpret_cast<const float4*>(&s_row[wave][0][sq * 16 + q4 * 4]);
            const float4 k4 = *reinterpret_cast<const float4*>(&s_row[wave][1][sq * 16 + q4 * 4]);
            const float4 d4 = *reinterpret_cast<const float4*>(&s_row[wave][2][sq * 16 + q4 * 4]);
            const float rr[4] = {r4.x, r4.y, r4.z, r4.w}, kk[4] = {k4.x, k4.y, k4.z, k4.w}, dd[4] = {d4.x, d4.y, d4.z, d4.w};
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                float& gq = G[q4 * 4 + e];
                const float rg = rr[e] * gyi;
                gv = fmaf(kk[e], fmaf(uu[q4 * 4 + e], rg, gq), gv);
                gq = fmaf(gq, dd[e], rg);
            }
        }
        gv = quad_sum(gv);
        if (sq == 0) {
            if (DIR == 0) gv_[o + i] += gv; else gv_[o + i] = gv;
        }
        lds_order();
    }
}

}  // namespace wkv6_detail
}  // namespace vrwkv
