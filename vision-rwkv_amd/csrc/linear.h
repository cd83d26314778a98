// A launch of several projections out = epilogue(A W^T), and the element-wise steps that follow them: shared by the kernels of
// the small tiles (block_fwd.hip) and the wide one (linear_wide.hip).
#pragma once
#include "gemm_tile.h"

namespace vrwkv {

// A (M, K) with row pitch lda, W (N, K), out (M, N), of one type, with fp32 accumulation.
enum { EPI_RELU_SQ = 1, EPI_TANH = 2, EPI_ADD_VEC = 4, EPI_RELU_SQ_BWD = 8, EPI_ROUND = 16 };
struct LinProblem {
    const void *a, *w;
    void* out;
    const void *gate, *vec, *res;   // all optional: v *= sigmoid(gate) (2 max(gate, 0) with EPI_RELU_SQ_BWD); v *= vec (or v += vec with EPI_ADD_VEC); v += res
    int N, K, lda, epi, tile0;
    void* raw;                      // optional: the product itself, beside the result.  EPI_ROUND: the steps above see it rounded to its type
};
constexpr int LIN_MAX = 5;
struct LinGroup {
    LinProblem p[LIN_MAX];
    int n, M;
};

// epilogue of V neighbouring channels n .. of token m, in place
template <typename IO, int V>
__device__ __forceinline__ void epilogue(const LinProblem& P, int m, int n, float (&v)[V]) {
    const IO *gate = (const IO*)P.gate, *vec = (const IO*)P.vec, *res = (const IO*)P.res;
    const size_t off = (size_t)m * P.N + n;
    float x[V];
    if (P.epi & EPI_ROUND) {
#pragma unroll
        for (int e = 0; e < V; ++e) v[e] = to_f32(from_f32<IO>(v[e]));
    }
    if (P.raw) store_vec<IO, V>((IO*)P.raw + off, v);
    if (P.epi & EPI_RELU_SQ) {
#pragma unroll
        for (int e = 0; e < V; ++e) { const float r = fmaxf(v[e], 0.f); v[e] = r * r; }
    }
    if (P.epi & EPI_TANH) {
#pragma unroll
        for (int e = 0; e < V; ++e) v[e] = tanhf(v[e]);
    }
    if (gate) {
        load_vec<IO, V>(gate + off, x);
#pragma unroll
        for (int e = 0; e < V; ++e) v[e] *= P.epi & EPI_RELU_SQ_BWD ? 2.f * fmaxf(x[e], 0.f) : fast_rcp(1.f + fast_exp2(-LOG2E * x[e]));
    }
    if (vec) {
        load_vec<IO, V>(vec + n, x);
#pragma unroll
        for (int e = 0; e < V; ++e) v[e] = P.epi & EPI_ADD_VEC ? v[e] + x[e] : v[e] * x[e];
    }
    if (res) {
        load_vec<IO, V>(res + off, x);
#pragma unroll
        for (int e = 0; e < V; ++e) v[e] += x[e];
    }
}

// Runs a group; picks kernel and tile by the size of the results (block_fwd.hip).  16-byte aligned pointers, N a multiple of 16, K of 32,
// lda of 8, byte offsets below 2^30: the callers' checks.
int linear_group(LinGroup& G, int dtype, hipStream_t st);
// LayerNorm, Q-Shift and two or three token mixes in one launch (ln_shift_mix.hip): whether it is the faster way, and the launch.  Tensors
// 16-byte aligned, x (B, T, C).  ln_out: optional, the normalised rows as well.
constexpr long long LN_SHIFT_MIX_MOST = 700000;          // values of x
bool ln_shift_mix_takes(int B, int T, int C, int g, int head_dim, int shift, int dtype);
int ln_shift_mix(const void* x, const void* ln_w, const void* ln_b, float eps, const float* mix, void* const* out, int n_mix, void* ln_out,
                 int B, int T, int C, int Hp, int Wp, int shift, int g, int head_dim, int dtype, hipStream_t st);
// The wide kernel (linear_wide.hip): whether it can run a group, and the launch.
bool wide_takes(const LinGroup& G, int dtype);
int wide_group(LinGroup& G, int dtype, hipStream_t st);

}  // namespace vrwkv
