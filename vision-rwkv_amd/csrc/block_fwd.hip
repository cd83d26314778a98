// Inference of one whole VRWKV / VRWKV6 block on few tokens: one entry point issues the block's kernels, with the
// projections on matrix cores here, several of them in one launch and the element-wise steps around them in their epilogues.
//
// A block of one 224 x 224 image (196 tokens) is 16 (VRWKV) or 26 (VRWKV6) operator calls of 2-20 us of GPU work each, and a call
// through the Python operators and the library costs about 20 us of host time, so the host sets the pace; on top the
// library picks tiles of 192 x 256 for 196 x 192 results (13 us a product).  Issued from here a VRWKV block is 9 launches, 7 on few tokens,
// where the norm and the shift behind it are one (ln_shift_mix.hip):
//   LN | shift + mixes | key, value, receptance | Bi-WKV with gate | output + residual
//   LN | shift + mixes | key with relu^2, receptance | value, gate, residual
// and 5 on fewer still, where the norm, the shift and the mixes are inside the projections of a half (linear_mix_kernel).
#include "linear.h"
#include "wave_sum.h"
#include <algorithm>
#include <type_traits>

namespace vrwkv {
namespace {

// ---- the projections ---------------------------------------------------------------------------------------------------
// out = epilogue(A W^T): A (M, K) with row pitch lda, W (N, K), out (M, N), of one type, with fp32 accumulation.  Both operands have
// the contraction index innermost, which is the order of the MFMA fragments (16 x 16 x 32: lane l holds row l & 15, eight
// k from 8 (l >> 4)), so they go from global memory to registers in 16-byte pieces without a stage in LDS.  At these sizes
// everything lies in the L2s and latency counts: a workgroup owns a tile of (16 MT)^2 results, its four waves take every
// fourth slice of 64 bytes of k each with D slices requested ahead, and add up through LDS in a fixed order.  The weights are the
// first operand, so a lane ends up with four neighbouring channels of a token: 8-byte accesses in the epilogue.
using gemm::f32x4;
using gemm::u32x4;
// one 16-byte fragment of either operand: 32 k in 16 bits; in fp32 16 k as four products of 4, lane group g taking the k
// 4 g .. of both operands
template <typename IO> __device__ __forceinline__ f32x4 mfma(u32x4 a, u32x4 b, f32x4 c) {
    if constexpr (std::is_same<IO, float>::value) {
        const f32x4 fa = __builtin_bit_cast(f32x4, a), fb = __builtin_bit_cast(f32x4, b);   // (of one element it takes element 0)
#pragma unroll
        for (int e = 0; e < 4; ++e) c = __builtin_amdgcn_mfma_f32_16x16x4f32(fa[e], fb[e], c, 0, 0, 0);
        return c;
    } else {
        return gemm::mfma16<IO>(a, b, c);
    }
}

// epilogue of four neighbouring channels n .. of token m
template <typename IO>
__device__ __forceinline__ void finish(const LinProblem& P, int m, int n, f32x4 s) {
    float v[4] = {s[0], s[1], s[2], s[3]};
    epilogue<IO, 4>(P, m, n, v);
    store_vec<IO, 4>((IO*)P.out + (size_t)m * P.N + n, v);
}

template <typename IO, int MT>
__global__ __launch_bounds__(256)
void linear_group_kernel(LinGroup G)
{
    constexpr int TILE = 16 * MT, D = MT == 4 ? 2 : 3;
    constexpr unsigned ES = sizeof(IO);
    __shared__ f32x4 red[4][MT * MT][WAVE];
    const int lane = threadIdx.x & 63, g4 = lane >> 4, c16 = lane & 15;
    const int w4 = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    int q = 0;
    while (q + 1 < G.n && (int)blockIdx.x >= G.p[q + 1].tile0) ++q;
    const LinProblem& P = G.p[q];
    const int N = P.N, K = P.K, M = G.M, nt = (N + TILE - 1) / TILE;
    const int tile = (int)blockIdx.x - P.tile0, m0 = tile / nt * TILE, n0 = tile % nt * TILE;
    // rows past M or N lie outside the descriptors and read 0
    const __amdgpu_buffer_rsrc_t rsa = make_rsrc(P.a, ((unsigned)(M - 1) * P.lda + K) * ES), rsw = make_rsrc(P.w, (unsigned)N * K * ES);
    unsigned oa[MT], ow[MT];
#pragma unroll
    for (int i = 0; i < MT; ++i) {
        oa[i] = (unsigned)(m0 + 16 * i + c16) * P.lda * ES + 16u * g4;
        ow[i] = (unsigned)(n0 + 16 * i + c16) * K * ES + 16u * g4;
    }
    u32x4 fa[D][MT], fw[D][MT];
    auto fetch = [&](int s, int d) {
#pragma unroll
        for (int i = 0; i < MT; ++i) {
            fw[d][i] = BufRaw<16>::ld(rsw, ow[i], 64u * s);
            fa[d][i] = BufRaw<16>::ld(rsa, oa[i], 64u * s);
        }
    };
    f32x4 acc[MT][MT];
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int j = 0; j < MT; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
    const int steps = K * ES / 64;
#pragma unroll
    for (int d = 0; d < D; ++d)
        if (w4 + 4 * d < steps) fetch(w4 + 4 * d, d);
    for (int s = w4; s < steps; s += 4 * D) {
#pragma unroll
        for (int d = 0; d < D; ++d) {
            const int cur = s + 4 * d;
            if (cur >= steps) break;                      // wave-uniform
#pragma unroll
            for (int i = 0; i < MT; ++i)
#pragma unroll
                for (int j = 0; j < MT; ++j) acc[i][j] = mfma<IO>(fw[d][j], fa[d][i], acc[i][j]);
            if (cur + 4 * D < steps) fetch(cur + 4 * D, d);
        }
    }
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int j = 0; j < MT; ++j) red[w4][i * MT + j][lane] = acc[i][j];
    __syncthreads();
    for (int t = w4; t < MT * MT; t += 4) {
        const int m = m0 + 16 * (t / MT) + c16, n = n0 + 16 * (t % MT) + 4 * g4;
        if (m >= M || n >= N) continue;
        finish<IO>(P, m, n, (red[0][t][lane] + red[1][t][lane]) + (red[2][t][lane] + red[3][t][lane]));
    }
}

// A pre-norm half's first steps inside the projections that take them: problem q multiplies mix q of LayerNorm(x) and its shifted rows.  On few tokens
// the launch in front (ln_shift_mix.hip) waits for its rows and sums, this one for its operands, and the host for either.  A workgroup owns 16 tokens x 64
// results: it normalises the rows that the mix of its tokens reads, those and the steps up and down around (a wave every fourth row, or pair of rows where
// half a wave holds one), forms the mix in LDS, rounded as the separate kernels round it and in their order, and every wave multiplies it with 16 rows of
// the weights, requested at the start.  What it costs is the rows normalised again by every workgroup of a token's results.
struct MixIn {
    const void *x, *ln_w, *ln_b;
    const float* mix;
    int T, Hp, Wp, shift, g, head_dim;
    float eps;
};
constexpr int MIX_TOKENS = 16, MIX_COLS = 64, MIX_ROWS = 64;     // of a workgroup; most rows that it normalises
__host__ __device__ inline unsigned mix_pitch(int C, unsigned es) { return C * es + 16u; }     // (16 more: rows begin in distinct banks)

template <typename IO, bool PAIRS>
__global__ __launch_bounds__(256)
void linear_mix_kernel(LinGroup G, MixIn X)
{
    constexpr int V = 16 / (int)sizeof(IO), RW = PAIRS ? 8 : 4, U = MIX_ROWS / RW, D = 6;
    constexpr unsigned ES = sizeof(IO);
    extern __shared__ __attribute__((aligned(16))) unsigned char rows[];
    const int lane = threadIdx.x & 63, g4 = lane >> 4, c16 = lane & 15;
    const int w4 = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    int q = 0;
    while (q + 1 < G.n && (int)blockIdx.x >= G.p[q + 1].tile0) ++q;
    const LinProblem& P = G.p[q];
    const int N = P.N, C = P.K, M = G.M, nt = N / MIX_COLS, nvec = C / V;
    const int tile = (int)blockIdx.x - P.tile0, m0 = tile / nt * MIX_TOKENS, n0 = tile % nt * MIX_COLS + 16 * w4;
    const int reach = X.shift * X.Wp, lo = max(m0 - reach, 0), R = min(m0 + MIX_TOKENS + reach, M) - lo;
    const unsigned pitch = mix_pitch(C, ES);
    unsigned char* const mixed = rows + (MIX_TOKENS + 2 * reach) * pitch;
    // ---- everything is requested together ----
    const int piece = PAIRS ? lane & 31 : lane, sub = PAIRS ? 2 * w4 + (lane >> 5) : w4;
    const __amdgpu_buffer_rsrc_t rsx = make_rsrc(X.x, (unsigned)M * C * ES), rsw = make_rsrc(P.w, (unsigned)N * C * ES);
    u32x4 raw[U];
#pragma unroll
    for (int i = 0; i < U; ++i) {
        raw[i] = u32x4{0u, 0u, 0u, 0u};
        if (RW * i < R) raw[i] = BufRaw<16>::ld(rsx, piece < nvec && RW * i + sub < R ? (unsigned)(lo + RW * i + sub) * C * ES + 16u * piece : OOB_OFFSET, 0);
    }
    nt_u32x4 lw = {0u, 0u, 0u, 0u}, lb = lw;
    if (piece < nvec) {
        lw = load_raw16<false>((const IO*)X.ln_w + piece * V);
        lb = load_raw16<false>((const IO*)X.ln_b + piece * V);
    }
    const unsigned ow = (unsigned)(n0 + c16) * C * ES + 16u * g4;
    const int steps = C * (int)ES / 64;
    u32x4 fw[D];
#pragma unroll
    for (int d = 0; d < D; ++d) fw[d] = BufRaw<16>::ld(rsw, d < steps ? ow : OOB_OFFSET, 64u * d);
    // ---- LayerNorm ----
    auto row_sum = [&](float x) {                         // as wave_sum; over the row's half wave where two share a wave
        x = dpp_add<0x140>(dpp_add<0x141>(dpp_add<0x4E>(dpp_add<0xB1>(x))));
        const int xi = __builtin_bit_cast(int, x);
        const float r0 = __builtin_bit_cast(float, __builtin_amdgcn_readlane(xi, 0)), r1 = __builtin_bit_cast(float, __builtin_amdgcn_readlane(xi, 16)),
                    r2 = __builtin_bit_cast(float, __builtin_amdgcn_readlane(xi, 32)), r3 = __builtin_bit_cast(float, __builtin_amdgcn_readlane(xi, 48));
        return PAIRS ? (lane < 32 ? r0 + r1 : r2 + r3) : (r0 + r1) + (r2 + r3);
    };
    float lnw[V], lnb[V];
    widen_raw16<IO, V>(lw, lnw);
    widen_raw16<IO, V>(lb, lnb);
#pragma unroll
    for (int i = 0; i < U; ++i) {
        if (RW * i >= R) break;
        float v[V], s = 0.f, sq = 0.f;
        widen_raw16<IO, V>(__builtin_bit_cast(nt_u32x4, raw[i]), v);
#pragma unroll
        for (int e = 0; e < V; ++e) s += v[e];
        const float mean = row_sum(s) / (float)C;
        if (piece < nvec) {
#pragma unroll
            for (int e = 0; e < V; ++e) { const float d = v[e] - mean; sq = fmaf(d, d, sq); }
        }
        const float rstd = rsqrtf(row_sum(sq) / (float)C + X.eps);
        IO n[V];
#pragma unroll
        for (int e = 0; e < V; ++e) n[e] = from_f32<IO>(fmaf((v[e] - mean) * rstd, lnw[e], lnb[e]));
        if (piece < nvec && RW * i + sub < R) __builtin_memcpy(rows + (RW * i + sub) * pitch + 16 * piece, n, 16);
    }
    __syncthreads();
    // ---- the mix of the 16 tokens: a thread keeps its token and takes every sixteenth piece ----
    {
        const int m = m0 + (threadIdx.x & 15), t = m % X.T, y0 = t / X.Wp, x0 = t % X.Wp;
        const bool in = t < X.Hp * X.Wp;                  // (a class token stands alone)
        const unsigned char* const own = rows + (m - lo) * pitch;
        for (int p = threadIdx.x >> 4; p < nvec; p += 16) {
            const int c = p * V, cq = X.head_dim > 0 ? c % X.head_dim : c, dir = X.g > 0 && cq < 4 * X.g ? cq / X.g : 4;
            nt_u32x4 out = {0u, 0u, 0u, 0u};
            if (m < M) {
                const bool moved = in && dir < 4;
                const bool there = !moved || (dir == 0 ? x0 >= X.shift : dir == 1 ? x0 + X.shift < X.Wp : dir == 2 ? y0 >= X.shift : y0 + X.shift < X.Hp);
                const int step = !moved || !there ? 0 : dir == 0 ? -X.shift : dir == 1 ? X.shift : dir == 2 ? -reach : reach;
                float xs[V], xx[V], mu[V];
                widen_raw16<IO, V>(*reinterpret_cast<const nt_u32x4*>(own + 16 * p), xs);
                widen_raw16<IO, V>(*reinterpret_cast<const nt_u32x4*>(own + step * (int)pitch + 16 * p), xx);
#pragma unroll
                for (int e = 0; e < V; e += 4) {
                    const float4 f = *reinterpret_cast<const float4*>(X.mix + (size_t)q * C + c + e);
                    mu[e] = f.x; mu[e + 1] = f.y; mu[e + 2] = f.z; mu[e + 3] = f.w;
                }
                IO o[V];
#pragma unroll
                for (int e = 0; e < V; ++e) {
                    const float x = there ? xx[e] : 0.f;
                    o[e] = from_f32<IO>(xs[e] * mu[e] + x * (1.f - mu[e]));
                }
                __builtin_memcpy(&out, o, 16);
            }
            *reinterpret_cast<nt_u32x4*>(mixed + (threadIdx.x & 15) * pitch + 16 * p) = out;
        }
    }
    __syncthreads();
    // ---- the products; slices of k in the order of linear_group_kernel: four sums over every fourth ----
    f32x4 acc[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) acc[i] = f32x4{0.f, 0.f, 0.f, 0.f};
    for (int s0 = 0; s0 < steps; s0 += 2 * D) {
#pragma unroll
        for (int d = 0; d < 2 * D; ++d) {
            const int s = s0 + d;
            if (s >= steps) break;                        // uniform
            const u32x4 fa = *reinterpret_cast<const u32x4*>(mixed + c16 * pitch + 64 * s + 16 * g4);
            acc[d & 3] = mfma<IO>(fw[d % D], fa, acc[d & 3]);
            if (s + D < steps) fw[d % D] = BufRaw<16>::ld(rsw, ow, 64u * (s + D));
        }
    }
    const int m = m0 + c16;
    if (m < M) finish<IO>(P, m, n0 + 4 * g4, (acc[0] + acc[1]) + (acc[2] + acc[3]));
}

// The same with 128 x 128 tiles staged in LDS, for 16-bit calls that fill enough compute units with them: 64 x 64 tiles read
// every operand piece twice as often straight from the L2s (three of 3136 x 768 x 768: 43 us, with these 21 us).
template <typename IO>
__global__ __launch_bounds__(256, 2)
void linear_tile_kernel(LinGroup G)
{
    __shared__ __attribute__((aligned(16))) char lds[gemm::Stage<false>::LDS];
    const int lane = threadIdx.x & 63, g4 = lane >> 4, c16 = lane & 15, w4 = threadIdx.x >> 6;
    // a contiguous eighth of the tiles per XCD: tiles of the same tokens share an L2
    int id = blockIdx.x;
    const int whole = gridDim.x / 8 * 8;
    if (id < whole) id = (id & 7) * (whole / 8) + (id >> 3);
    int q = 0;
    while (q + 1 < G.n && id >= G.p[q + 1].tile0) ++q;
    const LinProblem& P = G.p[q];
    const int nt = (P.N + gemm::TILE - 1) / gemm::TILE, tile = id - P.tile0;
    const int m0 = tile / nt * gemm::TILE, n0 = tile % nt * gemm::TILE;
    gemm::f32x4 acc[4][4];
    gemm::tile_product<IO, false>(lds, (const IO*)P.w, (const IO*)P.a, n0, m0, P.N, G.M, P.K, P.K, P.lda, 0, (P.K + 63) / 64, acc);
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const int n = n0 + 64 * (w4 & 1) + 16 * i + 4 * g4, m = m0 + 64 * (w4 >> 1) + 16 * j + c16;
            if (m < G.M && n < P.N) finish<IO>(P, m, n, acc[i][j]);
        }
}

int number_tiles(LinGroup& G, int side) {
    int tiles = 0;
    for (int i = 0; i < G.n; ++i) {
        G.p[i].tile0 = tiles;
        tiles += ((G.M + side - 1) / side) * ((G.p[i].N + side - 1) / side);
    }
    return tiles;
}
template <int MT>
void launch_group(LinGroup& G, int dtype, hipStream_t st) {
    const int tiles = number_tiles(G, 16 * MT);
    if constexpr (MT == 8) {
        if (dtype == VRWKV_BF16) hipLaunchKernelGGL((linear_tile_kernel<__hip_bfloat16>), dim3(tiles), dim3(256), 0, st, G);
        else hipLaunchKernelGGL((linear_tile_kernel<__half>), dim3(tiles), dim3(256), 0, st, G);
    } else if (dtype == VRWKV_BF16) hipLaunchKernelGGL((linear_group_kernel<__hip_bfloat16, MT>), dim3(tiles), dim3(256), 0, st, G);
    else if (dtype == VRWKV_F16) hipLaunchKernelGGL((linear_group_kernel<__half, MT>), dim3(tiles), dim3(256), 0, st, G);
    else hipLaunchKernelGGL((linear_group_kernel<float, MT>), dim3(tiles), dim3(256), 0, st, G);
}
}  // namespace

// Kernel and tile by the number of results: larger tiles read less from the L2s, smaller ones give more workgroups and shorten the chain
// of a wave.  64 x 64 from 128 tiles of that size on, 32 x 32 likewise; from 70 tiles of 128 x 128 on the wide kernel where it applies, else
// 128 x 128.  (Between 70 and 256 such tiles the two are alike on rows that lie in the caches, as below, but inside a block, where they do not,
// the wide kernel with its loads further ahead is faster: twelve blocks of 1568 x 768 1686 -> 1490 us, 12544 x 192 1322 -> 1160.)  us in bf16 with tiles of 16 / 32 / 64 / 128 / the wide kernel:
//   784 x 192 x 192   3.2  3.1  4.6  6.6  7.3     784 x 768 x 768     16.3 11.0  9.2 12.9 13.4     784 x 3072 x 768      55   34   26   40   37
//   three of them     5.6  4.7  4.9  6.9  7.7     three of them       39.7 24.0 15.6 14.2 14.6     1568 x 768 x 768      28.1 16.5 14.9 13.5 14.1
//   6272 x 192 x 192, three  -  -   12.3 10.0  9.4 3136 x 384 x 384, three   -  -  17.2 10.7 11.6  6272 x 768 x 768      -    -    31.3 19.2 15.2
//   3136 x 768 x 768  -    -   20.4 14.0 14.3     three of them       -    -   43.1 21.1 17.4      12544 x 768 x 768 three  -  -   158  64.1 52.5
// (M x K x N)
int linear_group(LinGroup& G, int dtype, hipStream_t st) {
    long long area = 0;
    for (int i = 0; i < G.n; ++i) area += (long long)G.M * G.p[i].N;
    const int force = option(OPT_LINEAR_TILE);
    const bool wide = dtype != VRWKV_F32;                // 128 x 128 tiles and wider ones are for 16 bits
    if ((force ? force == 16 : area >= 128LL * 128 * 70) && wide_takes(G, dtype)) return wide_group(G, dtype, st);
    const int mt = force && (wide || force < 8) ? std::min(force, 8)
                   : wide ? (area >= 128LL * 128 * 70 ? 8 : area >= 64LL * 64 * 128 ? 4 : area >= 32LL * 32 * 128 ? 2 : 1)
                          : (area >= 64LL * 64 * 256 ? 4 : area >= 32LL * 32 * 128 ? 2 : 1);
    if (mt == 8) launch_group<8>(G, dtype, st);
    else if (mt == 4) launch_group<4>(G, dtype, st);
    else if (mt == 2) launch_group<2>(G, dtype, st);
    else launch_group<1>(G, dtype, st);
    return check_launch("linear_group");
}
namespace {
// 16-bit rows of few tokens: the rows normalised again grow with tokens, channels and results alike.  Twelve blocks, two launches / this one, us (the host
// sets the pace of the small ones): 196 x 192 511 / 456 (replayed as a graph 424 / 383), 784 x 192 522 / 475, 1568 x 192 668 / 642, 3136 x 192 842 / 881;
// 196 x 384 547 / 530, 392 x 384 601 / 607, 784 x 384 764 / 903; fp32 196 x 192 584 / 585, 784 x 192 618 / 635.
constexpr long long LINEAR_MIX_PAIRS = 58000000, LINEAR_MIX_WIDE = 30000000;   // tokens x channels^2, with two rows a wave and with one
bool linear_mix_takes(const LinGroup& G, const MixIn& X, int C, int dtype) {
    const int es = 2, V = 16 / es, period = X.head_dim > 0 ? X.head_dim : C;
    if (dtype == VRWKV_F32 || option(OPT_LINEAR_TILE) || C / V > WAVE || (long long)G.M * C * C > (C / V <= 32 ? LINEAR_MIX_PAIRS : LINEAR_MIX_WIDE) || C % V || X.g < 0 || X.g % V || period % V || 4LL * X.g > period || C % period) return false;
    if (X.shift < 0 || X.Wp <= 0 || X.Hp <= 0 || X.shift > X.Wp || ((long long)X.Hp * X.Wp != X.T && (long long)X.Hp * X.Wp != X.T - 1)) return false;
    for (int i = 0; i < G.n; ++i)
        if (G.p[i].N % MIX_COLS) return false;
    const long long rows = MIX_TOKENS + 2LL * X.shift * X.Wp;
    return rows <= MIX_ROWS && (rows + MIX_TOKENS) * mix_pitch(C, es) <= 64 * 1024;
}
template <typename IO>
void launch_mix(LinGroup& G, const MixIn& X, int C, hipStream_t st) {
    int tiles = 0;
    for (int i = 0; i < G.n; ++i) {
        G.p[i].tile0 = tiles;
        tiles += (G.M + MIX_TOKENS - 1) / MIX_TOKENS * (G.p[i].N / MIX_COLS);
    }
    const unsigned lds = (2 * MIX_TOKENS + 2 * X.shift * X.Wp) * mix_pitch(C, sizeof(IO));
    if (C * (int)sizeof(IO) / 16 <= 32) hipLaunchKernelGGL((linear_mix_kernel<IO, true>), dim3(tiles), dim3(256), lds, st, G, X);
    else hipLaunchKernelGGL((linear_mix_kernel<IO, false>), dim3(tiles), dim3(256), lds, st, G, X);
}
int linear_mix(LinGroup& G, const MixIn& X, int C, int dtype, hipStream_t st) {
    if (dtype == VRWKV_BF16) launch_mix<__hip_bfloat16>(G, X, C, st);
    else launch_mix<__half>(G, X, C, st);
    return check_launch("linear_mix");
}

LinProblem linear(const void* a, const void* w, void* out, int N, int K, int lda = 0, int epi = 0) {
    return LinProblem{a, w, out, nullptr, nullptr, nullptr, N, K, lda ? lda : K, epi, 0, nullptr};
}

// ---- the block -----------------------------------------------------------------------------------------------------------
size_t al(size_t bytes) { return (bytes + 255) & ~(size_t)255; }
// token tensors of C channels that live at the same time: LN result, up to six mixes, x after the attention half, and the
// operator's tensors
struct Layout { size_t n, hidden, op, weights, total; };
Layout layout(int B, int T, int C, int hidden, int heads, int dtype) {
    Layout l;
    const size_t es = dtype == VRWKV_F32 ? 4 : 2;
    l.n = al((size_t)B * T * C * es);
    l.hidden = al((size_t)B * T * hidden * es);
    l.op = heads ? al(vrwkv_wkv6_fwd_workspace_bytes(B, T, C, heads)) : al(vrwkv_biwkv_fwd_workspace_bytes(B, T, C, dtype));
    // VRWKV: 9 tensors; VRWKV6: x1, LN, sx, xxx, five mixes, five maps (later r, k, v, w, gate), two fp32 tensors, low-rank rows
    const size_t tokens = heads ? 2 + 2 + 5 + 5 + 4 : 9;
    const size_t low = heads ? al((size_t)B * T * 160 * es) + al((size_t)B * T * 64 * es) : 0;
    l.weights = heads ? al((size_t)448 * C * es) + al((size_t)12 * C * sizeof(float)) : 0;   // (see weights6_kernel)
    l.total = tokens * l.n + 2 * l.hidden + low + l.op + l.weights;       // (hidden rows twice: before and after their norm)
    return l;
}

// ---- VRWKV6: the weights that the block wants otherwise than the modules hold them -----------------------------------------
// The low-rank matrices with the contraction index innermost (32 x 32 tiles turned through LDS) and the vectors in fp32.  Formed
// in every call, so that a write to a parameter leaves nothing behind: 448 C values, one launch of 3 us (twelve blocks of 784 x 768
// bf16 1953 -> 1990 us, of 196 x 192 893 -> 935, against copies kept between calls).  160 C of them are maa_w2, which only fp32 blocks and
// a misaligned maa_w2 read: the mixes of 16-bit ones take the matrix as it lies.
// Grid: 14 C / 32 tiles, then C / 256 (rounded up) workgroups for the vectors.
struct Weights6 {
    vrwkv_block6_params p;
    void *maa_w1, *maa_w2, *decay_w1, *decay_w2;
    float *att_mix, *ffn_mix, *maa, *u, *kn_w, *kn_b;
};
template <typename IO>
__global__ __launch_bounds__(256)
void weights6_kernel(Weights6 W, int C)
{
    __shared__ IO tile[32][33];
    const int per = C / 32;
    int id = blockIdx.x;
    if (id >= 14 * per) {
        const int c = (id - 14 * per) * 256 + threadIdx.x;
        if (c >= C) return;
        auto get = [&](const void* p, int bit) { return W.p.fp32_vectors >> bit & 1 ? ((const float*)p)[c] : to_f32(((const IO*)p)[c]); };
        const float x = 1.f - get(W.p.maa_x, 0);          // rounded to its own type, like the tensor operation
        W.att_mix[c] = 0.f;
        W.att_mix[C + c] = W.p.fp32_vectors & 1 ? x : to_f32(from_f32<IO>(x));
        for (int i = 0; i < 5; ++i) W.maa[i * C + c] = get(W.p.maa[i], 1 + i);
        W.ffn_mix[c] = get(W.p.ffn_mix_k, 6);
        W.ffn_mix[C + c] = get(W.p.ffn_mix_r, 7);
        W.u[c] = get(W.p.u, 8);
        if (W.p.att_kn_w) {
            W.kn_w[c] = to_f32(((const IO*)W.p.att_kn_w)[c]);
            W.kn_b[c] = to_f32(((const IO*)W.p.att_kn_b)[c]);
        }
        return;
    }
    const IO* src;
    IO* dst;
    int rows, cols, tr, tc;                               // the matrix as it lies, and the tile's place in it
    if (id < 5 * per) {
        src = (const IO*)W.p.maa_w1; dst = (IO*)W.maa_w1; rows = C; cols = 160; tr = id / 5; tc = id % 5;
    } else if ((id -= 5 * per) < 5 * per) {
        const size_t z = (size_t)(id / per) * 32 * C;
        src = (const IO*)W.p.maa_w2 + z; dst = (IO*)W.maa_w2 + z; rows = 32; cols = C; tr = 0; tc = id % per;
    } else if ((id -= 5 * per) < 2 * per) {
        src = (const IO*)W.p.decay_w1; dst = (IO*)W.decay_w1; rows = C; cols = 64; tr = id / 2; tc = id % 2;
    } else {
        id -= 2 * per;
        src = (const IO*)W.p.decay_w2; dst = (IO*)W.decay_w2; rows = 64; cols = C; tr = id / per; tc = id % per;
    }
    const int x = threadIdx.x & 31, y = threadIdx.x >> 5;
#pragma unroll
    for (int i = 0; i < 32; i += 8) tile[y + i][x] = src[(size_t)(32 * tr + y + i) * cols + 32 * tc + x];
    __syncthreads();
#pragma unroll
    for (int i = 0; i < 32; i += 8) dst[(size_t)(32 * tc + y + i) * rows + 32 * tr + x] = tile[x][y + i];
}

}  // namespace
}  // namespace vrwkv

#define TRY(call) do { const int rc_ = (call); if (rc_ != VRWKV_OK) return rc_; } while (0)

extern "C" size_t vrwkv_block_fwd_workspace_bytes(int B, int T, int C, int hidden, int heads, int dtype)
{
    if (B <= 0 || T <= 0 || C <= 0 || hidden <= 0 || heads < 0) return 0;
    return vrwkv::layout(B, T, C, hidden, heads, dtype).total;
}

static int block_fwd(const vrwkv_block_args* args, const vrwkv_block6_params* params, void* hip_stream)
{
    using namespace vrwkv;
    vrwkv_block_args with_params;
    const vrwkv_block_args* a = args;
    Weights6 W;
    if (args && params && args->heads > 0 && args->C > 0 && args->workspace) {
        // the fields that `params` stands for: the end of the workspace, filled below once the sizes are checked
        const size_t es = args->dtype == VRWKV_F32 ? 4 : 2, n = (size_t)args->C;
        const Layout L = layout(args->B, args->T, args->C, args->hidden, args->heads, args->dtype);
        char* m = (char*)args->workspace + L.total - L.weights;
        float* f = (float*)(m + al(448 * n * es));
        W = Weights6{*params, m, m + 160 * n * es, m + 320 * n * es, m + 384 * n * es, f, f + 2 * n, f + 4 * n, f + 9 * n, f + 10 * n, f + 11 * n};
        with_params = *args;
        a = &with_params;
        with_params.maa_w1 = W.maa_w1; with_params.maa_w2 = W.maa_w2; with_params.decay_w1 = W.decay_w1; with_params.decay_w2 = W.decay_w2;
        with_params.att_mix = W.att_mix; with_params.ffn_mix = W.ffn_mix; with_params.maa = W.maa; with_params.u = W.u;
        with_params.att_kn_w = params->att_kn_w ? W.kn_w : nullptr;
        with_params.att_kn_b = params->att_kn_b ? W.kn_b : nullptr;
        bool all = params->maa_w1 && params->maa_w2 && params->decay_w1 && params->decay_w2 && params->maa_x && params->ffn_mix_k &&
                   params->ffn_mix_r && params->u;
        for (const void* p : params->maa) all = all && p;
        if (!all) a = nullptr;
    }
    if (!a || !a->x || !a->out || !a->workspace || !a->ln1_w || !a->ln1_b || !a->ln2_w || !a->ln2_b || !a->att_mix || !a->ffn_mix ||
        !a->u || !a->key || !a->value || !a->receptance || !a->output || !a->ffn_key || !a->ffn_receptance || !a->ffn_value ||
        (a->heads ? !a->gate || !a->maa || !a->maa_w1 || !a->maa_w2 || !a->decay || !a->decay_w1 || !a->decay_w2 || !a->gn_w || !a->gn_b
                  : !a->w) ||
        (!a->att_kn_w != !a->att_kn_b) || (!a->ffn_kn_w != !a->ffn_kn_b)) {
        set_error("block_fwd: null pointer argument");
        return VRWKV_INVALID_ARG;
    }
    const int B = a->B, T = a->T, C = a->C, hidden = a->hidden, H = a->heads, dt = a->dtype;
    const size_t es = dt == VRWKV_F32 ? 4 : 2;
    if (dt != VRWKV_F32 && dt != VRWKV_BF16 && dt != VRWKV_F16) {
        set_error("block_fwd: unknown dtype %d", dt);
        return VRWKV_UNSUPPORTED_DTYPE;
    }
    const long long M = (long long)B * T;
    if (B <= 0 || T <= 0 || C <= 0 || C % 32 || hidden <= 0 || hidden % 32 || hidden > 16384 / (int)es || C > 8192 || H < 0 || (H && C != 64 * H) ||
        M * std::max({C, hidden, 160}) * (long long)es >= (1LL << 30) || (long long)C * hidden * (long long)es >= (1LL << 30)) {
        set_error("block_fwd: unsupported sizes (B=%d T=%d C=%d hidden=%d heads=%d)", B, T, C, hidden, H);
        return VRWKV_UNSUPPORTED_SHAPE;
    }
    const void* aligned[] = {a->x, a->out, a->workspace, a->ln1_w, a->ln1_b, a->ln2_w, a->ln2_b, a->gamma1, a->gamma2, a->key, a->value, a->receptance,
                             a->output, a->att_kn_w, a->att_kn_b, a->ffn_key, a->ffn_receptance, a->ffn_value, a->ffn_kn_w, a->ffn_kn_b,
                             a->gate, a->maa_w1, a->maa_w2, a->decay, a->decay_w1, a->decay_w2, a->gn_w, a->gn_b, a->w, a->u, a->att_mix, a->ffn_mix, a->maa};
    for (const void* p : aligned)
        if ((size_t)p & 15) {
            set_error("block_fwd: every tensor must be 16-byte aligned");
            return VRWKV_INVALID_ARG;
        }
    const Layout L = layout(B, T, C, hidden, H, dt);
    if (a->workspace_bytes < L.total) {
        set_error("block_fwd: workspace of %zu bytes, %zu needed", a->workspace_bytes, L.total);
        return VRWKV_WORKSPACE_TOO_SMALL;
    }
    char* at = (char*)a->workspace;
    auto take = [&](size_t bytes) { void* p = at; at += bytes; return p; };
    hipStream_t st = static_cast<hipStream_t>(hip_stream);
    if (a != args) {
        const dim3 grid((unsigned)(14 * (C / 32) + (C + 255) / 256)), block(256);
        if (dt == VRWKV_F32) hipLaunchKernelGGL((weights6_kernel<float>), grid, block, 0, st, W, C);
        else if (dt == VRWKV_BF16) hipLaunchKernelGGL((weights6_kernel<__hip_bfloat16>), grid, block, 0, st, W, C);
        else hipLaunchKernelGGL((weights6_kernel<__half>), grid, block, 0, st, W, C);
        TRY(check_launch("block_fwd (weights)"));
    }
    const int hd = H ? 64 : 0;
    void *x1 = take(L.n), *ln = take(L.n), *hid = take(L.hidden), *hid_raw = take(L.hidden), *op_ws = take(L.op);
    LinGroup G;
    G.M = (int)M;
    // branch -> x: gamma * branch + x in the projection's epilogue, or with the post-norm in a row kernel
    auto residual = [&](LinProblem p, const void* x, void* out, const void* gamma, const void* w, const void* b, float eps, void* tmp) {
        G.n = 1;
        if (!a->post_norm) { p.vec = gamma; p.res = x; p.out = out; }
        else p.out = tmp;
        G.p[0] = p;
        TRY(linear_group(G, dt, st));
        return a->post_norm ? vrwkv_rowfuse(tmp, x, w, b, gamma, out, M, C, 0, 2, eps, dt, st) : (int)VRWKV_OK;
    };

    const void* x = a->x;
    const void* src = x;                                  // input of a half
    // a half's first steps: the pre-norm, the shift and the mixes; `keep`: the normalised rows are wanted as well
    const int g = H ? 16 : a->quarter;
    auto mixes = [&](const void* in, const void* w, const void* b, float eps, const float* mix, void* const* out, int n, bool keep) -> int {
        if (a->post_norm) return vrwkv_qshift_mix(in, mix, out, n, B, T, C, a->Hp, a->Wp, a->shift_pixel, g, hd, dt, st);
        if (ln_shift_mix_takes(B, T, C, g, hd, a->shift_pixel, dt))
            return ln_shift_mix(in, w, b, eps, mix, out, n, keep ? ln : nullptr, B, T, C, a->Hp, a->Wp, a->shift_pixel, g, hd, dt, st);
        TRY(vrwkv_rowfuse(in, nullptr, w, b, nullptr, ln, M, C, 0, 0, eps, dt, st));
        return vrwkv_qshift_mix(ln, mix, out, n, B, T, C, a->Hp, a->Wp, a->shift_pixel, g, hd, dt, st);
    };
    // ... and the projections of the mixes, in one launch where that is the faster way (problem i takes mix i)
    auto mixed = [&](const void* in, const void* w, const void* b, float eps, const float* mix, void* const* out) -> int {
        const MixIn X{in, w, b, mix, T, a->Hp, a->Wp, a->shift_pixel, g, hd, eps};
        const int asked = option(OPT_LINEAR_MIX);
        if (!a->post_norm && asked != 2 && linear_mix_takes(G, X, C, dt)) return linear_mix(G, X, C, dt, st);
        if (asked == 1) {
            set_error("block_fwd: norm, shift and mixes are not inside the projections of this call");
            return VRWKV_UNSUPPORTED_SHAPE;
        }
        TRY(mixes(in, w, b, eps, mix, out, G.n, false));
        return linear_group(G, dt, st);
    };
    if (!a->post_norm) src = ln;
    char* half = at;                                      // both halves use what follows
    void* y;
    if (!H) {
        void* m[3] = {take(L.n), take(L.n), take(L.n)};
        void *k = take(L.n), *v = take(L.n), *r = take(L.n);
        G.n = 3;
        G.p[0] = linear(m[0], a->key, k, C, C);
        G.p[1] = linear(m[1], a->value, v, C, C);
        G.p[2] = linear(m[2], a->receptance, r, C, C);
        TRY(mixed(x, a->ln1_w, a->ln1_b, a->ln1_eps, a->att_mix, m));
        y = m[0];
        if (a->att_kn_w) {
            TRY(vrwkv_biwkv_fwd(a->w, a->u, k, v, m[1], B, T, C, dt, L.op ? op_ws : nullptr, L.op, st));
            TRY(vrwkv_rowfuse(m[1], r, a->att_kn_w, a->att_kn_b, nullptr, y, M, C, 0, 1, a->att_kn_eps, dt, st));
        } else {
            TRY(vrwkv_biwkv_fwd_gate(a->w, a->u, k, v, r, y, B, T, C, dt, L.op ? op_ws : nullptr, L.op, st));
        }
    } else {
        void* s[2] = {take(L.n), take(L.n)};              // shifted x, the mix that feeds the low-rank maps
        char* maps = at;
        void* five[5];
        for (void*& p : five) p = take(L.n);
        void* m[5];
        for (void*& p : m) p = take(L.n);
        float *yf = (float*)take(2 * L.n), *yn = (float*)take(2 * L.n);
        void *lo = take(al((size_t)M * 160 * es)), *dlo = take(al((size_t)M * 64 * es));
        TRY(mixes(x, a->ln1_w, a->ln1_b, a->ln1_eps, a->att_mix, s, 2, true));
        G.n = 1;
        G.p[0] = linear(s[1], a->maa_w1, lo, 160, C, 0, EPI_TANH);
        TRY(linear_group(G, dt, st));
        if (params && dt != VRWKV_F32 && !((uintptr_t)params->maa_w2 & 15)) {         // w, k, v, r, g, the five maps formed inside
            TRY(vrwkv_maa_lora_mix(src, s[0], lo, params->maa_w2, a->maa, m, M, C, dt, st));
        } else {
            G.n = 5;
            for (int i = 0; i < 5; ++i)                   // the five maps as one (5, M, C) tensor
                G.p[i] = linear((const char*)lo + 32 * es * i, (const char*)a->maa_w2 + (size_t)i * C * 32 * es, maps + (size_t)i * M * C * es, C, 32, 160);
            TRY(linear_group(G, dt, st));
            TRY(vrwkv_maa_mix(src, s[0], maps, a->maa, m, M, C, dt, st));
        }
        G.n = 5;
        G.p[0] = linear(m[0], a->decay_w1, dlo, 64, C, 0, EPI_TANH);
        G.p[1] = linear(m[1], a->key, five[1], C, C);
        G.p[2] = linear(m[2], a->value, five[2], C, C);
        G.p[3] = linear(m[3], a->receptance, five[3], C, C);
        G.p[4] = linear(m[4], a->gate, five[4], C, C);
        TRY(linear_group(G, dt, st));
        G.n = 1;
        G.p[0] = linear(dlo, a->decay_w2, five[0], C, 64, 0, EPI_ADD_VEC);
        G.p[0].vec = a->decay;
        TRY(linear_group(G, dt, st));
        TRY(vrwkv_wkv6_fwd(five[3], five[1], five[2], five[0], a->u, yf, B, T, C, H, dt, dt, 0, L.op ? op_ws : nullptr, L.op, st));
        if (a->att_kn_w) {
            TRY(vrwkv_rowfuse(yf, nullptr, a->att_kn_w, a->att_kn_b, nullptr, yn, M, C, 0, 0, a->att_kn_eps, VRWKV_F32, st));
            yf = yn;
        }
        y = m[0];
        TRY(vrwkv_groupnorm_gate(yf, five[4], a->gn_w, a->gn_b, y, M, C, 64, a->gn_eps, VRWKV_F32, dt, st));
    }
    TRY(residual(linear(y, a->output, nullptr, C, C), x, x1, a->gamma1, a->ln1_w, a->ln1_b, a->ln1_eps, ln));
    at = half;
    void *f[2] = {take(L.n), take(L.n)}, *fr = take(L.n), *ftmp = take(L.n);
    G.n = 2;
    G.p[0] = linear(f[0], a->ffn_key, a->ffn_kn_w ? hid_raw : hid, hidden, C, 0, a->ffn_kn_w ? 0 : EPI_RELU_SQ);
    G.p[1] = linear(f[1], a->ffn_receptance, fr, C, C);
    TRY(mixed(x1, a->ln2_w, a->ln2_b, a->ln2_eps, a->ffn_mix, f));
    if (a->ffn_kn_w) TRY(vrwkv_rowfuse(hid_raw, nullptr, a->ffn_kn_w, a->ffn_kn_b, nullptr, hid, M, hidden, 1, 0, a->ffn_kn_eps, dt, st));
    LinProblem p = linear(hid, a->ffn_value, nullptr, C, hidden);
    p.gate = fr;
    return residual(p, x1, a->out, a->gamma2, a->ln2_w, a->ln2_b, a->ln2_eps, ftmp);
}

extern "C" int vrwkv_linear_group(const vrwkv_linear* problems, int n, int M, int dtype, void* hip_stream)
{
    using namespace vrwkv;
    if (!problems || n <= 0 || n > LIN_MAX) {
        set_error("linear_group: null argument, or not 1 to %d problems", LIN_MAX);
        return VRWKV_INVALID_ARG;
    }
    if (dtype != VRWKV_F32 && dtype != VRWKV_BF16 && dtype != VRWKV_F16) {
        set_error("linear_group: unknown dtype %d", dtype);
        return VRWKV_UNSUPPORTED_DTYPE;
    }
    LinGroup G;
    G.n = n;
    G.M = M;
    const long long es = dtype == VRWKV_F32 ? 4 : 2;
    for (int i = 0; i < n; ++i) {
        const vrwkv_linear& p = problems[i];
        if (!p.a || !p.w || !p.out || (((size_t)p.a | (size_t)p.w | (size_t)p.out | (size_t)p.gate | (size_t)p.vec | (size_t)p.res | (size_t)p.raw) & 15)) {
            set_error("linear_group: null or misaligned (16 bytes) pointer argument");
            return VRWKV_INVALID_ARG;
        }
        if (M <= 0 || p.N <= 0 || p.K <= 0 || p.N % 16 || p.K % 32 || p.lda < p.K || p.lda % 8 || (M + 256LL) * std::max(p.lda, p.N) * es >= (1LL << 30) ||
            (p.N + 256LL) * p.K * es >= (1LL << 30)) {
            set_error("linear_group: unsupported sizes (M=%d N=%d K=%d lda=%d)", M, p.N, p.K, p.lda);
            return VRWKV_UNSUPPORTED_SHAPE;
        }
        if (p.epi & ~(EPI_RELU_SQ | EPI_TANH | EPI_ADD_VEC | EPI_RELU_SQ_BWD | EPI_ROUND) || (p.epi & EPI_RELU_SQ_BWD && !p.gate)) {
            set_error("linear_group: unknown epilogue %d", p.epi);
            return VRWKV_INVALID_ARG;
        }
        G.p[i] = LinProblem{p.a, p.w, p.out, p.gate, p.vec, p.res, p.N, p.K, p.lda, p.epi, 0, p.raw};
    }
    return linear_group(G, dtype, static_cast<hipStream_t>(hip_stream));
}

extern "C" int vrwkv_block_fwd(const vrwkv_block_args* args, void* hip_stream) { return block_fwd(args, nullptr, hip_stream); }

extern "C" int vrwkv_block6_fwd(const vrwkv_block_args* args, const vrwkv_block6_params* params, void* hip_stream)
{
    if (!args || !params || args->heads <= 0) {
        vrwkv::set_error("block6_fwd: null argument or no heads");
        return VRWKV_INVALID_ARG;
    }
    return block_fwd(args, params, hip_stream);
}
