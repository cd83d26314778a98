// The five data-dependent token mixes of VRWKV6 with the low-rank products inside (classification/mmcls_custom/models/backbones/vrwkv6.py:183-194):
//     m_i = lo_i w2_i,   out_i = x + (sx - x) * (maa_i + m_i),   i = w, k, v, r, g
// lo (rows, 5 x 32), w2 (5, 32, C).  vrwkv_maa_mix takes the five m_i from memory, where a batched product has left them: five token
// matrices written and read.  The contraction is 32 long, one matrix instruction, so here m_i is formed where it is used, rounded to the
// I/O type as the product's result was, and the backward forms it again instead of keeping it.
//
// What bounds both is memory.  A workgroup owns 64 channels and lays their columns of w2 down in LDS once, [channel][k] with 80-byte rows;
// a wave takes 16 tokens at a time.  The weights are the first operand, whose rows are handed out so that a lane ends up with
// channels 8 g4 .. + 7 and 32 + 8 g4 .. + 7 of one token (tile q, row r: channel 32 (q >> 1) + 8 (r >> 2) + 4 (q & 1) + (r & 3)): all
// accesses are 16 bytes, 64 in a row of a token.
// The backward's channel sums (gmaa): a transposing butterfly adds the 16 tokens of a wave and leaves one channel slot a lane, carried over a
// workgroup's tokens in five registers (80 sums a lane, added up at the end, spill); LDS adds the four waves, and one partial row per workgroup
// leaves for batch_sum_kernel.
//
// bf16, product and mix of their own -> here, forward | backward (the product's gradients come after it in either), us, results bit for bit
// the same: 12544 x 768 70 -> 38 | 89 -> 73     12544 x 384 40 -> 19 | 57 -> 36     12544 x 192 36 -> 13 | 27 -> 22     1568 x 768 19 -> 9 | 18 -> 16
// 196 x 192 20 -> 5 | 12 -> 9.  The bytes at 5 TB/s: 12544 x 768 28 | 54.
#include "gemm_tile.h"
#include "wkv6_chunk_common.h"
#include "../../include/vrwkv_hip.h"

namespace vrwkv {
namespace {

using gemm::f32x4;
using gemm::u32x4;
constexpr int LM_C = 64, LM_K = 32, LM_P = 40;         // channels of a workgroup, contraction length, row pitch in LDS
constexpr int LM_TOK = 64;                             // tokens of a step: four waves, 16 each
// Workgroups the token chunks are sized for, three and two rounds of what the registers let run at once: a workgroup lays down its weights while
// others move tokens.  One round instead, 12544 x 768: forward 46.7 -> 37.5 us, backward 82.3 -> 73.1; one step a workgroup the same.
constexpr int LM_WG = 3072, LM_WG_BWD = 1536;

struct LoraArgs {
    const void *x, *sx, *lo, *w2;
    const float* maa;
    const void* g[5];
    void *out[5], *gx, *gsx, *gm;
    float* part;
    long long rows;
    int C, steps;
};

template <typename IO> struct LoraLds {
    unsigned short W[5][LM_C][LM_P];
    float A[5][LM_C];
};

// the workgroup's columns of w2, [channel][k], and of the five vectors
template <typename IO>
__device__ __forceinline__ void stage(LoraLds<IO>& L, const LoraArgs& P, int c0) {
    // 16-byte pieces, neighbouring lanes at neighbouring k: their two-byte stores fall into neighbouring banks
    u32x4 piece[5];
#pragma unroll
    for (int i = 0; i < 5; ++i)
        piece[i] = *reinterpret_cast<const u32x4*>(static_cast<const unsigned short*>(P.w2) + (size_t)(LM_K * i + threadIdx.x % LM_K) * P.C + c0 + 8 * (threadIdx.x / LM_K));
#pragma unroll
    for (int i = 0; i < 5; ++i)
#pragma unroll
        for (int e = 0; e < 8; ++e) L.W[i][8 * (threadIdx.x / LM_K) + e][threadIdx.x % LM_K] = (unsigned short)(piece[i][e >> 1] >> (16 * (e & 1)));
    for (int q = threadIdx.x; q < 5 * LM_C; q += 256) L.A[q / LM_C][q % LM_C] = P.maa[(size_t)(q / LM_C) * P.C + c0 + q % LM_C];
    __syncthreads();
}

// maa_i + m_i of a lane's 16 channels: e < 8 channel 8 g4 + e, else 32 + 8 g4 + e - 8
template <typename IO>
__device__ __forceinline__ void factors(const LoraLds<IO>& L, int i, u32x4 lo, int lane, float (&f)[16]) {
    __builtin_amdgcn_sched_barrier(0);
    asm volatile("" : "+v"(lane));                         // read anew in every step: kept, the operands of five maps fill the registers
    const int g4 = lane >> 4, c16 = lane & 15;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        const int row = 32 * (q >> 1) + 8 * (c16 >> 2) + 4 * (q & 1) + (c16 & 3);
        const u32x4 w = *reinterpret_cast<const u32x4*>(&L.W[i][row][8 * g4]);
        const f32x4 m = gemm::mfma16<IO>(w, lo, f32x4{0.f, 0.f, 0.f, 0.f});
        const f32x4 a = *reinterpret_cast<const f32x4*>(&L.A[i][32 * (q >> 1) + 8 * g4 + 4 * (q & 1)]);
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            IO r = from_f32<IO>(m[e]);
            unsigned short bits;
            __builtin_memcpy(&bits, &r, 2);
            asm volatile("" : "+v"(bits));                 // a rounding to fp16 and back is contracted away otherwise
            __builtin_memcpy(&r, &bits, 2);
            f[4 * q + e] = a[e] + to_f32(r);
        }
    }
}

// a lane's 16 channels as they lie in memory, requested ahead of their use
struct Raw16 {
    u32x4 a, b;
};
template <typename IO>
__device__ __forceinline__ Raw16 fetch16(const void* p, size_t e0) {
    const IO* q = static_cast<const IO*>(p) + e0;
    return {*reinterpret_cast<const u32x4*>(q), *reinterpret_cast<const u32x4*>(q + 32)};
}
template <typename IO>
__device__ __forceinline__ void widen16(const Raw16& r, float (&v)[16]) {
    IO t[16];
    __builtin_memcpy(t, &r, 32);
#pragma unroll
    for (int e = 0; e < 16; ++e) v[e] = to_f32(t[e]);
}
template <typename IO>
__device__ __forceinline__ void store16(void* p, size_t e0, float (&v)[16]) {
    if constexpr (std::is_same<IO, __half>::value) {
        // fp32 values, as the other kernels round them: a mixed-precision multiply-add would round the exact sum to fp16 at once
#pragma unroll
        for (int e = 0; e < 16; ++e) asm volatile("" : "+v"(v[e]));
    }
    store_vec<IO, 8>(static_cast<IO*>(p) + e0, *reinterpret_cast<const float(*)[8]>(&v[0]));
    store_vec<IO, 8>(static_cast<IO*>(p) + e0 + 32, *reinterpret_cast<const float(*)[8]>(&v[8]));
}

template <typename IO>
__global__ __launch_bounds__(256)
void maa_lora_mix_kernel(LoraArgs P)
{
    __shared__ __attribute__((aligned(16))) LoraLds<IO> L;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, c0 = blockIdx.x * LM_C;
    stage<IO>(L, P, c0);
    for (int s = 0; s < P.steps; ++s) {
        const long long t = ((long long)blockIdx.y * P.steps + s) * LM_TOK + wave * 16 + (lane & 15);
        const long long tl = t < P.rows ? t : P.rows - 1;              // past the end: a valid row, not stored
        const size_t e0 = (size_t)tl * P.C + c0 + 8 * (lane >> 4);
        u32x4 lo[5];
#pragma unroll
        for (int i = 0; i < 5; ++i)
            lo[i] = *reinterpret_cast<const u32x4*>(static_cast<const IO*>(P.lo) + (size_t)tl * (5 * LM_K) + LM_K * i + 8 * (lane >> 4));
        const Raw16 xr = fetch16<IO>(P.x, e0), dr = fetch16<IO>(P.sx, e0);
        float x[16], d[16];
        widen16<IO>(xr, x);
        widen16<IO>(dr, d);
#pragma unroll
        for (int e = 0; e < 16; ++e) d[e] -= x[e];
#pragma unroll
        for (int i = 0; i < 5; ++i) {
            float f[16];
            factors<IO>(L, i, lo[i], lane, f);
#pragma unroll
            for (int e = 0; e < 16; ++e) f[e] = fmaf(d[e], f[e], x[e]);
            if (t < P.rows) store16<IO>(P.out[i], e0, f);
        }
    }
}

template <typename IO>
__global__ __launch_bounds__(256, 2)
void maa_lora_mix_bwd_kernel(LoraArgs P)
{
    __shared__ __attribute__((aligned(16))) LoraLds<IO> L;
    __shared__ float s_sum[4][5][LM_C];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, c0 = blockIdx.x * LM_C;
    const size_t n = (size_t)P.rows * P.C;
    stage<IO>(L, P, c0);
    float acc[5] = {0.f, 0.f, 0.f, 0.f, 0.f};              // of channel slot `slot`, over the 16 tokens of the lane's row of lanes
    int slot = 0;
    for (int s = 0; s < P.steps; ++s) {
        const long long t = ((long long)blockIdx.y * P.steps + s) * LM_TOK + wave * 16 + (lane & 15);
        const bool ok = t < P.rows;
        const long long tl = ok ? t : P.rows - 1;
        const size_t e0 = (size_t)tl * P.C + c0 + 8 * (lane >> 4);
        u32x4 lo[5];
#pragma unroll
        for (int i = 0; i < 5; ++i)
            lo[i] = *reinterpret_cast<const u32x4*>(static_cast<const IO*>(P.lo) + (size_t)tl * (5 * LM_K) + LM_K * i + 8 * (lane >> 4));
        const Raw16 xr = fetch16<IO>(P.x, e0), dr = fetch16<IO>(P.sx, e0);
        Raw16 gr[5];
#pragma unroll
        for (int i = 0; i < 5; ++i) gr[i] = fetch16<IO>(P.g[i], e0);
        float d[16], gx[16], gsx[16];
        widen16<IO>(xr, gx);
        widen16<IO>(dr, d);
#pragma unroll
        for (int e = 0; e < 16; ++e) { d[e] -= gx[e]; gx[e] = 0.f; gsx[e] = 0.f; }
#pragma unroll
        for (int i = 0; i < 5; ++i) {
            float f[16], g[16];
            factors<IO>(L, i, lo[i], lane, f);
            asm volatile("" : "+v"(gr[i].a), "+v"(gr[i].b));           // packed until here
            widen16<IO>(gr[i], g);
#pragma unroll
            for (int e = 0; e < 16; ++e) {
                gsx[e] = fmaf(g[e], f[e], gsx[e]);
                gx[e] = fmaf(g[e], 1.f - f[e], gx[e]);
                g[e] = ok ? g[e] * d[e] : 0.f;
                asm volatile("" : "+v"(gx[e]), "+v"(gsx[e]));          // formed here: left to the stores below, ten operands each wait for it
            }
            acc[i] += wkv6_detail::row_sums16(g, lane, slot);
            if (ok) store16<IO>(static_cast<IO*>(P.gm) + (size_t)i * n, e0, g);
        }
        if (ok) {
            store16<IO>(P.gx, e0, gx);
            store16<IO>(P.gsx, e0, gsx);
        }
    }
#pragma unroll
    for (int i = 0; i < 5; ++i) s_sum[wave][i][32 * (slot >> 3) + 8 * (lane >> 4) + (slot & 7)] = acc[i];
    __syncthreads();
    float* prow = P.part + (size_t)blockIdx.y * 5 * P.C;
    for (int q = threadIdx.x; q < 5 * LM_C; q += 256) {
        const int i = q / LM_C, c = q % LM_C;
        prow[(size_t)i * P.C + c0 + c] = (s_sum[0][i][c] + s_sum[1][i][c]) + (s_sum[2][i][c] + s_sum[3][i][c]);
    }
}

// token chunks: workgroups of equally many steps
void plan(long long rows, int C, int target, int& chunks, int& steps) {
    const long long all = (rows + LM_TOK - 1) / LM_TOK;
    const long long want = target / (C / LM_C) > 0 ? target / (C / LM_C) : 1;
    steps = (int)((all + want - 1) / want);
    chunks = (int)((all + steps - 1) / steps);
}

int check(const char* name, const LoraArgs& P, int io_dtype, uintptr_t bits) {
    if (P.rows <= 0 || P.C <= 0 || !P.x || !P.sx || !P.lo || !P.w2 || !P.maa) {
        set_error("%s: bad arguments (rows=%lld C=%d)", name, P.rows, P.C);
        return VRWKV_INVALID_ARG;
    }
    if (io_dtype != VRWKV_BF16 && io_dtype != VRWKV_F16) {
        set_error("%s: unsupported io_dtype code %d", name, io_dtype);
        return VRWKV_UNSUPPORTED_DTYPE;
    }
    bits |= (uintptr_t)P.x | (uintptr_t)P.sx | (uintptr_t)P.lo | (uintptr_t)P.w2;
    if (P.C % LM_C || P.C > 65536 || P.rows > (1LL << 30) || (bits & 15) || ((uintptr_t)P.maa & 3)) {
        set_error("%s: C=%d must be a multiple of %d and every token matrix 16-byte aligned", name, P.C, LM_C);
        return VRWKV_UNSUPPORTED_SHAPE;
    }
    return VRWKV_OK;
}

}  // namespace
}  // namespace vrwkv

using namespace vrwkv;

extern "C" int vrwkv_maa_lora_mix(const void* x, const void* sx, const void* lo, const void* w2, const float* maa, void* const* out,
                                  long long rows, int C, int io_dtype, void* hip_stream) {
    LoraArgs P = {};
    P.x = x, P.sx = sx, P.lo = lo, P.w2 = w2, P.maa = maa, P.rows = rows, P.C = C;
    uintptr_t bits = 0;
    for (int i = 0; i < 5; ++i) {
        if (!out || !out[i]) { set_error("maa_lora_mix: output %d is null", i); return VRWKV_INVALID_ARG; }
        P.out[i] = out[i];
        bits |= (uintptr_t)out[i];
    }
    if (const int rc = check("maa_lora_mix", P, io_dtype, bits)) return rc;
    int chunks;
    plan(rows, C, LM_WG, chunks, P.steps);
    if (chunks > 65535) { set_error("maa_lora_mix: too many rows"); return VRWKV_UNSUPPORTED_SHAPE; }
    const dim3 grid((unsigned)(C / LM_C), (unsigned)chunks);
    hipStream_t st = static_cast<hipStream_t>(hip_stream);
    if (io_dtype == VRWKV_BF16) hipLaunchKernelGGL((maa_lora_mix_kernel<__hip_bfloat16>), grid, dim3(256), 0, st, P);
    else hipLaunchKernelGGL((maa_lora_mix_kernel<__half>), grid, dim3(256), 0, st, P);
    return check_launch("maa_lora_mix");
}

extern "C" size_t vrwkv_maa_lora_mix_bwd_workspace_bytes(long long rows, int C) {
    if (rows <= 0 || C < LM_C) return 0;
    int chunks, steps;
    plan(rows, C, LM_WG_BWD, chunks, steps);
    return (size_t)chunks * 5 * C * sizeof(float);
}

extern "C" int vrwkv_maa_lora_mix_bwd(const void* x, const void* sx, const void* lo, const void* w2, const float* maa, const void* const* gout,
                                      void* gx, void* gsx, void* gm, float* gmaa, long long rows, int C, int io_dtype,
                                      void* workspace, size_t workspace_bytes, void* hip_stream) {
    LoraArgs P = {};
    P.x = x, P.sx = sx, P.lo = lo, P.w2 = w2, P.maa = maa, P.rows = rows, P.C = C, P.gx = gx, P.gsx = gsx, P.gm = gm;
    if (!gout || !gx || !gsx || !gm || !gmaa) { set_error("maa_lora_mix_bwd: null pointer argument"); return VRWKV_INVALID_ARG; }
    uintptr_t bits = (uintptr_t)gx | (uintptr_t)gsx | (uintptr_t)gm;
    for (int i = 0; i < 5; ++i) {
        if (!gout[i]) { set_error("maa_lora_mix_bwd: gradient %d is null", i); return VRWKV_INVALID_ARG; }
        P.g[i] = gout[i];
        bits |= (uintptr_t)gout[i];
    }
    if (const int rc = check("maa_lora_mix_bwd", P, io_dtype, bits)) return rc;
    const size_t need = vrwkv_maa_lora_mix_bwd_workspace_bytes(rows, C);
    if (!workspace || workspace_bytes < need || ((uintptr_t)workspace & 3)) {
        set_error("maa_lora_mix_bwd: a 4-byte aligned workspace of %zu bytes is required", need);
        return VRWKV_WORKSPACE_TOO_SMALL;
    }
    int chunks;
    plan(rows, C, LM_WG_BWD, chunks, P.steps);
    if (chunks > 65535) { set_error("maa_lora_mix_bwd: too many rows"); return VRWKV_UNSUPPORTED_SHAPE; }
    P.part = static_cast<float*>(workspace);
    const dim3 grid((unsigned)(C / LM_C), (unsigned)chunks);
    hipStream_t st = static_cast<hipStream_t>(hip_stream);
    if (io_dtype == VRWKV_BF16) hipLaunchKernelGGL((maa_lora_mix_bwd_kernel<__hip_bfloat16>), grid, dim3(256), 0, st, P);
    else hipLaunchKernelGGL((maa_lora_mix_bwd_kernel<__half>), grid, dim3(256), 0, st, P);
    launch_batch_sum(P.part, gmaa, nullptr, SumOut((float*)nullptr), chunks, 5 * C, st);
    return check_launch("maa_lora_mix_bwd");
}
