// Weight gradients of the projections: out (n; O, I) = sum over the tokens t of g[t][o] x[t][i], 16-bit operands with the tokens
// as rows, fp32 sums.  A deep contraction (12544 tokens) into a small matrix: a workgroup takes a 128 x 128 tile of the
// result and a range of the tokens and leaves its fp32 partial sum, a second kernel adds the ranges in a fixed order and
// rounds once.  Bound by the LDS reads of 64 x 64 quadrants and, with many ranges, by the partial sums' way through memory
// (14 ranges of 768 x 768: 33 MB out and in): two workgroups per compute unit (14 ranges; 7: 41 us, 28: 41 us) and at most 32
// ranges, or ranges of 24 slices where that is more, measure best (192 x 192 on 12544 tokens: 28 ranges 15 us, 98 ranges 23 us; on
// 100352: 32 ranges 61 us, 64 39, 128 35, 256 45; 96 x 96 on 301056: 32 ranges 162 us, 128 56, 256 47).  12544 tokens, bf16, own / the library's batched partial
// products in bf16 and their sum: 768 x 768 34 / 43 us, 384 x 384 22 / 37, 1536 x 384 33 / 42, 768 x 64 16 / 25; error against
// float64 1.7e-3 (the result's rounding) / 2.4e-3.
#include "gemm_tile.h"
#include <algorithm>

namespace vrwkv {
namespace {
using namespace gemm;

// Workgroup -> (tile, range): workgroups are dealt round-robin to the eight XCDs; those of one token range, which read the
// same rows, get numbers that are equal modulo 8 as far as the count allows, and share an L2.
template <typename IO>
__global__ __launch_bounds__(256, 3)
void wgrad_kernel(const IO* __restrict__ g_, const IO* __restrict__ x_, float* __restrict__ part, int M, int O, int I, int ldg, int ldx,
                  long long bsg, long long bsx, int tiles_i, int tiles, int splits, int slices_per)
{
    __shared__ __attribute__((aligned(16))) char lds[Stage<true>::LDS];
    const int lane = threadIdx.x & 63, g4 = lane >> 4, c16 = lane & 15, w4 = threadIdx.x >> 6;
    int id = blockIdx.x;
    const int whole = tiles * splits / 8 * 8;
    if (id < whole) id = (id & 7) * (whole / 8) + (id >> 3);
    const int split = id / tiles, tile = id % tiles, z = blockIdx.y;
    const int row0 = tile / tiles_i * TILE, col0 = tile % tiles_i * TILE;
    const int n = (M + 31) / 32, s0 = split * slices_per, s1 = min(n, s0 + slices_per);
    f32x4 acc[4][4];
    // the columns are the first operand, so a lane holds four neighbouring ones
    tile_product<IO, true>(lds, x_ + z * bsx, g_ + z * bsg, col0, row0, I, O, M, ldx, ldg, s0, s1, acc);
    float* out = part + ((size_t)z * splits + split) * O * I;
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const int c = col0 + 64 * (w4 & 1) + 16 * i + 4 * g4, r = row0 + 64 * (w4 >> 1) + 16 * j + c16;
            if (r < O && c < I) *reinterpret_cast<f32x4*>(out + (size_t)r * I + c) = acc[i][j];
        }
}

template <typename IO>
__global__ __launch_bounds__(256)
void wgrad_sum_kernel(const float* __restrict__ part, IO* __restrict__ out, long long quads, int splits)
{
    const long long q = (long long)blockIdx.x * 256 + threadIdx.x;
    if (q >= quads) return;
    const f32x4* p = reinterpret_cast<const f32x4*>(part) + (size_t)blockIdx.y * splits * quads + q;
    f32x4 s = {0.f, 0.f, 0.f, 0.f};
    constexpr int U = 8;
    for (int i = 0; i < splits; i += U) {
        f32x4 v[U];
#pragma unroll
        for (int j = 0; j < U; ++j) v[j] = i + j < splits ? p[(size_t)(i + j) * quads] : f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int j = 0; j < U; ++j) s += v[j];
    }
    const float r[4] = {s[0], s[1], s[2], s[3]};
    store_vec<IO, 4>(out + ((size_t)blockIdx.y * quads + q) * 4, r);
}

struct Plan { int tiles_o, tiles_i, splits, slices_per; };
Plan plan(int n, int M, int O, int I) {
    Plan p;
    p.tiles_o = (O + TILE - 1) / TILE;
    p.tiles_i = (I + TILE - 1) / TILE;
    const int slices = (M + 31) / 32, forced = option(OPT_WGRAD_SPLITS);
    const long long tiles = (long long)n * p.tiles_o * p.tiles_i;
    int s = forced ? forced : (int)std::max(1LL, 2LL * device_cus() / tiles);
    if (!forced) s = std::min(s, std::max(32, slices / 24));
    s = std::min(s, std::max(1, slices / 4));
    p.slices_per = (slices + s - 1) / s;
    p.splits = (slices + p.slices_per - 1) / p.slices_per;
    return p;
}
bool fits(int n, int M, int O, int I) {
    return n > 0 && n <= 65535 && M > 0 && O > 0 && I > 0 && O % 8 == 0 && I % 8 == 0 && O <= 65536 && I <= 65536 && (long long)O * I <= (1LL << 28);
}

template <typename IO>
int launch(const void* g, const void* x, void* out, float* ws, int n, int M, int O, int I, int ldg, int ldx, long long bsg, long long bsx,
           hipStream_t st) {
    const Plan p = plan(n, M, O, I);
    const int tiles = p.tiles_o * p.tiles_i;
    hipLaunchKernelGGL((wgrad_kernel<IO>), dim3((unsigned)(tiles * p.splits), n), dim3(256), 0, st, (const IO*)g, (const IO*)x, ws, M, O, I,
                       ldg, ldx, bsg, bsx, p.tiles_i, tiles, p.splits, p.slices_per);
    const long long quads = (long long)O * I / 4;
    hipLaunchKernelGGL((wgrad_sum_kernel<IO>), dim3((unsigned)((quads + 255) / 256), n), dim3(256), 0, st, ws, (IO*)out, quads, p.splits);
    return check_launch("wgrad");
}

}  // namespace
}  // namespace vrwkv

extern "C" size_t vrwkv_wgrad_workspace_bytes(int n, int M, int O, int I)
{
    using namespace vrwkv;
    return fits(n, M, O, I) ? (size_t)n * plan(n, M, O, I).splits * O * I * sizeof(float) : 0;
}

extern "C" int vrwkv_wgrad(const void* g, const void* x, void* out, int n, int M, int O, int I, int ldg, int ldx, long long stride_g,
                           long long stride_x, int dtype, void* workspace, size_t workspace_bytes, void* hip_stream)
{
    using namespace vrwkv;
    if (!g || !x || !out || !workspace || (((size_t)g | (size_t)x | (size_t)out | (size_t)workspace) & 15)) {
        set_error("wgrad: null or misaligned (16 bytes) pointer argument");
        return VRWKV_INVALID_ARG;
    }
    if (!fits(n, M, O, I) || ldg < O || ldx < I || ldg % 8 || ldx % 8 || stride_g % 8 || stride_x % 8 || stride_g < 0 || stride_x < 0 ||
        (long long)M * ldg >= (1LL << 30) || (long long)M * ldx >= (1LL << 30)) {
        set_error("wgrad: unsupported sizes (n=%d M=%d O=%d I=%d ldg=%d ldx=%d)", n, M, O, I, ldg, ldx);
        return VRWKV_UNSUPPORTED_SHAPE;
    }
    if (workspace_bytes < vrwkv_wgrad_workspace_bytes(n, M, O, I)) {
        set_error("wgrad: workspace of %zu bytes is too small", workspace_bytes);
        return VRWKV_WORKSPACE_TOO_SMALL;
    }
    hipStream_t st = static_cast<hipStream_t>(hip_stream);
    if (dtype == VRWKV_BF16) return launch<__hip_bfloat16>(g, x, out, (float*)workspace, n, M, O, I, ldg, ldx, stride_g, stride_x, st);
    if (dtype == VRWKV_F16) return launch<__half>(g, x, out, (float*)workspace, n, M, O, I, ldg, ldx, stride_g, stride_x, st);
    set_error("wgrad: dtype must be bf16 or fp16");
    return VRWKV_UNSUPPORTED_DTYPE;
}
