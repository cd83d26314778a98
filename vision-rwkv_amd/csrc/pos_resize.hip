// Bicubic resampling of a position table (Hi*Wi tokens of C channels) to another patch grid, and its adjoint: the
// interpolation of detection/mmdet_custom/models/utils/embed.py:6-47 (cubic convolution with A = -0.75, sample points
// (o + 0.5) Hi/Ho - 0.5, taps clamped to the border), on the table as it lies in memory.
//
// The library's kernel works on (1, C, Hi, Wi) images, gives one output pixel to a thread and walks the channels inside
// it: a 24 x 24 grid is three workgroups with a serial chain over C (4190 us for 12 x 12 -> 24 x 24 at C = 1024, and it
// needs the table transposed and back; the adjoint adds with atomics on top: 21.9 ms for both).  Here a thread owns neighbouring channels of one token, so
// every tap of a wave is one coalesced row piece and the chip sees tokens x C / VEC independent threads.
// Both directions are bound by launch and load latency (result and gradient through autograd 0.13 ms, all of it host time); the table and the result are a few MB at most.  The adjoint
// gathers (an input token reads the outputs whose taps reach it), so it needs no atomics and its sums have a fixed order.
#include "vrwkv_common.h"

namespace vrwkv {
namespace {

constexpr int PR_THREADS = 128;

// first tap of output position o and the four weights
__device__ __forceinline__ int cubic_taps(int o, float scale, float (&w)[4]) {
    const float A = -0.75f;
    const float real = scale * ((float)o + 0.5f) - 0.5f, fl = floorf(real), t = real - fl;
    auto near = [&](float x) { return ((A + 2.f) * x - (A + 3.f)) * x * x + 1.f; };              // |x| <= 1
    auto far = [&](float x) { return ((A * x - 5.f * A) * x + 8.f * A) * x - 4.f * A; };          // 1 < |x| < 2
    w[0] = far(t + 1.f);
    w[1] = near(t);
    w[2] = near(1.f - t);
    w[3] = far(2.f - t);
    return (int)fl - 1;
}

// Grid: (tokens of the result, channel blocks), block PR_THREADS.
template <typename IO, int VEC>
__global__ __launch_bounds__(PR_THREADS)
void pos_resize_kernel(const IO* __restrict__ src, IO* __restrict__ dst, int Hi, int Wi, int Wo, float sy, float sx, int C)
{
    const int c = (blockIdx.y * PR_THREADS + threadIdx.x) * VEC;
    if (c >= C) return;
    const int oy = blockIdx.x / Wo, ox = blockIdx.x % Wo;
    float wy[4], wx[4];
    const int y0 = cubic_taps(oy, sy, wy), x0 = cubic_taps(ox, sx, wx);
    typename RawVec<sizeof(IO) * VEC>::type raw[4][4];
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const int y = min(max(y0 + i, 0), Hi - 1), x = min(max(x0 + j, 0), Wi - 1);
            raw[i][j] = load_packed<IO, VEC>(src + ((size_t)y * Wi + x) * C + c);
        }
    float r[VEC];
#pragma unroll
    for (int e = 0; e < VEC; ++e) r[e] = 0.f;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        float row[VEC];
#pragma unroll
        for (int e = 0; e < VEC; ++e) row[e] = 0.f;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            float v[VEC];
            widen_packed<IO, VEC>(raw[i][j], v);
#pragma unroll
            for (int e = 0; e < VEC; ++e) row[e] = fmaf(wx[j], v[e], row[e]);
        }
#pragma unroll
        for (int e = 0; e < VEC; ++e) r[e] = fmaf(wy[i], row[e], r[e]);
    }
    store_vec<IO, VEC>(dst + (size_t)blockIdx.x * C + c, r);
}

// outputs whose taps can reach input position p: their sample point lies in [p - 2, p + 2); one more on either side for
// the rounding of the quotient (those get weight 0)
__device__ __forceinline__ void reach(int p, float scale, int No, int& lo, int& hi) {
    lo = max(0, (int)floorf(((float)p - 1.5f) / scale - 0.5f) - 1);
    hi = min(No - 1, (int)ceilf(((float)p + 2.5f) / scale - 0.5f) + 1);
}
// weight of input position p in output o, the clamped taps counted at the border
__device__ __forceinline__ float weight_of(int p, int o, int Ni, float scale) {
    float w[4], s = 0.f;
    const int f = cubic_taps(o, scale, w);
#pragma unroll
    for (int k = 0; k < 4; ++k) s += min(max(f + k, 0), Ni - 1) == p ? w[k] : 0.f;
    return s;
}

// Adjoint: one token of the table per workgroup row.  Grid: (Hi * Wi, channel blocks), block PR_THREADS.
template <typename IO, int VEC>
__global__ __launch_bounds__(PR_THREADS)
void pos_resize_adj_kernel(const IO* __restrict__ g, IO* __restrict__ dst, int Hi, int Wi, int Ho, int Wo, float sy, float sx, int C)
{
    const int c = (blockIdx.y * PR_THREADS + threadIdx.x) * VEC;
    if (c >= C) return;
    const int y = blockIdx.x / Wi, x = blockIdx.x % Wi;
    int ylo, yhi, xlo, xhi;
    reach(y, sy, Ho, ylo, yhi);
    reach(x, sx, Wo, xlo, xhi);
    float r[VEC];
#pragma unroll
    for (int e = 0; e < VEC; ++e) r[e] = 0.f;
    for (int oy = ylo; oy <= yhi; ++oy) {
        const float wy = weight_of(y, oy, Hi, sy);
        if (wy == 0.f) continue;                          // uniform over the workgroup
        float row[VEC];
#pragma unroll
        for (int e = 0; e < VEC; ++e) row[e] = 0.f;
        constexpr int U = 4;                              // loads in flight
        for (int ox = xlo; ox <= xhi; ox += U) {
            typename RawVec<sizeof(IO) * VEC>::type raw[U];
            float wx[U];
#pragma unroll
            for (int i = 0; i < U; ++i) {
                raw[i] = load_packed<IO, VEC>(g + ((size_t)oy * Wo + min(ox + i, xhi)) * C + c);
                wx[i] = weight_of(x, ox + i, Wi, sx);
            }
#pragma unroll
            for (int i = 0; i < U; ++i) {
                if (ox + i > xhi || wx[i] == 0.f) continue;          // an unreached output takes no part, whatever it holds
                float v[VEC];
                widen_packed<IO, VEC>(raw[i], v);
#pragma unroll
                for (int e = 0; e < VEC; ++e) row[e] = fmaf(wx[i], v[e], row[e]);
            }
        }
#pragma unroll
        for (int e = 0; e < VEC; ++e) r[e] = fmaf(wy, row[e], r[e]);
    }
    store_vec<IO, VEC>(dst + (size_t)blockIdx.x * C + c, r);
}

template <typename IO, int VEC>
int launch(const void* src, void* dst, int Hi, int Wi, int Ho, int Wo, int C, int adjoint, hipStream_t stream) {
    const float sy = (float)Hi / (float)Ho, sx = (float)Wi / (float)Wo;
    const unsigned cb = (unsigned)((C + PR_THREADS * VEC - 1) / (PR_THREADS * VEC));
    if (adjoint)
        hipLaunchKernelGGL((pos_resize_adj_kernel<IO, VEC>), dim3((unsigned)(Hi * Wi), cb), dim3(PR_THREADS), 0, stream,
                           (const IO*)src, (IO*)dst, Hi, Wi, Ho, Wo, sy, sx, C);
    else
        hipLaunchKernelGGL((pos_resize_kernel<IO, VEC>), dim3((unsigned)(Ho * Wo), cb), dim3(PR_THREADS), 0, stream,
                           (const IO*)src, (IO*)dst, Hi, Wi, Wo, sy, sx, C);
    return check_launch("pos_resize");
}
// pairs of channels where C and both pointers allow them (wider pieces leave too few threads on small grids), else single ones
template <typename IO>
int dispatch(const void* src, void* dst, int Hi, int Wi, int Ho, int Wo, int C, int adjoint, hipStream_t stream) {
    const bool pairs = C % 2 == 0 && ((size_t)src | (size_t)dst) % (2 * sizeof(IO)) == 0;
    return pairs ? launch<IO, 2>(src, dst, Hi, Wi, Ho, Wo, C, adjoint, stream) : launch<IO, 1>(src, dst, Hi, Wi, Ho, Wo, C, adjoint, stream);
}

}  // namespace
}  // namespace vrwkv

extern "C" int vrwkv_pos_resize(const void* src, void* dst, int Hi, int Wi, int Ho, int Wo, int C, int adjoint, int dtype, void* stream)
{
    using namespace vrwkv;
    if (!src || !dst || Hi <= 0 || Wi <= 0 || Ho <= 0 || Wo <= 0 || C <= 0) {
        set_error("vrwkv_pos_resize: null pointer or empty grid (%d x %d -> %d x %d, C=%d)", Hi, Wi, Ho, Wo, C);
        return VRWKV_INVALID_ARG;
    }
    if ((long long)Hi * Wi > 0x7fffffffLL || (long long)Ho * Wo > 0x7fffffffLL || C > 65535 * PR_THREADS) {
        set_error("vrwkv_pos_resize: a grid of more than 2^31 tokens or %d channels", C);
        return VRWKV_UNSUPPORTED_SHAPE;
    }
    hipStream_t s = (hipStream_t)stream;
    switch (dtype) {
        case VRWKV_F32: return dispatch<float>(src, dst, Hi, Wi, Ho, Wo, C, adjoint, s);
        case VRWKV_BF16: return dispatch<__hip_bfloat16>(src, dst, Hi, Wi, Ho, Wo, C, adjoint, s);
        case VRWKV_F16: return dispatch<__half>(src, dst, Hi, Wi, Ho, Wo, C, adjoint, s);
    }
    set_error("vrwkv_pos_resize: unknown dtype %d", dtype);
    return VRWKV_UNSUPPORTED_DTYPE;
}
