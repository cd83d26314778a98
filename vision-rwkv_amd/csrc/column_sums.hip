// Sums over the rows of a token matrix: the gradient of a vector that is added to every token (time_decay of VRWKV6).
//
// Memory bounds it: one read.  32 channel vectors x 8 rows a workgroup, four rows of a thread in flight, about 1024 workgroups whatever the
// width, and one partial row each, which batch_sum_kernel adds up in a fixed order.  torch's reduction, which runs 192 workgroups of 256
// threads along the rows and combines them through flags in memory, takes 22.8 us at 12544 x 768 bf16, the two launches here 11.0
// (784 x 768 9.1 / 4.4, 50000 x 192 21.2 / 9.1, 12544 x 768 fp32 24.4 / 12.4; 196 x 192 5.6 / 4.2).
#include "vrwkv_common.h"
#include "../../include/vrwkv_hip.h"

namespace vrwkv {
namespace {

constexpr int CS_CX = 32, CS_TY = 8, CS_ROWS = 4, CS_TARGET_WG = 1024;

int chunks_of(long long rows, int C, int vec) {
    const int gx = (C / vec + CS_CX - 1) / CS_CX;
    const long long most = (rows + CS_TY * CS_ROWS - 1) / (CS_TY * CS_ROWS);       // a chunk keeps every thread in work
    long long n = CS_TARGET_WG / gx;
    n = n < 1 ? 1 : n;
    return (int)(n < most ? n : most);
}

template <typename IO, int VEC>
__global__ __launch_bounds__(CS_CX * CS_TY)
void column_sums_kernel(const IO* __restrict__ x, float* __restrict__ part, long long rows, int C, long long per)
{
    __shared__ float s_acc[CS_TY][CS_CX * VEC];
    const int cx = threadIdx.x % CS_CX, ty = threadIdx.x / CS_CX;
    const int c = (blockIdx.x * CS_CX + cx) * VEC;
    const long long r0 = blockIdx.y * per, r1 = r0 + per < rows ? r0 + per : rows;
    float acc[VEC];
#pragma unroll
    for (int e = 0; e < VEC; ++e) acc[e] = 0.f;
    if (c < C) {
        using Packed = typename RawVec<sizeof(IO) * VEC>::type;
        for (long long r = r0 + ty; r < r1; r += CS_TY * CS_ROWS) {
            Packed p[CS_ROWS];
#pragma unroll
            for (int j = 0; j < CS_ROWS; ++j) {
                const long long rr = r + CS_TY * j;
                p[j] = load_packed<IO, VEC>(x + (size_t)(rr < r1 ? rr : r) * C + c);         // past the chunk: a valid row, not used
            }
#pragma unroll
            for (int j = 0; j < CS_ROWS; ++j) {
                float v[VEC];
                widen_packed<IO, VEC>(p[j], v);
#pragma unroll
                for (int e = 0; e < VEC; ++e) acc[e] += r + CS_TY * j < r1 ? v[e] : 0.f;
            }
        }
    }
#pragma unroll
    for (int e = 0; e < VEC; ++e) s_acc[ty][cx * VEC + e] = acc[e];
    __syncthreads();
    for (int o = threadIdx.x; o < CS_CX * VEC; o += CS_CX * CS_TY) {
        const int cg = blockIdx.x * CS_CX * VEC + o;
        if (cg >= C) continue;
        float sum = 0.f;
#pragma unroll
        for (int y = 0; y < CS_TY; ++y) sum += s_acc[y][o];
        part[(size_t)blockIdx.y * C + cg] = sum;
    }
}

template <typename IO, int VEC>
int launch(const void* x, void* out, long long rows, int C, int dtype, float* part, hipStream_t st) {
    const int n = chunks_of(rows, C, VEC);
    const long long per = (rows + n - 1) / n;
    hipLaunchKernelGGL((column_sums_kernel<IO, VEC>), dim3((unsigned)((C / VEC + CS_CX - 1) / CS_CX), (unsigned)n), dim3(CS_CX * CS_TY), 0, st,
                       static_cast<const IO*>(x), part, rows, C, per);
    launch_batch_sum(part, SumOut(out, dtype), nullptr, SumOut((float*)nullptr), n, C, st);
    return check_launch("column_sums");
}

template <typename IO>
int launch_io(const void* x, void* out, long long rows, int C, int dtype, bool wide, float* part, hipStream_t st) {
    constexpr int V = 16 / sizeof(IO);
    return wide && C % V == 0 ? launch<IO, V>(x, out, rows, C, dtype, part, st) : launch<IO, 1>(x, out, rows, C, dtype, part, st);
}

}  // namespace
}  // namespace vrwkv

using namespace vrwkv;

extern "C" size_t vrwkv_column_sums_workspace_bytes(long long rows, int C) {
    if (rows <= 0 || C <= 0) return 0;
    const int n = chunks_of(rows, C, C % 8 == 0 ? 8 : 1), n1 = chunks_of(rows, C, 1), n4 = chunks_of(rows, C, C % 4 == 0 ? 4 : 1);
    const int most = n > n1 ? (n > n4 ? n : n4) : (n1 > n4 ? n1 : n4);
    return (size_t)most * C * sizeof(float);
}

extern "C" int vrwkv_column_sums(const void* x, void* out, long long rows, int C, int dtype, void* workspace, size_t workspace_bytes, void* hip_stream) {
    if (rows <= 0 || C <= 0 || rows >= (1LL << 40) / C) {
        set_error("column_sums: bad sizes (rows=%lld C=%d)", rows, C);
        return VRWKV_INVALID_ARG;
    }
    if (!x || !out) {
        set_error("column_sums: null pointer argument");
        return VRWKV_INVALID_ARG;
    }
    const size_t need = vrwkv_column_sums_workspace_bytes(rows, C);
    if (!workspace || workspace_bytes < need || ((uintptr_t)workspace & 3)) {
        set_error("column_sums: a 4-byte aligned workspace of %zu bytes is required", need);
        return VRWKV_WORKSPACE_TOO_SMALL;
    }
    const bool wide = ((uintptr_t)x & 15) == 0;
    float* part = static_cast<float*>(workspace);
    hipStream_t st = static_cast<hipStream_t>(hip_stream);
    switch (dtype) {
        case VRWKV_F32:  return launch_io<float>(x, out, rows, C, dtype, wide, part, st);
        case VRWKV_BF16: return launch_io<__hip_bfloat16>(x, out, rows, C, dtype, wide, part, st);
        case VRWKV_F16:  return launch_io<__half>(x, out, rows, C, dtype, wide, part, st);
    }
    set_error("column_sums: unsupported dtype code %d", dtype);
    return VRWKV_UNSUPPORTED_DTYPE;
}
