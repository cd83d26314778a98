// Shared host/device helpers for the vrwkv HIP library (gfx950 only).
#pragma once
#include <hip/hip_runtime.h>
#include <hip/hip_bf16.h>
#include <hip/hip_fp16.h>
#include <cstdarg>
#include <cstdio>
#include <type_traits>
#include "../../include/vrwkv_hip.h"

namespace vrwkv {

// Thread-local message behind vrwkv_last_error().
void set_error(const char* fmt, ...);
// Returns VRWKV_OK, or VRWKV_LAUNCH_FAILED after recording hipGetLastError()'s text.
int check_launch(const char* what);
int device_cus();                 // compute units of the current device (256 when the query fails)

// Tuning / testing switches (0 = default behaviour).  Their initial values come from the environment variables
// VRWKV_<NAME IN CAPITALS>, read once per process; vrwkv_set_option changes them afterwards.
enum Option {
    OPT_BIWKV_L,            // tokens per wave of the Bi-WKV forward (4, 8, 16, 28)
    OPT_BIWKV_S,            // waves per workgroup on the long-sequence path
    OPT_BIWKV_GRID,         // persistent grid size
    OPT_BIWKV_NO_STAGE,     // register loads instead of LDS-staged rows
    OPT_BIWKV_NO_RESIDENT,  // two-kernel long-sequence path also where the one-launch kernel applies
    OPT_BIWKV_BWD_SERIAL,   // sequential Bi-WKV backward kernel
    OPT_WKV6_FWD_SCALAR,    // sequential-state wkv6 forward kernel
    OPT_WKV6_BWD_SCALAR,    // sequential wkv6 backward sweeps
    OPT_WKV6_BWD_UNFUSED,   // accepted, no effect (the backward is one kernel)
    OPT_WKV6_SEGMENTS,      // segments a wkv6 sequence is cut into
    OPT_LINEAR_TILE,        // tile of the block entry's projections (1, 2, 4, 8: 16 to 128 results on a side; 16: 256 channels wide)
    OPT_WGRAD_SPLITS,       // token ranges of a weight gradient
    OPT_LINEAR_MIX,         // norm, shift and mixes inside a half's projections: 1 or an error, 2 never
    N_OPTIONS
};
int option(Option o);

constexpr int WAVE = 64;
constexpr float LOG2E = 1.4426950408889634f;
constexpr float NEG_BIG = -1e38f;   // "empty state" exponent, bi_wkv_kernel.cu:14

#if defined(__HIPCC__)
__device__ __forceinline__ float to_f32(float x) { return x; }
__device__ __forceinline__ float to_f32(__hip_bfloat16 x) { return __bfloat162float(x); }
__device__ __forceinline__ float to_f32(__half x) { return __half2float(x); }
template <typename T> __device__ __forceinline__ T from_f32(float x);
template <> __device__ __forceinline__ float from_f32<float>(float x) { return x; }
template <> __device__ __forceinline__ __hip_bfloat16 from_f32<__hip_bfloat16>(float x) { return __float2bfloat16(x); }
template <> __device__ __forceinline__ __half from_f32<__half>(float x) { return __float2half(x); }

template <int BYTES> struct RawVec;
template <> struct RawVec<2>  { using type = unsigned short; };
template <> struct RawVec<4>  { using type = unsigned int; };
template <> struct RawVec<8>  { using type = uint2; };
template <> struct RawVec<16> { using type = uint4; };

// One vector load of VEC consecutive elements, widened to fp32.
template <typename IO, int VEC>
__device__ __forceinline__ void load_vec(const IO* __restrict__ p, float (&out)[VEC]) {
    using R = typename RawVec<sizeof(IO) * VEC>::type;
    R raw = *reinterpret_cast<const R*>(p);
    IO tmp[VEC];
    __builtin_memcpy(tmp, &raw, sizeof(raw));
#pragma unroll
    for (int e = 0; e < VEC; ++e) out[e] = to_f32(tmp[e]);
}
template <typename IO, int VEC>
__device__ __forceinline__ void store_vec(IO* __restrict__ p, const float (&in)[VEC]) {
    using R = typename RawVec<sizeof(IO) * VEC>::type;
    IO tmp[VEC];
#pragma unroll
    for (int e = 0; e < VEC; ++e) tmp[e] = from_f32<IO>(in[e]);
    R raw;
    __builtin_memcpy(&raw, tmp, sizeof(raw));
    *reinterpret_cast<R*>(p) = raw;
}
// A vector of VEC elements fetched now and widened where it is used (it waits in its packed form).
template <typename IO, int VEC>
__device__ __forceinline__ typename RawVec<sizeof(IO) * VEC>::type load_packed(const IO* __restrict__ p) {
    return *reinterpret_cast<const typename RawVec<sizeof(IO) * VEC>::type*>(p);
}
template <typename IO, int VEC>
__device__ __forceinline__ void widen_packed(typename RawVec<sizeof(IO) * VEC>::type raw, float (&out)[VEC]) {
    IO tmp[VEC];
    __builtin_memcpy(tmp, &raw, sizeof(raw));
#pragma unroll
    for (int e = 0; e < VEC; ++e) out[e] = to_f32(tmp[e]);
}
// The same with the non-temporal cache policy, for tensors that are streamed through once (16-byte vectors only).
typedef unsigned int nt_u32x4 __attribute__((ext_vector_type(4)));
template <typename IO, int VEC>
__device__ __forceinline__ void load_vec_nt(const IO* __restrict__ p, float (&out)[VEC]) {
    static_assert(sizeof(IO) * VEC == 16, "16-byte vectors");
    const nt_u32x4 raw = __builtin_nontemporal_load(reinterpret_cast<const nt_u32x4*>(p));
    IO tmp[VEC];
    __builtin_memcpy(tmp, &raw, sizeof(raw));
#pragma unroll
    for (int e = 0; e < VEC; ++e) out[e] = to_f32(tmp[e]);
}
// A 16-byte vector fetched now and widened where it is used (keeps four registers, not VEC, while it waits).
template <bool NT>
__device__ __forceinline__ nt_u32x4 load_raw16(const void* p) {
    return NT ? __builtin_nontemporal_load(reinterpret_cast<const nt_u32x4*>(p)) : *reinterpret_cast<const nt_u32x4*>(p);
}
template <typename IO, int VEC>
__device__ __forceinline__ void widen_raw16(nt_u32x4 raw, float (&out)[VEC]) {
    static_assert(sizeof(IO) * VEC == 16, "16-byte vectors");
    IO tmp[VEC];
    __builtin_memcpy(tmp, &raw, sizeof(raw));
#pragma unroll
    for (int e = 0; e < VEC; ++e) out[e] = to_f32(tmp[e]);
}
template <typename IO, int VEC>
__device__ __forceinline__ void store_vec_nt(IO* __restrict__ p, const float (&in)[VEC]) {
    static_assert(sizeof(IO) * VEC == 16, "16-byte vectors");
    IO tmp[VEC];
#pragma unroll
    for (int e = 0; e < VEC; ++e) tmp[e] = from_f32<IO>(in[e]);
    nt_u32x4 raw;
    __builtin_memcpy(&raw, tmp, sizeof(raw));
    __builtin_nontemporal_store(raw, reinterpret_cast<nt_u32x4*>(p));
}
// Workgroup barrier that orders LDS traffic only: unlike __syncthreads() it does not wait
// for outstanding global loads/stores (vmcnt), so prefetches stay in flight across it.
__device__ __forceinline__ void lds_barrier() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

// ---- raw buffer access (descriptor + 32-bit byte offsets; out-of-range accesses are dropped by the
//      hardware: loads return 0, stores do nothing) -------------------------------------------------
constexpr unsigned OOB_OFFSET = 0x80000000u;   // byte offset no descriptor here reaches
constexpr unsigned CPOL_NT = 2;                // gfx94x/gfx950 cache policy bit: non-temporal (data streamed once)
template <int BYTES> struct BufRaw;
template <> struct BufRaw<2> {
    using type = unsigned short;
    template <unsigned CP = 0> static __device__ __forceinline__ type ld(__amdgpu_buffer_rsrc_t r, unsigned v, unsigned s) { return __builtin_amdgcn_raw_buffer_load_b16(r, v, s, CP); }
    template <unsigned CP = 0> static __device__ __forceinline__ void st(type d, __amdgpu_buffer_rsrc_t r, unsigned v, unsigned s) { __builtin_amdgcn_raw_buffer_store_b16(d, r, v, s, CP); }
};
template <> struct BufRaw<4> {
    using type = unsigned int;
    template <unsigned CP = 0> static __device__ __forceinline__ type ld(__amdgpu_buffer_rsrc_t r, unsigned v, unsigned s) { return __builtin_amdgcn_raw_buffer_load_b32(r, v, s, CP); }
    template <unsigned CP = 0> static __device__ __forceinline__ void st(type d, __amdgpu_buffer_rsrc_t r, unsigned v, unsigned s) { __builtin_amdgcn_raw_buffer_store_b32(d, r, v, s, CP); }
};
template <> struct BufRaw<8> {
    typedef unsigned int type __attribute__((ext_vector_type(2)));
    template <unsigned CP = 0> static __device__ __forceinline__ type ld(__amdgpu_buffer_rsrc_t r, unsigned v, unsigned s) { return __builtin_amdgcn_raw_buffer_load_b64(r, v, s, CP); }
    template <unsigned CP = 0> static __device__ __forceinline__ void st(type d, __amdgpu_buffer_rsrc_t r, unsigned v, unsigned s) { __builtin_amdgcn_raw_buffer_store_b64(d, r, v, s, CP); }
};
template <> struct BufRaw<16> {
    typedef unsigned int type __attribute__((ext_vector_type(4)));
    template <unsigned CP = 0> static __device__ __forceinline__ type ld(__amdgpu_buffer_rsrc_t r, unsigned v, unsigned s) { return __builtin_amdgcn_raw_buffer_load_b128(r, v, s, CP); }
    // The data stays in its registers for two cycles more.  The compiler leaves none between a store of 16 bytes whose offset is a scalar register and an
    // instruction that overwrites its data.  In one kernel (fp32 results of the segmented wkv6 backward) the fourth word of the last lanes was then, now and
    // then, the overwriting instruction's, and with the two cycles no more: an observation of that kernel on gfx950, not a documented property.
    template <unsigned CP = 0> static __device__ __forceinline__ void st(type d, __amdgpu_buffer_rsrc_t r, unsigned v, unsigned s) {
        __builtin_amdgcn_raw_buffer_store_b128(d, r, v, s, CP);
        asm volatile("s_nop 1" : : "v"(d));
    }
};

__device__ __forceinline__ __amdgpu_buffer_rsrc_t make_rsrc(const void* base, unsigned bytes) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(base), 0, bytes, 0x00020000);
}
// ---- per-phase cycle stamps (instrumented build only: -DVRWKV_STAMPS, `make stamps`) ----------------------------
// A wave records the shader clock at numbered points of a tile into a buffer the host registered with
// vrwkv_debug_set_stamp_buffer_<tag>(buffer, n_workgroups): layout [workgroup][wave (8)][tile slot (VRWKV_STAMP_TILES)]
// [point (VRWKV_STAMP_POINTS)]; workgroups beyond the count the buffer was sized for record nothing.
#ifdef VRWKV_STAMPS
constexpr int VRWKV_STAMP_TILES = 4, VRWKV_STAMP_POINTS = 12;
static __device__ unsigned long long* g_stamp_buffer = nullptr;   // one per translation unit (device code is not linked across them)
static __device__ unsigned g_stamp_workgroups = 0;                // workgroups the buffer has room for
// defines vrwkv_debug_set_stamp_buffer_<tag>(device_buffer, n_workgroups) for the translation unit it is used in
#define VRWKV_DEFINE_STAMP_SETTER(tag)                                                                      \
    extern "C" int vrwkv_debug_set_stamp_buffer_##tag(void* device_buffer, unsigned n_workgroups) {          \
        unsigned long long* p = static_cast<unsigned long long*>(device_buffer);                             \
        if (hipMemcpyToSymbol(HIP_SYMBOL(::vrwkv::g_stamp_workgroups), &n_workgroups, sizeof(n_workgroups)) != hipSuccess) return 4; \
        return hipMemcpyToSymbol(HIP_SYMBOL(::vrwkv::g_stamp_buffer), &p, sizeof(p)) == hipSuccess ? 0 : 4;   \
    }
__device__ __forceinline__ void stamp(int wave, int slot, int point) {
    unsigned long long* buf = g_stamp_buffer;
    if (buf && blockIdx.x < g_stamp_workgroups && wave < 8 && slot < VRWKV_STAMP_TILES && point < VRWKV_STAMP_POINTS &&
        (threadIdx.x & 63) == 0) {
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        buf[(((size_t)blockIdx.x * 8 + wave) * VRWKV_STAMP_TILES + slot) * VRWKV_STAMP_POINTS + point] = __builtin_amdgcn_s_memtime();
    }
}
#define VRWKV_STAMP(wave, slot, point) ::vrwkv::stamp(wave, slot, point)
#else
#define VRWKV_STAMP(wave, slot, point) ((void)0)
#endif

__device__ __forceinline__ float fast_exp2(float x) { return __builtin_amdgcn_exp2f(x); }
__device__ __forceinline__ float fast_rcp(float x) { return __builtin_amdgcn_rcpf(x); }

// A parameter vector of the Bi-WKV operator (decay, bonus) as the caller holds it: fp32, bf16 or fp16, times a factor in the same type
// (the block's division by T, which tensor ops carry out as a multiplication by the reciprocal).  Read where it is used, so that no
// call begins with casts and divisions of 768 numbers (a launch of 2 to 3 us each, four of them a layer in training).
// An element is fetched as it lies, nothing before or behind it, and widened at its use: the fetch can be ahead.
struct ParamVec {
    const void* p;
    int dtype;
    float factor;                                         // 1: as it is
    ParamVec() = default;
    ParamVec(const float* q) : p(q), dtype(VRWKV_F32), factor(1.f) {}
    __host__ __device__ ParamVec(const void* q, int dt, float f) : p(q), dtype(dt), factor(f) {}
    explicit operator bool() const { return p != nullptr; }
    bool aligned() const { return ((size_t)p & (dtype == VRWKV_F32 ? 3 : 1)) == 0; }
    __host__ __device__ __forceinline__ unsigned fetch(int c) const {
        return dtype == VRWKV_F32 ? static_cast<const unsigned*>(p)[c] : static_cast<const unsigned short*>(p)[c];
    }
    __device__ __forceinline__ float value(unsigned bits) const {
        float x = __builtin_bit_cast(float, bits);
        if (dtype == VRWKV_BF16) x = __builtin_bit_cast(float, bits << 16);
        else if (dtype == VRWKV_F16) x = (float)__builtin_bit_cast(_Float16, (unsigned short)bits);
        if (factor != 1.f) {
            x *= factor;
            if (dtype == VRWKV_BF16) x = to_f32(from_f32<__hip_bfloat16>(x));
            else if (dtype == VRWKV_F16) x = to_f32(from_f32<__half>(x));
        }
        return x;
    }
};
// The same for vectors whose type is known at the launch: fp32 ones, which inference and the extension's own calls hand over, in nearly every kernel, and
// those of the rows' type in the forward that keeps 16-bit rows in registers.  The branches of ParamVec are small beside a kernel of 20 us, but all
// waves pass them while nothing else is on its way.  us, ParamVec / TypedVec: fp32 64 x 196 x 768 23.9 / 23.5, 30 x 196 x 767 18.5 / 17.7, backward 38.2 / 36.6;
// fp32 vectors beside bf16 rows 2 x 4150 x 768 27.6 / 26.1, 4 x 1024 x 768 with the gate 20.9 / 19.3; 16 x 577 x 768 bf16 22.1 / 21.5, fp16 22.5 / 21.6.
template <typename T> constexpr int type_code = std::is_same<T, float>::value ? VRWKV_F32 : std::is_same<T, __hip_bfloat16>::value ? VRWKV_BF16 : VRWKV_F16;
template <typename T>
struct TypedVec {
    const T* p;
    float factor;
    TypedVec() = default;
    explicit TypedVec(const ParamVec& v) : p(static_cast<const T*>(v.p)), factor(v.factor) {}
    __device__ __forceinline__ unsigned fetch(int c) const {
        typedef typename std::conditional<sizeof(T) == 4, unsigned, unsigned short>::type raw_t;
        return reinterpret_cast<const raw_t*>(p)[c];
    }
    __device__ __forceinline__ float value(unsigned bits) const {
        return ParamVec(nullptr, type_code<T>, factor).value(bits);
    }
};

// out[c] = sum_b part[b*C + c] for up to two (part, out) pairs (the second may be null).  1024 threads = 32 columns
// (one 128-byte piece of a row per half wave) x 32 slices of the batch, sixteen loads of a slice in flight at a time
// (512 partial rows in one round of loads); the slices are added in a fixed order (deterministic).
// Grid: ceil(C / BATCH_SUM_COLS), block: BATCH_SUM_THREADS.
constexpr int BATCH_SUM_THREADS = 1024, BATCH_SUM_COLS = 32, BATCH_SUM_SLICES = BATCH_SUM_THREADS / BATCH_SUM_COLS;
// The sums leave as O: fp32, or rounded to the type of the parameter they are the gradient of (a cast kernel per gradient less).
template <typename O>
__global__ __launch_bounds__(1024) inline void batch_sum_kernel(const float* __restrict__ part0, O* __restrict__ out0,
                                                                const float* __restrict__ part1, O* __restrict__ out1,
                                                                int B, int C, float factor = 1.f) {
    constexpr int NS = BATCH_SUM_SLICES, U = 16;
    __shared__ float red[2][NS][BATCH_SUM_COLS];
    const int cl = threadIdx.x % BATCH_SUM_COLS, slice = threadIdx.x / BATCH_SUM_COLS;
    const int c = blockIdx.x * BATCH_SUM_COLS + cl;
    float s0 = 0.f, s1 = 0.f;
    if (c < C) {
        int b = slice;
        for (; b + NS * (U - 1) < B; b += NS * U) {
            float t0[U], t1[U];
#pragma unroll
            for (int i = 0; i < U; ++i) {
                t0[i] = part0[(size_t)(b + NS * i) * C + c];
                t1[i] = part1 ? part1[(size_t)(b + NS * i) * C + c] : 0.f;
            }
#pragma unroll
            for (int i = 0; i < U; ++i) { s0 += t0[i]; s1 += t1[i]; }
        }
        for (; b < B; b += NS) {
            s0 += part0[(size_t)b * C + c];
            if (part1) s1 += part1[(size_t)b * C + c];
        }
    }
    red[0][slice][cl] = s0;
    red[1][slice][cl] = s1;
    __syncthreads();
    if (slice == 0 && c < C) {
        float t0 = 0.f, t1 = 0.f;
#pragma unroll
        for (int i = 0; i < NS; ++i) { t0 += red[0][i][cl]; t1 += red[1][i][cl]; }
        out0[c] = from_f32<O>(t0);
        if (part1) out1[c] = from_f32<O>(t1);
        if (factor != 1.f) {                              // of the sum in its own type, like a multiplication of its own
            out0[c] = from_f32<O>(to_f32(from_f32<O>(t0)) * factor);
            if (part1) out1[c] = from_f32<O>(to_f32(from_f32<O>(t1)) * factor);
        }
    }
}
// Where the sums go, and as what.
struct SumOut {
    void* p;
    int dtype;
    SumOut(float* q) : p(q), dtype(VRWKV_F32) {}
    SumOut(void* q, int dt) : p(q), dtype(dt) {}
    explicit operator bool() const { return p != nullptr; }
};
inline void launch_batch_sum(const float* part0, SumOut out0, const float* part1, SumOut out1, int B, int C, hipStream_t st, float factor = 1.f) {
    const dim3 grid((C + BATCH_SUM_COLS - 1) / BATCH_SUM_COLS), block(BATCH_SUM_THREADS);
    if (out0.dtype == VRWKV_F32) hipLaunchKernelGGL((batch_sum_kernel<float>), grid, block, 0, st, part0, (float*)out0.p, part1, (float*)out1.p, B, C, factor);
    else if (out0.dtype == VRWKV_BF16)
        hipLaunchKernelGGL((batch_sum_kernel<__hip_bfloat16>), grid, block, 0, st, part0, (__hip_bfloat16*)out0.p, part1, (__hip_bfloat16*)out1.p, B, C, factor);
    else hipLaunchKernelGGL((batch_sum_kernel<__half>), grid, block, 0, st, part0, (__half*)out0.p, part1, (__half*)out1.p, B, C, factor);
}
#endif

}  // namespace vrwkv
