// A 128 x 128 tile of a 16-bit matrix product with fp32 accumulation on gfx950 matrix cores: four waves, each a 64 x 64
// quadrant of 16 x 16 x 32 products, operands staged in LDS twice (one copy is read while the next slice, already requested
// from memory before the products, is written to the other).  R and S are the two operands, row r of the result belongs to R:
//   KOUT = false  R (rows, K), S (cols, K), the contraction index innermost.  Slices of 64 k; a row's eight 16-byte pieces lie
//                 rotated by an exclusive-or with the row, so that 16 rows read at one k hit different banks.
//   KOUT = true   R (K, rows), S (K, cols), the contraction index outermost (a sum over tokens).  Slices of 32 k, rows of 288
//                 bytes; the fragments are read across the rows (ds_read_b64_tr_b16).  A lane group takes the k 4 g4 .. and
//                 16 + 4 g4 .. -- the same order for both operands, and the eight rows of a half wave start 32 bytes apart.
// Pieces outside an operand are requested at an offset that no descriptor reaches and read 0.
#pragma once
#include "vrwkv_common.h"
#include <type_traits>

namespace vrwkv {
namespace gemm {

typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef unsigned u32x4 __attribute__((ext_vector_type(4)));
typedef unsigned u32x2 __attribute__((ext_vector_type(2)));
template <typename IO> __device__ __forceinline__ f32x4 mfma16(u32x4 a, u32x4 b, f32x4 c) {
    if constexpr (std::is_same<IO, __hip_bfloat16>::value)
        return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
    else
        return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, a), __builtin_bit_cast(f16x8, b), c, 0, 0, 0);
}

constexpr int TILE = 128;
template <bool KOUT> struct Stage {
    static constexpr int BK = KOUT ? 32 : 64;                             // k per slice
    static constexpr int PITCH = KOUT ? 288 : 128;                        // bytes of an LDS row
    static constexpr int BYTES = KOUT ? 32 * PITCH : TILE * PITCH;        // one operand's slice
    static constexpr int PIECES = KOUT ? 2 : 4;                           // 16-byte pieces of it per thread
    static constexpr int LDS = 4 * BYTES;                                 // two operands, two copies
};

// acc[i][j]: rows 64 (w4 & 1) + 16 i + 4 g4 + e, column 64 (w4 >> 1) + 16 j + c16 of the tile, summed over slices [s0, s1).
// r0 / s0_: first row / column; rows, cols, K: the operands' extents; ldr, lds_: row pitches in elements.
template <typename IO, bool KOUT>
__device__ __forceinline__ void tile_product(char* lds, const IO* R, const IO* S, int row0, int col0, int rows, int cols, int K,
                                             int ldr, int lds_, int slice0, int slice1, f32x4 (&acc)[4][4])
{
    using P = Stage<KOUT>;
    const int tid = threadIdx.x, lane = tid & 63, g4 = lane >> 4, c16 = lane & 15;
    const int w4 = __builtin_amdgcn_readfirstlane(tid >> 6);
    const __amdgpu_buffer_rsrc_t rr = make_rsrc(R, KOUT ? ((unsigned)(K - 1) * ldr + rows) * 2u : ((unsigned)(rows - 1) * ldr + K) * 2u);
    const __amdgpu_buffer_rsrc_t rs = make_rsrc(S, KOUT ? ((unsigned)(K - 1) * lds_ + cols) * 2u : ((unsigned)(cols - 1) * lds_ + K) * 2u);
    u32x4 br[P::PIECES], bs[P::PIECES];
    auto fetch = [&](int s) {
#pragma unroll
        for (int i = 0; i < P::PIECES; ++i) {
            unsigned fr, fs;
            if (KOUT) {
                const int k = 32 * s + (tid >> 4) + 16 * i, c = 8 * (tid & 15);
                fr = k < K && row0 + c < rows ? ((unsigned)k * ldr + row0 + c) * 2u : OOB_OFFSET;
                fs = k < K && col0 + c < cols ? ((unsigned)k * lds_ + col0 + c) * 2u : OOB_OFFSET;
            } else {
                const int r = (tid >> 3) + 32 * i, k = 64 * s + 8 * (tid & 7);
                fr = k < K && row0 + r < rows ? ((unsigned)(row0 + r) * ldr + k) * 2u : OOB_OFFSET;
                fs = k < K && col0 + r < cols ? ((unsigned)(col0 + r) * lds_ + k) * 2u : OOB_OFFSET;
            }
            br[i] = BufRaw<16>::ld(rr, fr, 0);
            bs[i] = BufRaw<16>::ld(rs, fs, 0);
        }
    };
    auto put = [&](int buf) {
        char* base = lds + 2 * buf * P::BYTES;
#pragma unroll
        for (int i = 0; i < P::PIECES; ++i) {
            const int row = KOUT ? (tid >> 4) + 16 * i : (tid >> 3) + 32 * i;
            const int at = KOUT ? 16 * (tid & 15) : 16 * ((tid & 7) ^ (row & 7));
            *reinterpret_cast<u32x4*>(base + row * P::PITCH + at) = br[i];
            *reinterpret_cast<u32x4*>(base + P::BYTES + row * P::PITCH + at) = bs[i];
        }
    };
    // fragment of rows x .. x + 15 of an operand's slice, k half h (KOUT = false)
    auto frag = [&](const char* base, int x, int h) -> u32x4 {
        if constexpr (!KOUT) {
            const int row = x + c16;
            return *reinterpret_cast<const u32x4*>(base + row * P::PITCH + 16 * ((4 * h + g4) ^ (row & 7)));
        } else {
            typedef short s16x4 __attribute__((ext_vector_type(4)));
            typedef __attribute__((address_space(3))) s16x4 lds_s16x4;
            const char* p = base + (4 * g4 + (c16 >> 2)) * P::PITCH + 2 * (x + 4 * (c16 & 3));
            const u32x2 a = __builtin_bit_cast(u32x2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4*)p));
            const u32x2 b = __builtin_bit_cast(u32x2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4*)(p + 16 * P::PITCH)));
            return u32x4{a[0], a[1], b[0], b[1]};
        }
    };
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
    if (slice0 >= slice1) return;                                         // uniform over the workgroup
    fetch(slice0);
    put(0);
    __syncthreads();
    for (int s = slice0; s < slice1; ++s) {
        const int buf = (s - slice0) & 1;
        if (s + 1 < slice1) fetch(s + 1);
        const char* base = lds + 2 * buf * P::BYTES;
#pragma unroll
        for (int h = 0; h < P::BK / 32; ++h) {
            u32x4 a[4], b[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                a[i] = frag(base, 64 * (w4 & 1) + 16 * i, h);
                b[i] = frag(base + P::BYTES, 64 * (w4 >> 1) + 16 * i, h);
            }
#pragma unroll
            for (int i = 0; i < 4; ++i)
#pragma unroll
                for (int j = 0; j < 4; ++j) acc[i][j] = mfma16<IO>(a[i], b[j], acc[i][j]);
        }
        if (s + 1 < slice1) put(buf ^ 1);
        lds_barrier();
    }
}

}  // namespace gemm
}  // namespace vrwkv
