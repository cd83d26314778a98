// Helpers shared by the chunked matrix-core wkv6 kernels (forward and backward scans) for gfx950: packed bf16
// head / tail splits, DPP moves, the transposing row-sum butterflies and the layout constants of the LDS operands.
#pragma once
#include "vrwkv_common.h"
#include "wkv6_fwd_scalar.h"
#include <type_traits>

namespace vrwkv {
namespace wkv6_detail {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x4 __attribute__((ext_vector_type(4)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

constexpr int LC = 32;           // chunk length
constexpr int HN = 64;           // head size
constexpr int PJ = 72;           // row pitch (bf16) of the [token][channel] operand arrays
constexpr int PS = 40;           // row pitch (bf16) of the [channel][token] operand arrays
constexpr float SAFE_DECAY = 60.f;

__device__ __forceinline__ bf16x8 cat8(bf16x4 a, bf16x4 b) {
    return __builtin_shufflevector(a, b, 0, 1, 2, 3, 4, 5, 6, 7);
}
typedef unsigned u32x4 __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef float f32x2 __attribute__((ext_vector_type(2)));
constexpr float LOG2_LOG2E = 0.5287663729448977f;     // log2(log2(e))
// two fp32 values rounded to bf16 in one register (a low, b high), and the halves widened back
__device__ __forceinline__ unsigned pack_bf16(float a, float b) {
    return __builtin_bit_cast(unsigned, __builtin_convertvector(f32x2{a, b}, bf16x2));
}
__device__ __forceinline__ float bf16_lo(unsigned w) { return __builtin_bit_cast(float, w << 16); }
__device__ __forceinline__ float bf16_hi(unsigned w) { return __builtin_bit_cast(float, w & 0xffff0000u); }
// The tails of a head / tail split: (x0 - head0, x1 - head1) rounded to bf16, with h = pack_bf16(x0, x1).  A head is
// subtracted by one dot-product instruction, x + (head0, head1) . (-1, 0), exact because the other product is zero; shifting
// the head out of its word first takes two.  (The weights are kept opaque: as constants the compiler folds them into an
// inline operand that stands for another pair.)
__device__ __forceinline__ unsigned tail_bf16(float x0, float x1, unsigned h) {
    unsigned lo = 0x0000bf80u, hi = 0xbf800000u;
    asm("" : "+s"(lo), "+s"(hi));
    const bf16x2 hv = __builtin_bit_cast(bf16x2, h);
    return pack_bf16(__builtin_amdgcn_fdot2_f32_bf16(hv, __builtin_bit_cast(bf16x2, lo), x0, false),
                     __builtin_amdgcn_fdot2_f32_bf16(hv, __builtin_bit_cast(bf16x2, hi), x1, false));
}
__device__ __forceinline__ void st_bf16_pair(__bf16* lo, __bf16* hi, unsigned w) {
    *reinterpret_cast<unsigned short*>(lo) = (unsigned short)w;
    *reinterpret_cast<unsigned short*>(hi) = (unsigned short)(w >> 16);
}

// head/tail split of eight fp32 accumulator values into two packed bf16 operands (two values per conversion); DOT forms the
// tails with tail_bf16
template <bool DOT = false>
__device__ __forceinline__ void split8(const float (&x)[8], bf16x8& hi, bf16x8& lo) {
    u32x4 h, l;
#pragma unroll
    for (int p = 0; p < 4; ++p) {
        const unsigned w = pack_bf16(x[2 * p], x[2 * p + 1]);
        h[p] = w;
        l[p] = DOT ? tail_bf16(x[2 * p], x[2 * p + 1], w) : pack_bf16(x[2 * p] - bf16_lo(w), x[2 * p + 1] - bf16_hi(w));
    }
    hi = __builtin_bit_cast(bf16x8, h);
    lo = __builtin_bit_cast(bf16x8, l);
}

// DPP move: lane reads `v` of the lane selected by CTRL (0 where there is none).
template <int CTRL>
__device__ __forceinline__ float dpp_get(float v) {
    return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), CTRL, 0xf, 0xf, true));
}
// 16 values per lane -> per 16-lane row, the row sums of all 16: lane l ends up with the sum over
// its row of value index 8*(l&1) + 4*((l>>1)&1) + 2*((l>>3)&1) + ((l>>2)&1).  Transposing butterfly:
// at each step a lane keeps one half of its values and hands the other half to its partner.
__device__ __forceinline__ float row_sums16(const float (&p)[16], int lane, int& index) {
    const bool b0 = lane & 1, b1 = lane & 2, b2 = lane & 4, b3 = lane & 8;
    float a8[8], a4[4], a2[2];
#pragma unroll
    for (int i = 0; i < 8; ++i) a8[i] = (b0 ? p[8 + i] : p[i]) + dpp_get<0xB1>(b0 ? p[i] : p[8 + i]);     // quad_perm [1,0,3,2]
#pragma unroll
    for (int i = 0; i < 4; ++i) a4[i] = (b1 ? a8[4 + i] : a8[i]) + dpp_get<0x4E>(b1 ? a8[i] : a8[4 + i]); // quad_perm [2,3,0,1]
#pragma unroll
    for (int i = 0; i < 2; ++i) a2[i] = (b3 ? a4[2 + i] : a4[i]) + dpp_get<0x128>(b3 ? a4[i] : a4[2 + i]); // row_ror:8
    const float give = b2 ? a2[0] : a2[1];
    const float from_lo = dpp_get<0x114>(give), from_hi = dpp_get<0x104>(give);   // row_shr:4 (from l-4), row_shl:4 (from l+4)
    const float recv = b2 ? from_lo : from_hi;                            // both moves run with every lane active
    index = (b0 ? 8 : 0) + (b1 ? 4 : 0) + (b3 ? 2 : 0) + (b2 ? 1 : 0);
    return (b2 ? a2[1] : a2[0]) + recv;
}

// ---- element-wise stages with two channels per lane ---------------------------------------------------------------
// A half wave owns four tokens of the chunk, a lane two neighbouring channels: rows are read in 4- or 8-byte pieces, half
// as many accesses as one channel per lane needs.  Wave w4 of a pass holds the token groups 2 w4 (lanes 0..31) and
// 2 w4 + 1 (lanes 32..63) of the eight groups of a chunk.

// log2 decays of four tokens x two channels from the packed rows of w: -log2(e) exp(w) = -exp2(w log2(e) + log2(log2(e)))
template <typename WT, bool W_IS_EW, typename Raw>
__device__ __forceinline__ void pair_log_decays(const Raw (&raw)[4], float (&d)[2][4]) {
#pragma unroll
    for (int m = 0; m < 4; ++m) {
        WT t[2];
        __builtin_memcpy(t, &raw[m], sizeof(raw[m]));
#pragma unroll
        for (int e = 0; e < 2; ++e) {
            const float fw = to_f32(t[e]);
            d[e][m] = W_IS_EW ? fw * LOG2E : -fast_exp2(fmaf(fw, LOG2E, LOG2_LOG2E));
        }
    }
}
// two packed elements widened
template <typename IO, typename Raw>
__device__ __forceinline__ void pair_widen(Raw raw, float (&o)[2]) {
    IO t[2];
    __builtin_memcpy(t, &raw, sizeof(raw));
    o[0] = to_f32(t[0]);
    o[1] = to_f32(t[1]);
}
// From the groups' totals tot[8][64]: the sums in front of the lane's group and behind it, for its channels c, c + 1.
// The other waves' groups enter with wave-uniform weights, this wave's other half by a select.
__device__ __forceinline__ void pair_group_sums(const float (*tot)[HN], int w4, int lane, int c, float (&before)[2], float (&rest)[2]) {
    before[0] = before[1] = rest[0] = rest[1] = 0.f;
#pragma unroll
    for (int g = 0; g < 8; ++g) {
        const f32x2 t = *reinterpret_cast<const f32x2*>(&tot[g][c]);
        const float wb = (g >> 1) < w4 ? 1.f : 0.f, wr = (g >> 1) > w4 ? 1.f : 0.f;
#pragma unroll
        for (int e = 0; e < 2; ++e) { before[e] = fmaf(wb, t[e], before[e]); rest[e] = fmaf(wr, t[e], rest[e]); }
    }
    const bool upper = lane >= 32;
    const f32x2 sib = *reinterpret_cast<const f32x2*>(&tot[2 * w4 + (upper ? 0 : 1)][c]);
#pragma unroll
    for (int e = 0; e < 2; ++e) {
        before[e] += upper ? sib[e] : 0.f;
        rest[e] += upper ? 0.f : sib[e];
    }
}

// ---- operands read across the rows of a [channel][token] array ------------------------------------------------------
// ds_read_b64_tr_b16: inside 16 lanes, lane i receives element (i & 3) of the 8-byte pieces that lanes (i >> 2),
// 4 + (i >> 2), 8 + (i >> 2), 12 + (i >> 2) address.
__device__ __forceinline__ bf16x4 lds_read_tr4(const __bf16* p) {
    typedef short s16x4 __attribute__((ext_vector_type(4)));
    typedef __attribute__((address_space(3))) s16x4 lds_s16x4;
    return __builtin_bit_cast(bf16x4, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4*)p));
}

}  // namespace wkv6_detail
}  // namespace vrwkv
