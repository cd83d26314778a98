// Splitting a wkv6 sequence over workgroups (gfx950): the states that the chunked kernels start a segment with.
//
// A (b,h) sequence is a chain over its 32-token chunks, so a call with few sequences leaves most of the chip idle and
// pays the chain's latency (24 sequences of 4150 tokens: 130 steps of 2.8 us).  Such a call cuts every sequence into
// nseg segments of whole chunks.  This kernel computes, for every segment by itself, the state its own tokens leave
// behind in both token directions and the segment's total decay; a scan over the segments turns them into the states that
// enter each segment, and the main kernel's passes start from those.  Per segment and direction, with P the
// cumulative log2 decay from the segment's first token (Pex exclusive of the token):
//   up    L[j][i] = sum_m 2^(Pend - P_m)[j] k_m[j] v_m[i]      the state behind the segment's last token
//   down  L[j][i] = sum_m 2^(Pex_m)[j]      k_m[j] v_m[i]      the state in front of its first token
// The chunks are walked upwards: the up state is rescaled by the chunk's decay and added to, the down state takes its
// factors relative to the segment's start (all exponents <= 0), so one pass over k, v, w serves both.
//
// Bound by latency and vector-ALU work, not by memory (k, v, w are read once, 32 KB of states per segment written): one
// workgroup of four waves per segment, element-wise stage and matrix stage alternating, rows requested two chunks ahead;
// a third of the main kernel's work per chunk.
#pragma once
#include "wkv6_chunk_common.h"

namespace vrwkv {
namespace wkv6_detail {

constexpr int SEG_MAX = 64;                          // segments per sequence (one flag per lane of a wave)
constexpr int SEG_STATE = HN * HN;                   // floats of one state
constexpr int SEG_FLOATS = 2 * SEG_STATE + HN;       // up state, down state, total decay per channel

// Segments of a sequence: the number with the least estimated time, in microseconds measured on bf16 calls.  Per chunk, a
// workgroup of the main kernel takes 2.8 when the chip is nearly empty, 3.6 with one on every CU, 5.6 with two (the most
// that fit), one of the state kernel 1.55 / 2.4; the scan takes 4 to 8, the two extra launches about 7 more.  Measured at
// 24 sequences of 130 chunks: uncut 358, 2 segments 276, 6 103, 10 69, 21 64, 32 72; at 48 sequences of 32 chunks: uncut
// 90, 10 segments 44; at 192 sequences of 32 chunks uncut 93, best cut 108.
inline int wkv6_segments(long long sequences, int nchunk, int cus) {
    auto time = [&](int nseg) {
        const int cps = (nchunk + nseg - 1) / nseg;
        const long long groups = sequences * nseg;
        const double rounds = (double)((groups + 2 * cus - 1) / (2 * cus));
        if (nseg == 1) return 2.0 + rounds * cps * (groups > cus ? 4.5 : 2.8);
        return 20.0 + 0.1 * nseg + rounds * cps * (groups > cus ? 5.6 + 2.4 : 3.6 + 1.55);
    };
    int best = 1;
    double best_time = 0.9 * time(1);
    for (int nseg = 2; nseg <= SEG_MAX && nseg <= nchunk && sequences * nseg <= 4LL * cus; ++nseg) {
        const double t = time(nseg);
        if (t < best_time) { best = nseg; best_time = t; }
    }
    const int cps = (nchunk + best - 1) / best;
    return (nchunk + cps - 1) / cps;                 // every segment non-empty
}

// Workgroup -> (sequence, segment): workgroups are dealt round-robin to the eight XCDs, so the segments of a sequence,
// which read each other's states, are given numbers that are equal modulo 8 and share an L2.
__host__ __device__ inline unsigned seg_grid(long long sequences, int nseg) { return (unsigned)((sequences + 7) / 8 * 8 * nseg); }
__device__ __forceinline__ void seg_of_block(unsigned block, int nseg, int& bh, int& seg) {
    const unsigned y = block >> 3;
    bh = (int)((block & 7) + 8 * (y / nseg));
    seg = (int)(y % nseg);
}

inline size_t seg_workspace_bytes(long long sequences, int nseg) {
    return nseg > 1 ? (size_t)sequences * nseg * (SEG_FLOATS * sizeof(float) + sizeof(int)) : 0;
}

// State fragment of a wave in the main kernel's accumulator order: tile jt of wave w4 holds rows j = 16 jt + 4 g4 + r,
// column i = 16 w4 + c16, as one 16-byte piece per lane.
__device__ __forceinline__ size_t seg_frag(int w4, int jt, int lane) { return (size_t)((w4 * 4 + jt) * 64 + lane) * 4; }

// Exclusive scan over the segments of a sequence: the local states are replaced in place by the states entering the
// segments.  A thread owns four rows of one column in one direction; its loads over the segments are independent of each
// other and go out eight at a time.  Grid: (4, 2, sequences), block 256.  (Folding in the main kernel instead, every
// segment reading all segments before it, moved 160 MB through the L2s at 24 sequences of 21 segments: 10 us more.)
__global__ __launch_bounds__(256) inline void wkv6_seg_fold_kernel(float* __restrict__ ws, int nseg)
{
    const int piece = blockIdx.x * 256 + threadIdx.x;                     // 16-byte piece of the state
    const bool up = blockIdx.y == 0;
    const int j0 = 16 * ((piece >> 6) & 3) + 4 * ((piece >> 4) & 3);      // its rows (see seg_frag)
    const ptrdiff_t step = up ? SEG_FLOATS : -(ptrdiff_t)SEG_FLOATS;
    float* p = ws + ((size_t)blockIdx.z * nseg + (up ? 0 : nseg - 1)) * SEG_FLOATS;
    float* l = p + (up ? 0 : SEG_STATE) + 4 * piece;
    const float* d = p + 2 * SEG_STATE + j0;
    f32x4 s = {0.f, 0.f, 0.f, 0.f};
    constexpr int U = 8;
    for (int q = 0; q < nseg; q += U) {
        f32x4 lv[U], dv[U];
#pragma unroll
        for (int i = 0; i < U; ++i)
            if (q + i < nseg) {
                lv[i] = *reinterpret_cast<const f32x4*>(l + i * step);
                dv[i] = *reinterpret_cast<const f32x4*>(d + i * step);
            }
#pragma unroll
        for (int i = 0; i < U; ++i)
            if (q + i < nseg) {
                *reinterpret_cast<f32x4*>(l + i * step) = s;
#pragma unroll
                for (int e = 0; e < 4; ++e) s[e] = fmaf(dv[i][e], s[e], lv[i][e]);
            }
        l += U * step;
        d += U * step;
    }
}

template <typename IO> struct SegLds {
    static constexpr bool VSPLIT = !__is_same(IO, __hip_bfloat16);
    __bf16 Ah[HN][PS], Al[HN][PS], Dh[HN][PS], Dl[HN][PS], Vt[HN][PS], Vtl[VSPLIT ? HN : 1][PS];   // [channel][token]
    float C2[HN], Tot[2][8][HN];
};

// Element-wise stage: a half wave owns four tokens of the chunk, a lane two neighbouring channels (one 4- or 8-byte
// load per row).
template <typename IO, typename WT, bool W_IS_EW>
__global__ __launch_bounds__(256)
void wkv6_seg_state_kernel(const IO* __restrict__ k_, const IO* __restrict__ v_, const WT* __restrict__ w_,
                           float* __restrict__ ws, int* __restrict__ flags, int T, int C, int H, long long sequences, int nseg)
{
    constexpr bool VSPLIT = SegLds<IO>::VSPLIT;
    __shared__ __attribute__((aligned(16))) SegLds<IO> L;
    const int lane = threadIdx.x & 63;
    const int w4 = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    int bh, seg;
    seg_of_block(blockIdx.x, nseg, bh, seg);
    if (bh >= sequences) return;
    const int b = bh / H, h = bh % H;
    const size_t base = (size_t)b * T * C + (size_t)h * HN;
    const int nchunk = (T + LC - 1) / LC, cps = (nchunk + nseg - 1) / nseg;
    const int c0 = seg * cps, c1 = min(c0 + cps, nchunk);
    const int grp = 2 * w4 + (lane >> 5), cp = 2 * (lane & 31);           // token group (tokens 4 grp ..), first channel
    using RawIO = typename BufRaw<2 * sizeof(IO)>::type;
    using RawW = typename BufRaw<2 * sizeof(WT)>::type;
    const unsigned span_io = (unsigned)(((size_t)(T - 1) * C + HN) * sizeof(IO)), span_w = (unsigned)(((size_t)(T - 1) * C + HN) * sizeof(WT));
    const __amdgpu_buffer_rsrc_t rsk = make_rsrc(k_ + base, span_io), rsv = make_rsrc(v_ + base, span_io), rsw = make_rsrc(w_ + base, span_w);
    RawIO kraw[2][4], vraw[2][4];                                         // rows of two chunks: the current one and the next
    RawW wraw[2][4];
    // rows past T (last chunk only) lie outside the descriptors and read 0: k = 0 switches such a token off, and its
    // decay is set to 1 below
    auto fetch = [&](int c, int s) {
        const unsigned t0 = (unsigned)(c * LC + 4 * grp);
#pragma unroll
        for (int m = 0; m < 4; ++m) {
            const unsigned e = (t0 + m) * C + cp;
            wraw[s][m] = BufRaw<2 * sizeof(WT)>::ld(rsw, e * (unsigned)sizeof(WT), 0);
            kraw[s][m] = BufRaw<2 * sizeof(IO)>::ld(rsk, e * (unsigned)sizeof(IO), 0);
            vraw[s][m] = BufRaw<2 * sizeof(IO)>::ld(rsv, e * (unsigned)sizeof(IO), 0);
        }
    };
    auto two = [](RawIO raw, float (&o)[2]) { IO t[2]; __builtin_memcpy(t, &raw, sizeof(raw)); o[0] = to_f32(t[0]); o[1] = to_f32(t[1]); };
    float p[2][4];                                                        // cumulative log2 decays inside the group
    auto decays = [&](int c, int s) {
#pragma unroll
        for (int m = 0; m < 4; ++m) {
            WT t[2];
            __builtin_memcpy(t, &wraw[s][m], sizeof(wraw[s][m]));
#pragma unroll
            for (int e = 0; e < 2; ++e) {
                const float fw = to_f32(t[e]);
                p[e][m] = W_IS_EW ? fw * LOG2E : -fast_exp2(fmaf(fw, LOG2E, LOG2_LOG2E));
            }
        }
        if ((c + 1) * LC > T) {                                           // wave-uniform: some token of the chunk is past T
#pragma unroll
            for (int m = 0; m < 4; ++m)
                if (c * LC + 4 * grp + m >= T) p[0][m] = p[1][m] = 0.f;
        }
#pragma unroll
        for (int m = 1; m < 4; ++m) { p[0][m] += p[0][m - 1]; p[1][m] += p[1][m - 1]; }
        *reinterpret_cast<f32x2*>(&L.Tot[s][grp][cp]) = f32x2{p[0][3], p[1][3]};
    };
    f32x4 A[4], D[4];                                                     // up and down states, rows j = 16 jt + 4 g4 + r, column i
#pragma unroll
    for (int jt = 0; jt < 4; ++jt) A[jt] = D[jt] = f32x4{0.f, 0.f, 0.f, 0.f};
    float base_p[2] = {0.f, 0.f};                                         // log2 decay from the segment's start to the chunk
    bool out_of_range = false;
    fetch(c0, 0);
    fetch(c0 + 1, 1);                                                     // (past the segment's end: read and not used)
    decays(c0, 0);
    lds_barrier();
    auto step = [&](int c, auto buf_) {
        constexpr int buf = buf_;
        // log2 decay in front of the lane's group and behind it: sums over the groups of the other waves with wave-uniform
        // weights, then this wave's other half
        float before[2] = {0.f, 0.f}, rest[2] = {0.f, 0.f};
        const bool upper = lane >= 32;
#pragma unroll
        for (int g = 0; g < 8; ++g) {
            const f32x2 t = *reinterpret_cast<const f32x2*>(&L.Tot[buf][g][cp]);
            const float wb = (g >> 1) < w4 ? 1.f : 0.f, wr = (g >> 1) > w4 ? 1.f : 0.f;
#pragma unroll
            for (int e = 0; e < 2; ++e) { before[e] = fmaf(wb, t[e], before[e]); rest[e] = fmaf(wr, t[e], rest[e]); }
        }
        const f32x2 sib = *reinterpret_cast<const f32x2*>(&L.Tot[buf][grp ^ 1][cp]);
#pragma unroll
        for (int e = 0; e < 2; ++e) {
            before[e] += upper ? sib[e] : 0.f;
            rest[e] += upper ? 0.f : sib[e];
        }
        unsigned ah[2][2], al[2][2], dh[2][2], dl[2][2], vh[2][2], vl[2][2];
        float p31[2];
#pragma unroll
        for (int e = 0; e < 2; ++e) {
            p31[e] = before[e] + p[e][3] + rest[e];
            out_of_range |= !(p31[e] >= -SAFE_DECAY * LOG2E);
        }
#pragma unroll
        for (int m = 0; m < 4; m += 2) {
            float k0[2], k1[2], v0[2], v1[2];
            two(kraw[buf][m], k0); two(kraw[buf][m + 1], k1);
            two(vraw[buf][m], v0); two(vraw[buf][m + 1], v1);
#pragma unroll
            for (int e = 0; e < 2; ++e) {
                const float tail = p[e][3] + rest[e];
                const float fa0 = fast_exp2(tail - p[e][m]), fa1 = fast_exp2(tail - p[e][m + 1]);
                const float pre = base_p[e] + before[e];
                const float fd0 = fast_exp2(m ? pre + p[e][m - 1] : pre), fd1 = fast_exp2(pre + p[e][m]);
                const float a0 = k0[e] * fa0, a1 = k1[e] * fa1, d0 = k0[e] * fd0, d1 = k1[e] * fd1;
                ah[e][m / 2] = pack_bf16(a0, a1);
                al[e][m / 2] = pack_bf16(a0 - bf16_lo(ah[e][m / 2]), a1 - bf16_hi(ah[e][m / 2]));
                dh[e][m / 2] = pack_bf16(d0, d1);
                dl[e][m / 2] = pack_bf16(d0 - bf16_lo(dh[e][m / 2]), d1 - bf16_hi(dh[e][m / 2]));
                vh[e][m / 2] = pack_bf16(v0[e], v1[e]);
                if constexpr (VSPLIT) vl[e][m / 2] = pack_bf16(v0[e] - bf16_lo(vh[e][m / 2]), v1[e] - bf16_hi(vh[e][m / 2]));
            }
        }
#pragma unroll
        for (int e = 0; e < 2; ++e) {
            auto put = [&](__bf16 (*arr)[PS], const unsigned (&x)[2]) { *reinterpret_cast<uint2*>(&arr[cp + e][4 * grp]) = make_uint2(x[0], x[1]); };
            put(L.Ah, ah[e]); put(L.Al, al[e]); put(L.Dh, dh[e]); put(L.Dl, dl[e]); put(L.Vt, vh[e]);
            if constexpr (VSPLIT) put(L.Vtl, vl[e]);
            base_p[e] += p31[e];
        }
        if (grp == 0) *reinterpret_cast<f32x2*>(&L.C2[cp]) = f32x2{fast_exp2(p31[0]), fast_exp2(p31[1])};
        lds_barrier();
        fetch(c + 2, buf);
        {
            const int g4 = lane >> 4, c16 = lane & 15, icol = 16 * w4 + c16;
            const bf16x8 bv = *reinterpret_cast<const bf16x8*>(&L.Vt[icol][8 * g4]);
            bf16x8 bvl;
            if constexpr (VSPLIT) bvl = *reinterpret_cast<const bf16x8*>(&L.Vtl[icol][8 * g4]);
#pragma unroll
            for (int jt = 0; jt < 4; ++jt) {
                const f32x4 c2 = *reinterpret_cast<const f32x4*>(&L.C2[16 * jt + 4 * g4]);
                const bf16x8 xah = *reinterpret_cast<const bf16x8*>(&L.Ah[16 * jt + c16][8 * g4]);
                const bf16x8 xal = *reinterpret_cast<const bf16x8*>(&L.Al[16 * jt + c16][8 * g4]);
                const bf16x8 xdh = *reinterpret_cast<const bf16x8*>(&L.Dh[16 * jt + c16][8 * g4]);
                const bf16x8 xdl = *reinterpret_cast<const bf16x8*>(&L.Dl[16 * jt + c16][8 * g4]);
                A[jt] *= c2;
                A[jt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(xah, bv, A[jt], 0, 0, 0);
                D[jt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(xdh, bv, D[jt], 0, 0, 0);
                A[jt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(xal, bv, A[jt], 0, 0, 0);
                D[jt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(xdl, bv, D[jt], 0, 0, 0);
                if constexpr (VSPLIT) {
                    A[jt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(xah, bvl, A[jt], 0, 0, 0);
                    D[jt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(xdh, bvl, D[jt], 0, 0, 0);
                }
            }
        }
        decays(c + 1, buf ^ 1);
        lds_barrier();
    };
    for (int c = c0; c < c1; c += 2) {
        step(c, std::integral_constant<int, 0>{});
        if (c + 1 < c1) step(c + 1, std::integral_constant<int, 1>{});
    }
    float* out = ws + ((size_t)bh * nseg + seg) * SEG_FLOATS;
#pragma unroll
    for (int jt = 0; jt < 4; ++jt) {
        *reinterpret_cast<f32x4*>(out + seg_frag(w4, jt, lane)) = A[jt];
        *reinterpret_cast<f32x4*>(out + SEG_STATE + seg_frag(w4, jt, lane)) = D[jt];
    }
    // every wave's half waves saw the same chunk totals: wave 0's first half speaks for all
    if (w4 == 0) {
        if (lane < 32) *reinterpret_cast<f32x2*>(out + 2 * SEG_STATE + cp) = f32x2{fast_exp2(base_p[0]), fast_exp2(base_p[1])};
        const bool any = __builtin_amdgcn_ballot_w64(out_of_range) != 0ull;
        if (lane == 0) flags[(size_t)bh * nseg + seg] = any ? 1 : 0;
    }
}

}  // namespace wkv6_detail
}  // namespace vrwkv
