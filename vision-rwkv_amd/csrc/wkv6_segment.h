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
#include <algorithm>

namespace vrwkv {
namespace wkv6_detail {

constexpr int PART_WAVES = 8, PART = 16 * PART_WAVES;   // waves of a workgroup of the tile kernels, tokens it holds at a time
constexpr int SEG_MAX = 64;                          // segments per sequence (one flag per lane of a wave)
constexpr int SEG_SEQUENCES = 65535;                 // sequences of a cut call (the fold kernel's grid; by the rule below, 4 per CU at most)
constexpr int SEG_STATE = HN * HN;                   // floats of one state
constexpr int SEG_FLOATS = 2 * SEG_STATE + HN;       // forward: up state, down state, total decay per channel
constexpr int BWD_SEG_FLOATS = 4 * SEG_STATE + HN;   // backward: S up, G up, S down, G down, total decay per channel

// Segments of a sequence: the number with the least estimated time, where that is less than uncut by a margin.  Sequences of up to
// 256 tokens stay whole, forward and backward: the results of a (b,h) then do not depend on how many others are in the call.
// Those of longer sequences do, in their last bits (a caller that minds leaves the forward's workspace away).
//
// Backward (both sweeps), in microseconds measured on bf16 calls: a step (one chunk) of the main kernel while its CU holds one workgroup, and more per
// further workgroup that its CU has to run (two at a time fit); the state kernel's step per workgroup on a CU; the scan and the extra launches.
// At 24 sequences of 130 chunks uncut 1381, 10 segments 194, 21 163, 32 193; at 192 of 32 chunks
// uncut 376, 4 segments 310; at 9 of 7 chunks uncut 78, 7 segments 42; at 192 of 7 chunks uncut 84, best cut 103
struct SegCosts { double one, each, state, fixed, per_segment; };
constexpr SegCosts SEG_BWD = {11.5, 9.0, 1.5, 32.0, 0.1};
inline int wkv6_segments(long long sequences, int nchunk, int cus, const SegCosts& k, double& us) {
    auto time = [&](int nseg) {
        const int cps = (nchunk + nseg - 1) / nseg;
        const long long per_cu = (sequences * nseg + cus - 1) / cus;
        const double main = cps * (per_cu == 1 ? k.one : k.each * per_cu);
        return nseg == 1 ? main : main + cps * k.state * per_cu + k.fixed + k.per_segment * nseg;
    };
    int best = 1;
    double best_time = 0.8 * time(1);
    for (int nseg = 2; nchunk > 8 && nseg <= SEG_MAX && nseg <= nchunk && sequences * nseg <= 4LL * cus; ++nseg) {
        const double t = time(nseg);
        if (t < best_time) { best = nseg; best_time = t; }
    }
    us = time(best);
    const int cps = (nchunk + best - 1) / best;
    return (nchunk + cps - 1) / cps;                 // every segment non-empty
}

// Forward: the estimate follows the launches as they are.  The grid has a multiple of eight workgroups per segment number (seg_grid), and a compute
// unit runs one to four of them: `step` is a chunk in the main and the state kernel together for each of those counts; `traffic` is the states' way out
// of the state kernel, through the scan and into the main kernel by the thousand segments, `token_traffic` the rows' by the thousand chunks; `fixed` the
// extra launches.  In microseconds, fitted for each type of r, k, v to 1 to 252 sequences of 9 to 130 chunks, uncut and in 2 to 64 segments: 19 000 times, the
// estimate 4.5 % off (standard deviation).  Counts chosen against the best of the sweep: 0.2 % behind on average, 4 (fp32 7) at most.  On 3 200 further shapes
// they are 10 % ahead on average of what the backward's estimate would choose, and at most 6 % behind that or uncut.  us, uncut | segments:
//   fp32   36 sequences of 130 chunks 364 | 6 113, 7 162, 10 127
//          48 of 24                    71 | 6 52, 8 47, 12 56
//          84 of 24                    72 | 2 68, 3 84, 5 65
//         120 of 33                    98 | 2 95, 4 99
// bf16 sequences can also be cut into segments of 128 tokens, one part of the tile kernel each (wkv6_fwd_tile.h): `parts`.  That cut's time is estimated
// from the segments, all of them and those of a sequence (the scan); for a few sequences finer segments of the chunked kernels are ahead (3 of 10 chunks
// 16.5 against 20.3), and where the others leave a sequence whole it has to be a fifth faster by the estimate, which is that far off (192 of 13).  us, uncut | segments (the 128-token cut in brackets):
//          24 of 130                  354 | 10 65, 17 61, 26 76, [33] 62            192 of 32    94 | 4 95, [8] 95, 11 119
//          48 of 64                   174 | 8 59, 10 61, [16] 55, 32 81             192 of 13    41 | 2 58, [4] 50, 5 56
//          96 of 19                    56 | 3 54, [5] 37, 10 54                      96 of 10    32 | 2 36, [3] 36, 5 35
// In fp16 and fp32 a part's operands leave room for one workgroup a compute unit: where all have one, and no sequence more than sixteen, as each folds the
// states of the others; sequences that the others leave whole stay so unless a third is gained.  us, chunked kernels -> parts, fp16 / fp32: 48 sequences of 577 tokens 33 -> 23 / 34 -> 26, 24 of 1024 32 -> 24 / 32 -> 27,
// 24 of 300 23 -> 21 / 23.6 -> 23.4, 12 of 2048 35 -> 26 / 34 -> 30, 3 of 577 20.2 -> 20.2 / 20.6 -> 23.5.
constexpr int FOLD_SEGMENTS = 16;
struct FwdSegCosts { double uncut, uncut_fixed, uncut_traffic, step[4], fixed, per_segment, traffic, token_traffic; };
constexpr FwdSegCosts SEG_FWD[3] = {{2.72, 4.0, 2.23, {3.73, 7.06, 11.09, 14.80}, 9.8, 0.14, 28.5, 3.39},       // VRWKV_F32
                                    {2.65, 5.1, 1.09, {3.53, 5.14, 8.16, 10.48}, 10.8, 0.14, 20.3, 3.44},       // VRWKV_BF16
                                    {2.80, 4.9, 1.33, {3.99, 7.28, 10.68, 14.05}, 9.6, 0.14, 29.9, 1.70}};      // VRWKV_F16
inline int wkv6_fwd_segments(long long sequences, int nchunk, int cus, int type, bool& parts) {
    const FwdSegCosts& k = SEG_FWD[type];
    parts = false;
    const long long padded = (sequences + 7) / 8 * 8;
    if (nchunk <= 8 || padded > cus) return 1;       // more sequences than compute units: a cut only adds work
    int best = 1;
    const double chunks = 1e-3 * (double)nchunk * (double)sequences;
    double best_time = 0.95 * (nchunk * k.uncut + k.uncut_fixed + k.uncut_traffic * chunks);
    for (int nseg = 2; nseg <= SEG_MAX && nseg <= nchunk && padded * nseg <= 4LL * cus; ++nseg) {
        const int cps = (nchunk + nseg - 1) / nseg, per_cu = (int)((padded * nseg + cus - 1) / cus);
        const double t = cps * k.step[per_cu - 1] + k.fixed + k.per_segment * nseg + k.traffic * 1e-3 * (double)(sequences * nseg) + k.token_traffic * chunks;
        if (t < best_time) { best = nseg; best_time = t; }
    }
    constexpr int part = PART / LC;                  // chunks of a part
    if (type == VRWKV_BF16) {
        const int cps = std::max(part, (nchunk + SEG_MAX - 1) / SEG_MAX), nseg = (nchunk + cps - 1) / cps;
        const double t = std::max(19.0 + 0.45 * nseg, 15.0 + 0.25 * nseg + 0.052 * (double)(sequences * nseg));
        parts = t < (best == 1 ? 0.84 : 1.0) * best_time && cps <= 2 * part;
        if (parts) return nseg;
    } else {
        const int nseg = (nchunk + part - 1) / part;
        const double t = (type == VRWKV_F32 ? 21.5 : 19.0) + 0.4 * nseg + 0.01 * (double)(sequences * nseg);
        parts = nseg <= FOLD_SEGMENTS && padded * nseg <= cus && t < (best == 1 ? 0.73 : 0.95) * best_time;
        if (parts) return nseg;
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

// bytes of the segments' states (floats_per_segment each) and flags
inline size_t seg_bytes(long long sequences, int nseg, int floats_per_segment) {
    return nseg > 1 ? (size_t)sequences * nseg * (floats_per_segment * sizeof(float) + sizeof(int)) : 0;
}

// State fragment of a wave in the main kernel's accumulator order: tile jt of wave w4 holds rows j = 16 jt + 4 g4 + r,
// column i = 16 w4 + c16, as one 16-byte piece per lane.
__device__ __forceinline__ size_t seg_frag(int w4, int jt, int lane) { return (size_t)((w4 * 4 + jt) * 64 + lane) * 4; }

// Exclusive scan over the segments of a sequence: the local states (NMAT of them per segment, the upward ones first) are
// replaced in place by the states entering the segments.  A thread owns four neighbouring values of one state -- rows of a
// column, with the decay per row, or (COLS) the other way round; its loads over the segments are independent of each other
// and go out eight at a time.  Grid: (4, NMAT, sequences), block 256.  (Folding in the main kernel instead, every segment
// reading all segments before it, moved 160 MB through the L2s at 24 sequences of 21 segments: 10 us more.)
template <int NMAT, bool COLS>
__global__ __launch_bounds__(256) void wkv6_seg_fold_kernel(float* __restrict__ ws, int nseg)
{
    constexpr int FLOATS = NMAT * SEG_STATE + HN;
    const int piece = blockIdx.x * 256 + threadIdx.x;                     // 16-byte piece of the state (see seg_frag)
    const bool up = blockIdx.y < NMAT / 2;
    const int j0 = COLS ? 16 * (piece >> 8) + (piece & 15) : 16 * ((piece >> 6) & 3) + 4 * ((piece >> 4) & 3);
    const ptrdiff_t step = up ? FLOATS : -(ptrdiff_t)FLOATS;
    float* p = ws + ((size_t)blockIdx.z * nseg + (up ? 0 : nseg - 1)) * FLOATS;
    float* l = p + blockIdx.y * SEG_STATE + 4 * piece;
    const float* d = p + NMAT * SEG_STATE + j0;
    f32x4 s = {0.f, 0.f, 0.f, 0.f};
    constexpr int U = 8;
    for (int q = 0; q < nseg; q += U) {
        f32x4 lv[U], dv[U];
#pragma unroll
        for (int i = 0; i < U; ++i)
            if (q + i < nseg) {
                lv[i] = *reinterpret_cast<const f32x4*>(l + i * step);
                if (COLS) { const float x = d[i * step]; dv[i] = f32x4{x, x, x, x}; }
                else dv[i] = *reinterpret_cast<const f32x4*>(d + i * step);
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

// Operand arrays in LDS: rows of 64 bf16 (eight 16-byte chunks), chunk c of row t at place c ^ (t & 7), so that 16-byte accesses of eight rows and
// 8-byte transposing reads of four fall into distinct banks without padding.
__device__ __forceinline__ unsigned row_chunk(unsigned row, unsigned chunk) { return row * 128u + ((chunk ^ (row & 7u)) << 4); }
// 16 channels (tile ct) of an array x the 32 tokens of block q, as an operand: slot (g4, e) is token 4 g4 + e (e < 4), 16 + 4 g4 + e - 4 (e >= 4)
__device__ __forceinline__ bf16x8 read_across(const unsigned char* arr, int q, int ct, int lane) {
    const int g4 = lane >> 4, c16 = lane & 15;
    const unsigned char* p = arr + row_chunk(4 * g4 + (c16 >> 2), 2 * ct + ((c16 >> 1) & 1)) + 8 * (c16 & 1) + 4096 * q;
    return cat8(lds_read_tr4(reinterpret_cast<const __bf16*>(p)), lds_read_tr4(reinterpret_cast<const __bf16*>(p + 2048)));
}
// eight packed elements of a row, in 16-byte pieces, widened
template <typename T>
__device__ __forceinline__ void widen8(const u32x4* raw, float (&o)[8]) {
    T t[8];
    __builtin_memcpy(t, raw, sizeof(t));
#pragma unroll
    for (int e = 0; e < 8; ++e) o[e] = to_f32(t[e]);
}
// Log2 decays of a row's eight channels from its logits, summed over the row's predecessors among the wave's 16 tokens (lanes of a row of 16)
template <typename WT, bool W_IS_EW>
__device__ __forceinline__ void summed_decays(const u32x4* raw, bool past, float (&x)[8]) {
    widen8<WT>(raw, x);
#pragma unroll
    for (int e = 0; e < 8; ++e) {
        float d = W_IS_EW ? x[e] * LOG2E : -fast_exp2(fmaf(x[e], LOG2E, LOG2_LOG2E));
        d = past ? 0.f : d;
        d += dpp_get<0x111>(d);                      // row_shr:1, 2, 4, 8
        d += dpp_get<0x112>(d);
        d += dpp_get<0x114>(d);
        d += dpp_get<0x118>(d);
        x[e] = d;
    }
}

// How far a part may decay.  The factors of wkv6_fwd_tile.h and wkv6_bwd_tile.h lie between 2^-c and 2^c, c = |P_end| / 2, on r, k, and through those on the
// products of two or three rows that are summed next (k v, r gy, gy v r, gy v k), which have to stay in fp32: times 2^c below 2^114 (2^13 terms at most), and
// times 2^-c above 2^-92 by the largest of the part (2^17 for the split operands' last bits and as much again for rows that are smaller than the largest).
// c <= 100 in any case.  Up to c = 40, beyond which a model's decays hardly go, the data is not looked at: products from 2^-69 to 2^74 are good there, what
// the chunked kernels ask for at the end of their own range (60 nats over 32 tokens).  What does not fit is those kernels'.  Looking costs the parts beyond
// c = 40 a barrier and their rows' arrival ahead of it (64 x 196 x 768 bf16 forward 46.4 -> 47.6 to 49 us, backward 158 -> 170), the others nothing.
constexpr float PART_FREE = 80.f, PART_RANGE = 200.f;                     // log2
template <typename T>
__device__ __forceinline__ float largest16(const u32x4* a, const u32x4* b) {         // |x| of a lane's 16 elements
    float x[8], y[8], m = 0.f;
    widen8<T>(a, x);
    widen8<T>(b, y);
#pragma unroll
    for (int e = 0; e < 8; ++e) m = fmaxf(m, fmaxf(fabsf(x[e]), fabsf(y[e])));
    return m;
}
__device__ __forceinline__ float largest_of_wave(float m) {
    m = fmaxf(m, dpp_get<0x111>(m));                 // row_shr:1, 2, 4, 8
    m = fmaxf(m, dpp_get<0x112>(m));
    m = fmaxf(m, dpp_get<0x114>(m));
    m = fmaxf(m, dpp_get<0x118>(m));
    const int x = __builtin_bit_cast(int, m);
    auto row = [&](int l) { return __builtin_bit_cast(float, __builtin_amdgcn_readlane(x, l)); };
    return fmaxf(fmaxf(row(15), row(31)), fmaxf(row(47), row(63)));
}
__device__ __forceinline__ float log2_of_largest(float m) { return m > 0.f ? __builtin_amdgcn_logf(m) : 0.f; }   // (rows of zeros take no part)
__device__ __forceinline__ float part_decay(float smallest, float largest) {         // most log2 decay, from log2 of the products
    return fminf(PART_RANGE, 2.f * fminf(92.f + smallest, 114.f - largest));
}

template <typename IO> struct SegLds {
    static constexpr bool VSPLIT = !__is_same(IO, __hip_bfloat16);
    __bf16 Ah[HN][PS], Al[HN][PS], Dh[HN][PS], Dl[HN][PS], Vt[HN][PS], Vtl[VSPLIT ? HN : 1][PS];   // [channel][token]
    float C2[HN], Tot[2][8][HN];
};

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
    float p[2][4];                                                        // cumulative log2 decays inside the group
    auto decays = [&](int c, int s) {
        pair_log_decays<WT, W_IS_EW>(wraw[s], p);
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
        float before[2], rest[2];                                         // log2 decay in front of the lane's group and behind it
        pair_group_sums(L.Tot[buf], w4, lane, cp, before, rest);
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
            pair_widen<IO>(kraw[buf][m], k0); pair_widen<IO>(kraw[buf][m + 1], k1);
            pair_widen<IO>(vraw[buf][m], v0); pair_widen<IO>(vraw[buf][m + 1], v1);
#pragma unroll
            for (int e = 0; e < 2; ++e) {
                const float tail = p[e][3] + rest[e];
                const float fa0 = fast_exp2(tail - p[e][m]), fa1 = fast_exp2(tail - p[e][m + 1]);
                const float pre = base_p[e] + before[e];
                const float fd0 = fast_exp2(m ? pre + p[e][m - 1] : pre), fd1 = fast_exp2(pre + p[e][m]);
                const float a0 = k0[e] * fa0, a1 = k1[e] * fa1, d0 = k0[e] * fd0, d1 = k1[e] * fd1;
                ah[e][m / 2] = pack_bf16(a0, a1);
                al[e][m / 2] = tail_bf16(a0, a1, ah[e][m / 2]);
                dh[e][m / 2] = pack_bf16(d0, d1);
                dl[e][m / 2] = tail_bf16(d0, d1, dh[e][m / 2]);
                vh[e][m / 2] = pack_bf16(v0[e], v1[e]);
                if constexpr (VSPLIT) vl[e][m / 2] = tail_bf16(v0[e], v1[e], vh[e][m / 2]);
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

// The same in parts of up to 128 tokens: eight waves, a wave prepares 16 tokens in the layout of the matrix operands (lane = token c16, eight channels of
// each half) and then forms a quarter of the columns x half the rows of both states over the part's tokens.  All exponents are <= 0.  Two barriers per 128
// tokens where the kernel above has two per 32; bound by the latency of its loads (two workgroups a compute unit) and by the states' way out.
// 24 sequences of 4150 tokens in 17 segments 22 -> 17.6 us.  The operands of a split v leave room for one workgroup (fp32 there 21 -> 29 us): for calls that
// do not have more.
template <typename IO, typename WT, bool W_IS_EW>
__global__ __launch_bounds__(64 * PART_WAVES, 4)
void wkv6_part_state_kernel(const IO* __restrict__ k_, const IO* __restrict__ v_, const WT* __restrict__ w_,
                           float* __restrict__ ws, int* __restrict__ flags, int T, int C, int H, long long sequences, int nseg)
{
    constexpr bool VSPLIT = !__is_same(IO, __hip_bfloat16);
    constexpr unsigned ES = (unsigned)sizeof(IO), WS = (unsigned)sizeof(WT), ARR = PART * 128u;
    constexpr unsigned AH = 0, AL = ARR, DH = 2 * ARR, DL = 3 * ARR, VH = 4 * ARR, VL = 5 * ARR;
    __shared__ __attribute__((aligned(16))) unsigned char lds[(VSPLIT ? 6 : 5) * ARR];
    int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    int bh, seg;
    seg_of_block(blockIdx.x, nseg, bh, seg);
    if (bh >= sequences) return;
    const size_t base = (size_t)(bh / H) * T * C + (size_t)(bh % H) * HN;
    const int nchunk = (T + LC - 1) / LC, cps = (nchunk + nseg - 1) / nseg;
    const int first = seg * cps * LC, n = min(cps * LC, T - first);
    // rows past T (last part only) lie outside the descriptors and read 0: k = 0 switches such a token off, and its decay is set to 1
    auto fetch = [&](const void* p, int t0, auto& raw, unsigned es) {
        const __amdgpu_buffer_rsrc_t rs = make_rsrc(static_cast<const char*>(p) + base * es, (unsigned)(((size_t)(T - 1) * C + HN) * es));
        constexpr int pieces = sizeof(raw[0]) / 16;
        const unsigned vo = ((unsigned)(lane & 15) * C + 8 * (lane >> 4)) * es, so = (unsigned)(t0 + 16 * wave) * C * es;
#pragma unroll
        for (int kb = 0; kb < 2; ++kb)
#pragma unroll
            for (int i = 0; i < pieces; ++i) raw[kb][i] = BufRaw<16>::ld(rs, vo + 32u * kb * es + 16u * i, so);
    };
    const int jt0 = 2 * (wave >> 2), it0 = wave & 3;                      // the wave's tiles: rows 16 (jt0 + q) + 4 g4 + r, column 16 it0 + c16
    f32x4 A[2], D[2];                                                     // up and down states
    A[0] = A[1] = D[0] = D[1] = f32x4{0.f, 0.f, 0.f, 0.f};
    float base_p = 0.f;                                                   // log2 decay from the segment's start to the part, channel `lane`
    bool out_of_range = false;
    u32x4 wraw[2][WS / 2], kraw[2][ES / 2], vraw[2][ES / 2];
    fetch(w_, first, wraw, WS);
    fetch(k_, first, kraw, ES);
    fetch(v_, first, vraw, ES);
#pragma unroll 1
    for (int at = 0; at < n; at += PART) {
        asm volatile("" : "+v"(lane));
        const int np = min(n - at, PART), nb = (np + LC - 1) / LC, g4 = lane >> 4, c16 = lane & 15;
        float x[2][8];
#pragma unroll
        for (int kb = 0; kb < 2; ++kb) {
            summed_decays<WT, W_IS_EW>(wraw[kb], 16 * wave + c16 >= np, x[kb]);
            if (c16 == 15) {
#pragma unroll
                for (int hf = 0; hf < 2; ++hf)
                    *reinterpret_cast<f32x4*>(lds + AH + 256 * wave + 128 * kb + 32 * g4 + 16 * hf) =
                        f32x4{x[kb][4 * hf], x[kb][4 * hf + 1], x[kb][4 * hf + 2], x[kb][4 * hf + 3]};
            }
        }
        lds_barrier();
        float total = 0.f;
        {
            float before = 0.f, t[PART_WAVES];
#pragma unroll
            for (int g = 0; g < PART_WAVES; ++g) {
                t[g] = *reinterpret_cast<const float*>(lds + AH + 256 * g + 4 * lane);
                before += g < wave ? t[g] : 0.f;
                total += t[g];
            }
#pragma unroll
            for (int g = 0; g < PART_WAVES; g += 2) out_of_range |= !(t[g] + t[g + 1] >= -SAFE_DECAY * LOG2E);    // a 32-token chunk
            float* const own = reinterpret_cast<float*>(lds + AL + 2048 * wave);                                  // (in the wave's own rows)
            own[lane] = before;
            own[HN + lane] = total;
            own[2 * HN + lane] = base_p;
        }
        lds_barrier();                                                    // the sums are read: their place is written below
        f32x4 bs[2][2], tt[2][2], bp[2][2];
#pragma unroll
        for (int kb = 0; kb < 2; ++kb)
#pragma unroll
            for (int hf = 0; hf < 2; ++hf) {
                const unsigned char* own = lds + AL + 2048 * wave + 128 * kb + 32 * g4 + 16 * hf;
                bs[kb][hf] = *reinterpret_cast<const f32x4*>(own);
                tt[kb][hf] = *reinterpret_cast<const f32x4*>(own + 256) - bs[kb][hf];         // from the wave's start to the part's end
                bp[kb][hf] = *reinterpret_cast<const f32x4*>(own + 512) + bs[kb][hf];         // from the segment's start to the wave's
            }
#pragma unroll
        for (int kb = 0; kb < 2; ++kb) {
            const unsigned to = row_chunk(16 * wave + c16, 4 * kb + g4);
            float k8[8], o8[8];
            bf16x8 hi, lo;
            widen8<IO>(kraw[kb], k8);
#pragma unroll
            for (int e = 0; e < 8; ++e) o8[e] = k8[e] * fast_exp2(tt[kb][e >> 2][e & 3] - x[kb][e]);
            split8<true>(o8, hi, lo);
            *reinterpret_cast<bf16x8*>(lds + AH + to) = hi;
            *reinterpret_cast<bf16x8*>(lds + AL + to) = lo;
#pragma unroll
            for (int e = 0; e < 8; ++e) o8[e] = k8[e] * fast_exp2(bp[kb][e >> 2][e & 3] + dpp_get<0x111>(x[kb][e]));
            split8<true>(o8, hi, lo);
            *reinterpret_cast<bf16x8*>(lds + DH + to) = hi;
            *reinterpret_cast<bf16x8*>(lds + DL + to) = lo;
            if constexpr (!VSPLIT) {
                *reinterpret_cast<u32x4*>(lds + VH + to) = vraw[kb][0];
            } else {
                widen8<IO>(vraw[kb], o8);
                split8<true>(o8, hi, lo);
                *reinterpret_cast<bf16x8*>(lds + VH + to) = hi;
                *reinterpret_cast<bf16x8*>(lds + VL + to) = lo;
            }
        }
        lds_barrier();
        if (at + PART < n) {
            fetch(w_, first + at + PART, wraw, WS);
            fetch(k_, first + at + PART, kraw, ES);
            fetch(v_, first + at + PART, vraw, ES);
        }
        if (at > 0) {                                                     // the up state over this part's decay
            const float f = fast_exp2(total);
#pragma unroll
            for (int q = 0; q < 2; ++q)
#pragma unroll
                for (int e = 0; e < 4; ++e) A[q][e] *= __shfl(f, 16 * (jt0 + q) + 4 * g4 + e);
        }
#pragma unroll 1
        for (int q = 0; q < nb; ++q) {
            const bf16x8 vv = read_across(lds + VH, q, it0, lane);
#pragma unroll
            for (int j = 0; j < 2; ++j) {
                const bf16x8 ah = read_across(lds + AH, q, jt0 + j, lane), al = read_across(lds + AL, q, jt0 + j, lane);
                const bf16x8 dh = read_across(lds + DH, q, jt0 + j, lane), dl = read_across(lds + DL, q, jt0 + j, lane);
                A[j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ah, vv, A[j], 0, 0, 0);
                D[j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(dh, vv, D[j], 0, 0, 0);
                A[j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(al, vv, A[j], 0, 0, 0);
                D[j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(dl, vv, D[j], 0, 0, 0);
                if constexpr (VSPLIT) {
                    const bf16x8 vl = read_across(lds + VL, q, it0, lane);
                    A[j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ah, vl, A[j], 0, 0, 0);
                    D[j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(dh, vl, D[j], 0, 0, 0);
                }
            }
        }
        base_p += total;
        lds_barrier();                                                    // the operands' place is written next
    }
    float* out = ws + ((size_t)bh * nseg + seg) * SEG_FLOATS;
#pragma unroll
    for (int q = 0; q < 2; ++q) {
        *reinterpret_cast<f32x4*>(out + seg_frag(it0, jt0 + q, lane)) = A[q];
        *reinterpret_cast<f32x4*>(out + SEG_STATE + seg_frag(it0, jt0 + q, lane)) = D[q];
    }
    if (wave == 0) {                                                      // every wave saw all totals
        out[2 * SEG_STATE + lane] = fast_exp2(base_p);
        const bool any = __builtin_amdgcn_ballot_w64(out_of_range) != 0ull;
        if (lane == 0) flags[(size_t)bh * nseg + seg] = any ? 1 : 0;
    }
}

// The same for the backward's sweeps, which carry two states each: S (k, v) and the adjoint state G (r, gy), up and down.
// A wave owns 16 columns j and the rows i of all four (the order in which the sweeps read them).
template <typename IO> struct BwdSegLds {
    static constexpr bool VSPLIT = !__is_same(IO, __hip_bfloat16);
    __bf16 Op[4][2][HN][PS];                                              // k up, r up, k down, r down: head, tail
    __bf16 Vt[HN][PS], Vtl[VSPLIT ? HN : 1][PS], Gh[HN][PS], Gl[HN][PS];
    float C2[HN], Tot[8][HN];
};
template <typename IO, typename WT, bool W_IS_EW>
__global__ __launch_bounds__(256, 2)
void wkv6_bwd_seg_state_kernel(const IO* __restrict__ r_, const IO* __restrict__ k_, const IO* __restrict__ v_, const WT* __restrict__ w_,
                               const float* __restrict__ gy_, float* __restrict__ ws, int* __restrict__ flags, int T, int C, int H,
                               long long sequences, int nseg)
{
    constexpr bool VSPLIT = BwdSegLds<IO>::VSPLIT;
    constexpr unsigned ES = (unsigned)sizeof(IO), WS = (unsigned)sizeof(WT);
    __shared__ __attribute__((aligned(16))) BwdSegLds<IO> L;
    const int lane = threadIdx.x & 63;
    const int w4 = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    int bh, seg;
    seg_of_block(blockIdx.x, nseg, bh, seg);
    if (bh >= sequences) return;
    const int b = bh / H, h = bh % H;
    const size_t base = (size_t)b * T * C + (size_t)h * HN;
    const int nchunk = (T + LC - 1) / LC, cps = (nchunk + nseg - 1) / nseg;
    const int c0 = seg * cps, c1 = min(c0 + cps, nchunk);
    const int grp = 2 * w4 + (lane >> 5), cp = 2 * (lane & 31);
    using RawIO = typename BufRaw<2 * ES>::type;
    using RawW = typename BufRaw<2 * WS>::type;
    const unsigned n_el = (unsigned)((size_t)(T - 1) * C + HN);
    const __amdgpu_buffer_rsrc_t rsr = make_rsrc(r_ + base, n_el * ES), rsk = make_rsrc(k_ + base, n_el * ES), rsv = make_rsrc(v_ + base, n_el * ES),
                                 rsw = make_rsrc(w_ + base, n_el * WS), rsg = make_rsrc(gy_ + base, n_el * 4);
    RawIO rraw[4], kraw[4], vraw[4];
    RawW wraw[4];
    f32x2 graw[4];
    auto fetch = [&](int c) {
#pragma unroll
        for (int m = 0; m < 4; ++m) {
            const unsigned e = (unsigned)(c * LC + 4 * grp + m) * C + cp;
            wraw[m] = BufRaw<2 * WS>::ld(rsw, e * WS, 0);
            rraw[m] = BufRaw<2 * ES>::ld(rsr, e * ES, 0);
            kraw[m] = BufRaw<2 * ES>::ld(rsk, e * ES, 0);
            vraw[m] = BufRaw<2 * ES>::ld(rsv, e * ES, 0);
            graw[m] = __builtin_bit_cast(f32x2, BufRaw<8>::ld(rsg, e * 4u, 0));
        }
    };
    float p[2][4];
    auto decays = [&](int c) {
        pair_log_decays<WT, W_IS_EW>(wraw, p);
        if ((c + 1) * LC > T) {
#pragma unroll
            for (int m = 0; m < 4; ++m)
                if (c * LC + 4 * grp + m >= T) p[0][m] = p[1][m] = 0.f;
        }
#pragma unroll
        for (int m = 1; m < 4; ++m) { p[0][m] += p[0][m - 1]; p[1][m] += p[1][m - 1]; }
        *reinterpret_cast<f32x2*>(&L.Tot[grp][cp]) = f32x2{p[0][3], p[1][3]};
    };
    f32x4 st[4][4];                                                       // S up, G up, S down, G down; tile it: rows i = 16 it + 4 g4 + r
#pragma unroll
    for (int q = 0; q < 4; ++q)
#pragma unroll
        for (int it = 0; it < 4; ++it) st[q][it] = f32x4{0.f, 0.f, 0.f, 0.f};
    float base_p[2] = {0.f, 0.f};
    bool out_of_range = false;
    fetch(c0);
    decays(c0);
    lds_barrier();
    for (int c = c0; c < c1; ++c) {
        float before[2], rest[2], tail[2], pre[2], p31[2];
        pair_group_sums(L.Tot, w4, lane, cp, before, rest);
#pragma unroll
        for (int e = 0; e < 2; ++e) {
            tail[e] = p[e][3] + rest[e];
            p31[e] = before[e] + tail[e];
            pre[e] = base_p[e] + before[e];
            out_of_range |= !(p31[e] >= -SAFE_DECAY * LOG2E);
        }
        unsigned op[4][2][2][2], vh[2][2], vl[2][2], gh[2][2], gl[2][2];  // [operand][head, tail][channel][token pair]
        auto split = [&](float x0, float x1, unsigned& hi, unsigned& lo) {
            hi = pack_bf16(x0, x1);
            lo = tail_bf16(x0, x1, hi);
        };
#pragma unroll
        for (int m = 0; m < 4; m += 2) {
            float r0[2], r1[2], k0[2], k1[2], v0[2], v1[2];
            pair_widen<IO>(rraw[m], r0); pair_widen<IO>(rraw[m + 1], r1);
            pair_widen<IO>(kraw[m], k0); pair_widen<IO>(kraw[m + 1], k1);
            pair_widen<IO>(vraw[m], v0); pair_widen<IO>(vraw[m + 1], v1);
#pragma unroll
            for (int e = 0; e < 2; ++e) {
                const float fa0 = fast_exp2(tail[e] - p[e][m]), fa1 = fast_exp2(tail[e] - p[e][m + 1]);
                const float fd0 = fast_exp2(m ? pre[e] + p[e][m - 1] : pre[e]), fd1 = fast_exp2(pre[e] + p[e][m]);
                split(k0[e] * fa0, k1[e] * fa1, op[0][0][e][m / 2], op[0][1][e][m / 2]);
                split(r0[e] * fa0, r1[e] * fa1, op[1][0][e][m / 2], op[1][1][e][m / 2]);
                split(k0[e] * fd0, k1[e] * fd1, op[2][0][e][m / 2], op[2][1][e][m / 2]);
                split(r0[e] * fd0, r1[e] * fd1, op[3][0][e][m / 2], op[3][1][e][m / 2]);
                split(graw[m][e], graw[m + 1][e], gh[e][m / 2], gl[e][m / 2]);
                split(v0[e], v1[e], vh[e][m / 2], vl[e][m / 2]);
            }
        }
#pragma unroll
        for (int e = 0; e < 2; ++e) {
            auto put = [&](__bf16 (*arr)[PS], const unsigned (&x)[2]) { *reinterpret_cast<uint2*>(&arr[cp + e][4 * grp]) = make_uint2(x[0], x[1]); };
#pragma unroll
            for (int q = 0; q < 4; ++q) { put(L.Op[q][0], op[q][0][e]); put(L.Op[q][1], op[q][1][e]); }
            put(L.Vt, vh[e]);
            if constexpr (VSPLIT) put(L.Vtl, vl[e]);
            put(L.Gh, gh[e]);
            put(L.Gl, gl[e]);
            base_p[e] += p31[e];
        }
        if (grp == 0) *reinterpret_cast<f32x2*>(&L.C2[cp]) = f32x2{fast_exp2(p31[0]), fast_exp2(p31[1])};
        lds_barrier();
        if (c + 1 < c1) fetch(c + 1);
        {
            const int g4 = lane >> 4, c16 = lane & 15, j = 16 * w4 + c16;
            const float c2 = L.C2[j];
            bf16x8 bh_[4], bl_[4];
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                bh_[q] = *reinterpret_cast<const bf16x8*>(&L.Op[q][0][j][8 * g4]);
                bl_[q] = *reinterpret_cast<const bf16x8*>(&L.Op[q][1][j][8 * g4]);
            }
#pragma unroll
            for (int it = 0; it < 4; ++it) {
                const bf16x8 av = *reinterpret_cast<const bf16x8*>(&L.Vt[16 * it + c16][8 * g4]);
                bf16x8 avl;
                if constexpr (VSPLIT) avl = *reinterpret_cast<const bf16x8*>(&L.Vtl[16 * it + c16][8 * g4]);
                const bf16x8 ag = *reinterpret_cast<const bf16x8*>(&L.Gh[16 * it + c16][8 * g4]);
                const bf16x8 agl = *reinterpret_cast<const bf16x8*>(&L.Gl[16 * it + c16][8 * g4]);
                st[0][it] *= c2;
                st[1][it] *= c2;
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    const bool g = q & 1;
                    st[q][it] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(g ? ag : av, bh_[q], st[q][it], 0, 0, 0);
                    st[q][it] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(g ? ag : av, bl_[q], st[q][it], 0, 0, 0);
                    if (g) st[q][it] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(agl, bh_[q], st[q][it], 0, 0, 0);
                    if constexpr (VSPLIT)
                        if (!g) st[q][it] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(avl, bh_[q], st[q][it], 0, 0, 0);
                }
            }
        }
        if (c + 1 < c1) decays(c + 1);
        lds_barrier();
    }
    float* out = ws + ((size_t)bh * nseg + seg) * BWD_SEG_FLOATS;
#pragma unroll
    for (int q = 0; q < 4; ++q)
#pragma unroll
        for (int it = 0; it < 4; ++it) *reinterpret_cast<f32x4*>(out + q * SEG_STATE + seg_frag(w4, it, lane)) = st[q][it];
    if (w4 == 0) {
        if (lane < 32) *reinterpret_cast<f32x2*>(out + 4 * SEG_STATE + cp) = f32x2{fast_exp2(base_p[0]), fast_exp2(base_p[1])};
        const bool any = __builtin_amdgcn_ballot_w64(out_of_range) != 0ull;
        if (lane == 0) flags[(size_t)bh * nseg + seg] = any ? 1 : 0;
    }
}

}  // namespace wkv6_detail
}  // namespace vrwkv
