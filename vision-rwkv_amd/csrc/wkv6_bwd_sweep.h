// wkv6 backward, chunked matrix-core kernel for gfx950 (bf16 MFMA, fp32 accumulate; r, k, v in bf16, fp16 or fp32).
//
// The forward is the sum of two causal passes over the tokens (ascending with the bonus u, descending without).  With
// S_n the state in front of token n in a pass's order, d_n = exp(ld_n), and the adjoint state G_n:
//   S_{n+1} = diag(d_n) S_n + k_n v_n^T,   G_n = r_n gy_n^T + diag(d_n) G_{n+1}
//   gr_n[j] = (S_n gy_n)[j],  gk_n[j] = (G_{n+1} v_n)[j],  gv_n[i] = (G_{n+1}^T k_n)[i]      (+ the bonus terms)
//   gw_n[j] = ld_n[j] (sum_{m>n} (a_m - b_m) - b_n)[j],    a = r (S gy),  b = k (G v)
// (formulas of classification/mmcls_custom/models/backbones/cuda_v6/wkv6_cuda.cu:99-346).
//
// A sweep over the tokens in one direction builds the state S of one pass and the adjoint state G of the other: both
// collect "earlier" tokens with the decay strictly between the two tokens.  So one sweep upwards and one downwards give
// everything, and a sweep reads r, k, v, w, gy once for gr, gk and gv together.  On chunks of 32 tokens in scan order,
// with P the in-chunk cumulative log decay, Pex = P - ld, P31 its end, f1 = e^(Pex-P31), f2 = e^(P31-P):
//   Z_S = diag(e^P31) S,   Z_G = diag(e^P31) G
//   gr_t = f1_t ( sum_{s<t} (k f2)_s (v_s . gy_t)  +  Z_S gy_t )           S' = Z_S + (k f2)^T v
//   gk_t = f1_t ( sum_{s<t} (r f2)_s (gy_s . v_t)  +  Z_G v_t )            G' = Z_G + (r f2)^T gy
//   gv_t =        sum_{s<t} ((r f2)_s . (k f1)_t) gy_s  +  Z_G^T (k f1)_t
// -- three instances of one form (matrix_stage below).  The sweep upwards stores its gr, gk, gv in fp32, the sweep
// downwards reads them back, adds its own and the bonus terms and forms gw: with the sums of both sweeps at hand,
//   gw_n = ld_n (X + sum_{m>n} q_m - t_n),   q = r (gr_up - gr_dn) + k (gk_up - gk_dn),  t = k gk_dn + r gr_dn,
// X = 0 at the sequence's end (between segments of a cut sequence X = sum_i (S G of both passes), taken where the upward
// sweep turns round).
//
// One workgroup of eight waves per (b,h), both sweeps after each other, two workgroups per CU: four waves per SIMD, which is
// what hides the LDS and matrix latencies of the step.  Measured at 64 x 196 x 768 bf16: 190-215 us; four waves with 256
// registers each, two per SIMD, 278; six scans with 1.35 GB of traffic, one per result and pass, 310.  What bounds it is the
// step's latency and the vector ALUs (46 % busy; per step and workgroup 4700 vector instructions beside 480 MFMA), not
// memory (0.61 GB by FETCH_SIZE and WRITE_SIZE).  A chunk step is an element-wise stage (wave: four tokens, lane: channel), a matrix stage and a closing
// stage in the element-wise stage's layout, two LDS-only barriers (the decay sums of the next chunk and gw of the previous
// one ride on them).  In the matrix stage the waves divide the three results: waves 0, 1 form gr and own S (half its
// columns j each, 64 x 32 in their accumulators), waves 2, 3 gk and G with the value channel as the contraction, waves
// 4..7 a quarter of gv each and G the other way round.  Every operand read then belongs to one result (columns of all three
// per wave would read three times as much of LDS).
// Operands lie in LDS once, as [channel][token]: element-wise lanes store four tokens of a channel at a time, and the
// matrix stage reads them along the tokens (16-byte reads) or across (ds_read_b64_tr_b16).  Computed operands (and fp16 /
// fp32 inputs) are split into bf16 head + tail, products head*head + head*tail + tail*head.  128 registers: the matrix stage
// runs in phases that read their operands anew instead of keeping them.
//
// Range: the factors need |P31| <= 60 in every chunk.  A sequence with a chunk outside that range is redone by the same
// workgroup with the sequential sweeps of wkv6_bwd_seq.h.
#pragma once
#include "wkv6_segment.h"
#include "wkv6_bwd_seq.h"

namespace vrwkv {
namespace wkv6_detail {

struct BwdArgs {
    const void *r, *k, *v, *w;                       // (B,T,C): IO, IO, IO, WT
    const float *u, *gy;
    void *gr, *gk, *gv, *gw;                         // results: IO / WT when out16 / w16, else fp32
    float *pr, *pk, *pv, *pw;                        // fp32 sums of the upward sweep (the results themselves when they are fp32)
    float *a, *gu_part;                              // sequential fallback's (2, B,T,C) scratch; (B*nseg, C) partial gu
    size_t a_size;                                   // elements of a tensor
    const float* seg_ws;                             // states entering the segments (nseg > 1); wkv6_bwd_tile.h: those that the segments leave by themselves
    float* seg_own;                                  // room for the former beside the latter
    const int* seg_flags;
    int T, C, H, sequences, nseg, out16, w16;
};

constexpr int BP = 36;                               // row pitch (bf16) of the operand arrays: 18 dwords, so that the 8-byte stores of
                                                     // 32 rows fall into distinct banks
constexpr int RP = 68;                               // row pitch (floats) of the result rows: 16-byte writes of 16 rows hit all banks
// column of the first of a group's four tokens in the [channel][token] arrays: slots in the order of the matrix
// instructions, so that an operand is 16 consecutive bytes (slot (g4, e) <-> token 4 g4 + e for e < 4, 16 + 4 g4 + e - 4 above)
__device__ __forceinline__ int tok_col(int group) { return (group & 3) * 8 + (group >> 2) * 4; }

template <bool VSPLIT>
struct __attribute__((aligned(16))) BwdLds {
    __bf16 KF1h[HN][BP], KF1l[HN][BP], KF2h[HN][BP], KF2l[HN][BP], RF2h[HN][BP], RF2l[HN][BP], GYh[HN][BP], GYl[HN][BP];
    __bf16 Vh[HN][BP], Vl[VSPLIT ? HN : 1][BP];
    float Res[2][LC][RP];                            // gr / f1, gk / f1 of the chunk: [token][channel]
    float F1[LC][HN];                                // the factors f1: kept here over the matrix stage
    float C2[HN], Tot[8][HN], Q[8][HN], X[2][HN], Bon[4][LC], Diag[LC];
};

// Sixteen tokens (tile tb) x 32 channels (half kb) as a matrix operand: lane c16 = token, slot (g4, e) = channel
// 32 kb + 4 g4 + e (e < 4), 32 kb + 16 + 4 g4 + e - 4 (e >= 4) -- the order in which accumulator tiles hold their rows.
__device__ __forceinline__ bf16x8 token_rows(const __bf16 (*arr)[BP], int tb, int kb, int lane) {
    const int g4 = lane >> 4, c16 = lane & 15;
    const __bf16* p = &arr[32 * kb + 4 * g4 + (c16 >> 2)][8 * (c16 & 3) + 4 * tb];
    return cat8(lds_read_tr4(p), lds_read_tr4(p + 16 * BP));
}
__device__ __forceinline__ bf16x8 channel_rows(const __bf16 (*arr)[BP], int row, int g4) {
    const __bf16* p = &arr[row][8 * g4];
    return cat8(*reinterpret_cast<const bf16x4*>(p), *reinterpret_cast<const bf16x4*>(p + 4));
}
__device__ __forceinline__ bf16x8 words_of(unsigned a, unsigned b, unsigned c, unsigned d) { return __builtin_bit_cast(bf16x8, u32x4{a, b, c, d}); }
__device__ __forceinline__ f32x4 mfma(bf16x8 a, bf16x8 b, f32x4 c) { return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0); }

// out^T[o][t] = sum_{s<t} Val[o][s] D[s][t] + sum_c Z[c][o] Q[c][t],  D[s][t] = sum_c Kc[c][s] Q[c][t],  then
// state[c][o] = Z[c][o] + sum_s Kc[c][s] Val[o][s].  st[4 ot + ct]: rows c = 16 ct + 4 g4 + r, column o = 16 (o0 + ot) + c16.
// QS, KS, VS: Q, Kc, Val come as head + tail; LL: tail x tail products too (gr and gk: gw is a difference of their sums, whose
// worst element is at 1.5e-3 of rms at 64 x 196 x 768 with them and at 4.2e-3 without).  ROWS: the state's decay belongs to
// its rows (c), else to its columns (o).  DIAG 1: D[t][t] is written to diag.  DIAG 2: the four partial sums bon[..][t] are
// added to D[t][t] (head + tail).  The phases are kept apart by scheduling barriers: operands of two of them do not fit.
template <bool QS, bool KS, bool VS, bool LL, int NO, bool ROWS, int DIAG, typename Emit>
__device__ __forceinline__ void matrix_stage(const __bf16 (*Qh)[BP], const __bf16 (*Ql)[BP], const __bf16 (*Kh)[BP], const __bf16 (*Kl)[BP],
                                             const __bf16 (*Vh)[BP], const __bf16 (*Vl)[BP], const float* C2, f32x4 (&st)[8], int o0,
                                             int lane, float* diag, const float (*bon)[LC], Emit emit)
{
    const f32x4 zero = {0.f, 0.f, 0.f, 0.f};
    // a fresh copy of the lane number per phase: operands that two phases read are read twice, not carried along
    auto phase = [&]() {
        __builtin_amdgcn_sched_barrier(0);
        asm volatile("" : "+v"(lane));
    };
    // ---- token-token products, blocks (s, t) = (0,0), (0,1), (1,1) of 16 x 16; (1,0) has s > t throughout ----
    f32x4 d[3] = {zero, zero, zero};
#pragma unroll
    for (int kb = 0; kb < 2; ++kb) {
        bf16x8 qh[2], ql[2], kh[2], kl[2];
#pragma unroll
        for (int tb = 0; tb < 2; ++tb) {
            qh[tb] = token_rows(Qh, tb, kb, lane);
            kh[tb] = token_rows(Kh, tb, kb, lane);
            if (QS) ql[tb] = token_rows(Ql, tb, kb, lane);
            if (KS) kl[tb] = token_rows(Kl, tb, kb, lane);
        }
#pragma unroll
        for (int b = 0; b < 3; ++b) d[b] = mfma(kh[b >> 1], qh[(b + 1) >> 1], d[b]);
        if (QS) {
#pragma unroll
            for (int b = 0; b < 3; ++b) d[b] = mfma(kh[b >> 1], ql[(b + 1) >> 1], d[b]);
        }
        if (KS) {
#pragma unroll
            for (int b = 0; b < 3; ++b) d[b] = mfma(kl[b >> 1], qh[(b + 1) >> 1], d[b]);
        }
        phase();
    }
    // ---- out = Z Q: the decayed state straight from its accumulators ----
    f32x4 acc[NO][2];
#pragma unroll
    for (int ot = 0; ot < NO; ++ot) acc[ot][0] = acc[ot][1] = zero;
#pragma unroll
    for (int kb = 0; kb < 2; ++kb) {
        const int g4 = lane >> 4, c16 = lane & 15;
        bf16x8 qh[2], ql[2];
#pragma unroll
        for (int tb = 0; tb < 2; ++tb) {
            qh[tb] = token_rows(Qh, tb, kb, lane);
            if (QS) ql[tb] = token_rows(Ql, tb, kb, lane);
        }
#pragma unroll
        for (int ot = 0; ot < NO; ++ot) {
            float z8[8];
#pragma unroll
            for (int hf = 0; hf < 2; ++hf) {
                f32x4& s = st[4 * ot + 2 * kb + hf];
                if (ROWS) s *= *reinterpret_cast<const f32x4*>(&C2[16 * (2 * kb + hf) + 4 * g4]);
                else s *= C2[16 * (o0 + ot) + c16];
#pragma unroll
                for (int e = 0; e < 4; ++e) z8[4 * hf + e] = s[e];
            }
            bf16x8 zh, zl;
            split8<true>(z8, zh, zl);
#pragma unroll
            for (int tb = 0; tb < 2; ++tb) acc[ot][tb] = mfma(zh, qh[tb], acc[ot][tb]);
#pragma unroll
            for (int tb = 0; tb < 2; ++tb) acc[ot][tb] = mfma(zl, qh[tb], acc[ot][tb]);
            if (QS) {
#pragma unroll
                for (int tb = 0; tb < 2; ++tb) acc[ot][tb] = mfma(zh, ql[tb], acc[ot][tb]);
                if (LL) {
#pragma unroll
                    for (int tb = 0; tb < 2; ++tb) acc[ot][tb] = mfma(zl, ql[tb], acc[ot][tb]);
                }
            }
            __builtin_amdgcn_sched_barrier(0);
        }
        phase();
    }
    // ---- D keeps s < t: a lane holds t = c16, s = 4 g4 + r; masks on the packed words of the two diagonal blocks ----
    bf16x8 dh[2], dl[2];
    {
        const int g4 = lane >> 4, c16 = lane & 15;
        unsigned hw[3][2], lw[3][2];
        const int off = c16 - 4 * g4;                                     // t - s of register 0
#pragma unroll
        for (int b = 0; b < 3; ++b)
#pragma unroll
            for (int p = 0; p < 2; ++p) {
                const float x0 = d[b][2 * p], x1 = d[b][2 * p + 1];
                hw[b][p] = pack_bf16(x0, x1);
                lw[b][p] = tail_bf16(x0, x1, hw[b][p]);
            }
#pragma unroll
        for (int tb = 0; tb < 2; ++tb) {
            const int b = 2 * tb;
            if (DIAG == 1) {
                const float x = off == 0 ? d[b][0] : off == 1 ? d[b][1] : off == 2 ? d[b][2] : d[b][3];
                if (off >= 0 && off < 4) diag[16 * tb + c16] = x;
            }
            unsigned gh = 0u, gl = 0u;
            if (DIAG == 2) {
                const int t = 16 * tb + c16;
                const float x = (bon[0][t] + bon[1][t]) + (bon[2][t] + bon[3][t]);
                gh = pack_bf16(x, x);
                gl = pack_bf16(x - bf16_lo(gh), x - bf16_lo(gh));
            }
#pragma unroll
            for (int p = 0; p < 2; ++p) {
                const unsigned keep = (2 * p < off ? 0xffffu : 0u) | (2 * p + 1 < off ? 0xffff0000u : 0u);
                hw[b][p] &= keep;
                lw[b][p] &= keep;
                if (DIAG == 2) {
                    const unsigned on = (2 * p == off ? 0xffffu : 0u) | (2 * p + 1 == off ? 0xffff0000u : 0u);
                    hw[b][p] |= gh & on;
                    lw[b][p] |= gl & on;
                }
            }
        }
        dh[0] = words_of(hw[0][0], hw[0][1], 0u, 0u);
        dl[0] = words_of(lw[0][0], lw[0][1], 0u, 0u);
        dh[1] = words_of(hw[1][0], hw[1][1], hw[2][0], hw[2][1]);
        dl[1] = words_of(lw[1][0], lw[1][1], lw[2][0], lw[2][1]);
    }
    // ---- out += Val D, and the state takes the chunk's tokens ----
#pragma unroll
    for (int ot = 0; ot < NO; ++ot) {
        phase();
        const int g4 = lane >> 4, c16 = lane & 15;
        const bf16x8 vh = channel_rows(Vh, 16 * (o0 + ot) + c16, g4);
        bf16x8 vl;
        if (VS) vl = channel_rows(Vl, 16 * (o0 + ot) + c16, g4);
#pragma unroll
        for (int ch = 0; ch < 2; ++ch) {                                  // two row tiles of the state at a time
            bf16x8 kh[2], kl[2];
#pragma unroll
            for (int q = 0; q < 2; ++q) {
                kh[q] = channel_rows(Kh, 16 * (2 * ch + q) + c16, g4);
                if (KS) kl[q] = channel_rows(Kl, 16 * (2 * ch + q) + c16, g4);
            }
            f32x4 &s0 = st[4 * ot + 2 * ch], &s1 = st[4 * ot + 2 * ch + 1], &a = acc[ot][ch];
            a = mfma(vh, dh[ch], a);
            s0 = mfma(kh[0], vh, s0);
            s1 = mfma(kh[1], vh, s1);
            a = mfma(vh, dl[ch], a);
            if (VS) {
                s0 = mfma(kh[0], vl, s0);
                s1 = mfma(kh[1], vl, s1);
                a = mfma(vl, dh[ch], a);
            }
            if (KS) {
                s0 = mfma(kl[0], vh, s0);
                s1 = mfma(kl[1], vh, s1);
            }
            if (VS && LL) a = mfma(vl, dl[ch], a);
            __builtin_amdgcn_sched_barrier(0);
        }
        emit(ot, acc[ot]);
    }
}

// One (b,h) sequence, or the segment `seg` of one, by a workgroup of eight waves (no wave may still be using L).
template <typename IO, typename WT, bool W_IS_EW>
__device__ __forceinline__
void bwd_sweep_sequence(const BwdArgs& A, BwdLds<!__is_same(IO, __hip_bfloat16)>& L, int& sFlag, int bh, int seg)
{
    constexpr bool EXACT = __is_same(IO, __hip_bfloat16);
    constexpr unsigned ES = (unsigned)sizeof(IO), WS = (unsigned)sizeof(WT);
    static_assert(sizeof(BwdLds<!EXACT>) >= 2 * SEQ_STAGE_FLOATS * sizeof(float), "the sequential sweeps' staging must fit");

    const int lane = threadIdx.x & 63;                                    // channel in the element-wise and closing stages
    const int w8 = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);      // token group there (tokens 4 w8 .. 4 w8 + 3 of the chunk)
    const int T = A.T, C = A.C, nseg = A.nseg;
    const int b = bh / A.H, h = bh % A.H;
    const size_t base = (size_t)b * T * C + (size_t)h * HN;
    const int cps = ((T + LC - 1) / LC + nseg - 1) / nseg, c0 = seg * cps;
    const int nchunk = min(cps, (T + LC - 1) / LC - c0);
    float* const gu_out = A.gu_part + ((size_t)b * nseg + seg) * C + h * HN;
    bool bail = false;
    if (threadIdx.x == 0) sFlag = 0;
    if (threadIdx.x < 4 * LC) L.Bon[0][threadIdx.x] = 0.f;               // the upward sweep has no bonus
    __syncthreads();
    if (nseg > 1) {
        const int f = lane < nseg ? A.seg_flags[(size_t)bh * nseg + lane] : 0;
        if (__builtin_amdgcn_ballot_w64(f != 0) != 0ull) {               // the whole sequence is left to its first segment
            if (seg != 0) {
                if (threadIdx.x < HN) gu_out[threadIdx.x] = 0.f;
                return;
            }
            bail = true;
        }
    }

    if (!bail) {
    using RawIO = typename BufRaw<ES>::type;
    using RawW = typename BufRaw<WS>::type;
    using Raw4 = typename BufRaw<16>::type;
    const unsigned n_el = (unsigned)((size_t)(T - 1) * C + HN);          // elements from the block's first to its last
    // A descriptor is put together where it is used, from a pointer the compiler cannot see through: eleven of them kept
    // across the loops spill scalar registers by the dozen.
    auto desc = [&](const void* tensor, unsigned element, unsigned elements) {
        size_t q = reinterpret_cast<size_t>(tensor) + base * element;
        asm volatile("" : "+s"(q));
        return make_rsrc(reinterpret_cast<const void*>(q), elements * element);
    };
    auto cvt = [](RawIO raw) { IO t; __builtin_memcpy(&t, &raw, sizeof(t)); return to_f32(t); };
    auto put_out = [&](float x, __amdgpu_buffer_rsrc_t r, bool narrow, auto type, unsigned el, unsigned s) {
        using OT = decltype(type);
        if (sizeof(OT) == 2 && narrow) {
            const OT q = from_f32<OT>(x);
            typename BufRaw<2>::type raw;
            __builtin_memcpy(&raw, &q, 2);
            BufRaw<2>::st(raw, r, el * 2u, s * 2u);
        } else {
            BufRaw<4>::st(__builtin_bit_cast(unsigned, x), r, el * 4u, s * 4u);
        }
    };
    const float* seg_in = A.seg_ws + ((size_t)bh * nseg + seg) * BWD_SEG_FLOATS;
    const int o0 = w8 < 4 ? 2 * (w8 & 1) : w8 - 4;                       // first output tile of 16 columns in the matrix stage

    // ---- states: waves 0..3: 8 tiles (rows i, 32 columns j); waves 4..7: 4 tiles (rows j, 16 columns i) ----
    f32x4 st[8];
    auto load_state = [&](const float* m) {
        int l = lane;
        asm volatile("" : "+v"(l));                                       // addresses formed here, not kept from the kernel's start
        const __amdgpu_buffer_rsrc_t rs = make_rsrc(m, SEG_STATE * 4);
        if (w8 < 4) {
#pragma unroll
            for (int q = 0; q < 8; ++q) st[q] = __builtin_bit_cast(f32x4, BufRaw<16>::ld(rs, l * 16u, (unsigned)(o0 * 4 + q) * 1024u));
        } else {                                                          // the same state the other way round
            const int g4 = l >> 4, c16 = l & 15;
            const unsigned vo = (unsigned)((c16 >> 2) * 16 + 4 * g4) * 16u + (c16 & 3) * 4u;
#pragma unroll
            for (int q = 0; q < 4; ++q)
#pragma unroll
                for (int e = 0; e < 4; ++e) st[q][e] = __builtin_bit_cast(float, BufRaw<4>::ld(rs, vo, (unsigned)(q * 4 + o0) * 1024u + e * 16u));
        }
    };
#pragma unroll
    for (int q = 0; q < 8; ++q) st[q] = f32x4{0.f, 0.f, 0.f, 0.f};
    if (nseg > 1) load_state(seg_in + (w8 < 2 ? 0 : 1) * SEG_STATE);     // upward sweep: S of the ascending pass, G of the descending one

    const float uu = A.u[h * HN + lane];
    float xrun = 0.f, gu = 0.f;

#pragma unroll 1
    for (int sweep = 0; sweep < 2; ++sweep) {
        const bool dn = sweep == 1;
        if (dn) {
            if (nseg > 1 && w8 < 4) {
                // X at the segment's end: sum_i S[j][i] G[j][i] of both passes, S / G of one direction as they stand in
                // waves 0, 1 / 2, 3, the other direction's as it enters here from behind
                int l = lane;
                asm volatile("" : "+v"(l));
                const __amdgpu_buffer_rsrc_t rs = make_rsrc(seg_in + (w8 < 2 ? 3 : 2) * SEG_STATE, SEG_STATE * 4);
#pragma unroll
                for (int ot = 0; ot < 2; ++ot) {
                    float x = 0.f;
#pragma unroll
                    for (int it = 0; it < 4; ++it) {
                        const f32x4 o = __builtin_bit_cast(f32x4, BufRaw<16>::ld(rs, l * 16u, (unsigned)((o0 + ot) * 4 + it) * 1024u));
#pragma unroll
                        for (int e = 0; e < 4; ++e) x = fmaf(st[4 * ot + it][e], o[e], x);
                    }
                    x += __shfl_xor(x, 16);
                    x += __shfl_xor(x, 32);
                    if (lane < 16) L.X[w8 >> 1][16 * (o0 + ot) + lane] = x;
                }
            }
            __syncthreads();                                              // the upward sweep's results are read back by other waves
            if (nseg > 1) {
                xrun = L.X[0][lane] + L.X[1][lane];
                load_state(seg_in + (w8 < 2 ? 2 : 3) * SEG_STATE);       // downward sweep: S of the descending pass, G of the ascending one
            } else {
#pragma unroll
                for (int q = 0; q < 8; ++q) st[q] = f32x4{0.f, 0.f, 0.f, 0.f};
            }
        }
        // Scan position 4 w8 + m of chunk c is token 32 c + 4 w8 + m upwards, 32 c + 31 - 4 w8 - m downwards.  Rows past T lie
        // outside the descriptors (loads give 0, which switches the token off, stores are dropped).
        int Cs = C, ws = w8, lane_s = lane;                               // opaque copies, renewed in every step (see below)
        auto row = [&](int c, int m) -> unsigned { return (unsigned)(c * LC + (dn ? 31 - 4 * ws - m : 4 * ws + m)) * Cs; };
        auto chunk_of = [&](int ch) { return c0 + (dn ? nchunk - 1 - ch : ch); };
        RawIO rraw[4], kraw[4], vraw[4];
        RawW wraw[4];
        float graw[4];
        auto fetch_w = [&](int c) {
            const __amdgpu_buffer_rsrc_t rsw = desc(A.w, WS, n_el);
#pragma unroll
            for (int m = 0; m < 4; ++m) wraw[m] = BufRaw<WS>::ld(rsw, lane_s * WS, row(c, m) * WS);
        };
        auto fetch = [&](int c) {
            const __amdgpu_buffer_rsrc_t rsr = desc(A.r, ES, n_el), rsk = desc(A.k, ES, n_el), rsv = desc(A.v, ES, n_el), rsg = desc(A.gy, 4, n_el);
#pragma unroll
            for (int m = 0; m < 4; ++m) {
                const unsigned s = row(c, m);
                rraw[m] = BufRaw<ES>::ld(rsr, lane_s * ES, s * ES);
                kraw[m] = BufRaw<ES>::ld(rsk, lane_s * ES, s * ES);
                vraw[m] = BufRaw<ES>::ld(rsv, lane_s * ES, s * ES);
                graw[m] = __builtin_bit_cast(float, BufRaw<4>::ld(rsg, lane_s * 4u, s * 4u));
            }
        };
        // log2 decays of the wave's tokens (ld) and their sums from the group's start (p)
        float ld[4], p[4];
        auto decays = [&](int c) {
#pragma unroll
            for (int m = 0; m < 4; ++m) {
                WT t;
                __builtin_memcpy(&t, &wraw[m], sizeof(t));
                const float fw = to_f32(t);
                ld[m] = W_IS_EW ? fw * LOG2E : -fast_exp2(fmaf(fw, LOG2E, LOG2_LOG2E));
            }
            if ((c + 1) * LC > T) {                                       // wave-uniform: some token of the chunk is past T
#pragma unroll
                for (int m = 0; m < 4; ++m)
                    if (c * LC + (dn ? 31 - 4 * ws - m : 4 * ws + m) >= T) ld[m] = 0.f;
            }
            p[0] = ld[0];
#pragma unroll
            for (int m = 1; m < 4; ++m) p[m] = p[m - 1] + ld[m];
            L.Tot[ws][lane_s] = p[3];
        };
        // sums of a table [group][channel] over the groups before this one and behind it (wave-uniform weights)
        auto group_sums = [&](const float (*tab)[HN], float& before, float& rest) {
            before = rest = 0.f;
#pragma unroll
            for (int g = 0; g < 8; ++g) {
                const float t = tab[g][lane_s];
                int wb = g < ws ? 0x3f800000 : 0, wr = g > ws ? 0x3f800000 : 0;       // 1.0f or 0.0f in a scalar register
                asm volatile("" : "+s"(wb), "+s"(wr));
                before = fmaf(__builtin_bit_cast(float, wb), t, before);
                rest = fmaf(__builtin_bit_cast(float, wr), t, rest);
            }
        };
        float hq[4], ldc[4];
        // gw of a chunk's tokens, once every wave has left its sum of q: ld (X + sum of q over the tokens scanned before - t)
        auto put_gw = [&](int c) {
            float before, rest;
            group_sums(L.Q, before, rest);
            const __amdgpu_buffer_rsrc_t rgw = desc(A.gw, A.w16 ? WS : 4u, n_el);
#pragma unroll
            for (int m = 0; m < 4; ++m) put_out(ldc[m] * (1.0f / LOG2E) * ((xrun + before) + hq[m]), rgw, A.w16, WT{}, lane_s, row(c, m));
            xrun += before + L.Q[ws][lane_s] + rest;
        };
        fetch_w(chunk_of(0));
        fetch(chunk_of(0));
        decays(chunk_of(0));
        lds_barrier();
#pragma unroll 1
        for (int ch = 0; ch < nchunk; ++ch) {
            const int cc = chunk_of(ch);
            // Addresses, row offsets and weights are formed again in every step from opaque copies of the lane and wave
            // numbers and of C: kept across the loop they would take dozens of registers of either kind.
            auto renew = [&]() {
                lane_s = lane;
                Cs = C;
                ws = w8;
                asm volatile("" : "+v"(lane_s), "+s"(Cs), "+s"(ws));
            };
            renew();
            // ================================ element-wise stage ================================
            {
                float before, rest;
                group_sums(L.Tot, before, rest);
                const float tail = p[3] + rest, p31 = before + tail;
                if (nseg == 1 && !dn && ws == 0 && __builtin_amdgcn_ballot_w64(!(p31 >= -SAFE_DECAY * LOG2E)) != 0ull && lane_s == 0) sFlag = 1;
                if (ws == 0) L.C2[lane_s] = fast_exp2(p31);
                auto split = [&](float x0, float x1, unsigned& hi, unsigned& lo) {
                    hi = pack_bf16(x0, x1);
                    lo = tail_bf16(x0, x1, hi);
                };
                auto put = [&](__bf16 (*arr)[BP], unsigned x0, unsigned x1) { *reinterpret_cast<uint2*>(&arr[lane_s][tok_col(ws)]) = make_uint2(x0, x1); };
                float rr[4], kk[4], f1[4], f2[4];
#pragma unroll
                for (int m = 0; m < 4; ++m) {
                    f1[m] = fast_exp2(m ? p[m - 1] - tail : -tail);       // e^(Pex - P31), e^(P31 - P)
                    f2[m] = fast_exp2(tail - p[m]);
                    L.F1[4 * ws + m][lane_s] = f1[m];
                    rr[m] = cvt(rraw[m]);
                    kk[m] = cvt(kraw[m]);
                }
                unsigned h[2], l[2];
                auto quad = [&](const float (&x)[4], __bf16 (*hi)[BP], __bf16 (*lo)[BP]) {
                    split(x[0], x[1], h[0], l[0]);
                    split(x[2], x[3], h[1], l[1]);
                    put(hi, h[0], h[1]);
                    put(lo, l[0], l[1]);
                };
                const float k1[4] = {kk[0] * f1[0], kk[1] * f1[1], kk[2] * f1[2], kk[3] * f1[3]};
                quad(k1, L.KF1h, L.KF1l);
                const float k2[4] = {kk[0] * f2[0], kk[1] * f2[1], kk[2] * f2[2], kk[3] * f2[3]};
                quad(k2, L.KF2h, L.KF2l);
                const float r2[4] = {rr[0] * f2[0], rr[1] * f2[1], rr[2] * f2[2], rr[3] * f2[3]};
                quad(r2, L.RF2h, L.RF2l);
                quad(graw, L.GYh, L.GYl);
                if constexpr (EXACT) {                                    // the bf16 bits as loaded
                    put(L.Vh, (unsigned)vraw[0] | ((unsigned)vraw[1] << 16), (unsigned)vraw[2] | ((unsigned)vraw[3] << 16));
                } else {
                    const float v4[4] = {cvt(vraw[0]), cvt(vraw[1]), cvt(vraw[2]), cvt(vraw[3])};
                    quad(v4, L.Vh, L.Vl);
                }
                if (dn) {                                                 // bonus_t = sum_j u[j] r_t[j] k_t[j], by rows of 16 lanes
                    const bool b0 = lane_s & 1, b1 = lane_s & 2;
                    float pu[4], a2[2];
#pragma unroll
                    for (int m = 0; m < 4; ++m) pu[m] = rr[m] * uu * kk[m];
#pragma unroll
                    for (int i = 0; i < 2; ++i) a2[i] = (b0 ? pu[2 + i] : pu[i]) + dpp_get<0xB1>(b0 ? pu[i] : pu[2 + i]);
                    float a1 = (b1 ? a2[1] : a2[0]) + dpp_get<0x4E>(b1 ? a2[0] : a2[1]);
                    a1 += dpp_get<0x124>(a1);                             // row_ror:4, row_ror:8: the other quads of the 16 lanes
                    a1 += dpp_get<0x128>(a1);
                    if ((lane_s & 15) < 4) L.Bon[lane_s >> 4][4 * ws + (b0 ? 2 : 0) + (b1 ? 1 : 0)] = a1;
                }
            }
            lds_barrier();
            if (sFlag) { bail = true; break; }
            renew();
            fetch_w(ch + 1 < nchunk ? chunk_of(ch + 1) : cc);
            if (dn && ch > 0) put_gw(chunk_of(ch - 1));
            renew();
            // =================================== matrix stage ===================================
            {
                const int g4 = lane_s >> 4, c16 = lane_s & 15;
                auto to_lds = [&](float (*res)[RP]) {
                    return [=](int ot, const f32x4 (&acc)[2]) {
#pragma unroll
                        for (int tb = 0; tb < 2; ++tb) *reinterpret_cast<f32x4*>(&res[16 * tb + c16][16 * (o0 + ot) + 4 * g4]) = acc[tb];
                    };
                };
                if (ws < 2) {
                    matrix_stage<true, !EXACT, true, true, 2, false, 1>(L.GYh, L.GYl, L.Vh, L.Vl, L.KF2h, L.KF2l, L.C2, st, o0, lane_s, L.Diag, nullptr,
                                                                        to_lds(L.Res[0]));
                } else if (ws < 4) {
                    matrix_stage<!EXACT, true, true, true, 2, false, 0>(L.Vh, L.Vl, L.GYh, L.GYl, L.RF2h, L.RF2l, L.C2, st, o0, lane_s, nullptr, nullptr,
                                                                        to_lds(L.Res[1]));
                } else {
                    // gv leaves from here: a lane_s holds four neighbouring channels of a token
                    const unsigned v_el = (unsigned)((dn ? 15 - c16 : c16) * Cs + 16 * o0 + 4 * g4);
                    const __amdgpu_buffer_rsrc_t rpv = desc(A.pv, 4, n_el);
                    matrix_stage<true, true, true, false, 1, true, 2>(L.KF1h, L.KF1l, L.RF2h, L.RF2l, L.GYh, L.GYl, L.C2, st, o0, lane_s, nullptr, L.Bon,
                        [&](int, const f32x4 (&acc)[2]) {
#pragma unroll
                            for (int tb = 0; tb < 2; ++tb) {
                                const unsigned s_el = (unsigned)(cc * LC + (dn ? 16 - 16 * tb : 16 * tb)) * Cs;
                                if (!dn) {
                                    BufRaw<16>::st(__builtin_bit_cast(Raw4, acc[tb]), rpv, v_el * 4u, s_el * 4u);
                                    continue;
                                }
                                const f32x4 g = __builtin_bit_cast(f32x4, BufRaw<16>::ld(rpv, v_el * 4u, s_el * 4u)) + acc[tb];
                                if (ES == 2 && A.out16) {
                                    IO q[4];
#pragma unroll
                                    for (int e = 0; e < 4; ++e) q[e] = from_f32<IO>(g[e]);
                                    typename BufRaw<8>::type raw;
                                    __builtin_memcpy(&raw, q, 8);
                                    BufRaw<8>::st(raw, desc(A.gv, ES, n_el), v_el * 2u, s_el * 2u);
                                } else {
                                    BufRaw<16>::st(__builtin_bit_cast(Raw4, g), desc(A.gv, 4, n_el), v_el * 4u, s_el * 4u);
                                }
                            }
                        });
                }
            }
            renew();
#pragma unroll
            for (int m = 0; m < 4; ++m) ldc[m] = ld[m];
            // for the closing stage: the upward sweep's gr and gk of the wave's tokens, r and k once more (upwards the
            // descriptors are empty: no access); then the next chunk's rows and decays
            float upr[4], upk[4];
            RawIO rc[4], kc[4];
            {
                const unsigned n = dn ? n_el : 0u;
                const __amdgpu_buffer_rsrc_t rsr = desc(A.r, ES, n), rsk = desc(A.k, ES, n), rpr = desc(A.pr, 4, n), rpk = desc(A.pk, 4, n);
#pragma unroll
                for (int m = 0; m < 4; ++m) {
                    const unsigned s = row(cc, m);
                    upr[m] = __builtin_bit_cast(float, BufRaw<4>::ld(rpr, lane_s * 4u, s * 4u));
                    upk[m] = __builtin_bit_cast(float, BufRaw<4>::ld(rpk, lane_s * 4u, s * 4u));
                    rc[m] = BufRaw<ES>::ld(rsr, lane_s * ES, s * ES);
                    kc[m] = BufRaw<ES>::ld(rsk, lane_s * ES, s * ES);
                }
            }
            decays(ch + 1 < nchunk ? chunk_of(ch + 1) : cc);
            fetch(ch + 1 < nchunk ? chunk_of(ch + 1) : cc);
            lds_barrier();
            // =================================== closing stage ==================================
            float f1[4];
#pragma unroll
            for (int m = 0; m < 4; ++m) f1[m] = L.F1[4 * ws + m][lane_s];
            if (!dn) {
                const __amdgpu_buffer_rsrc_t rpr = desc(A.pr, 4, n_el), rpk = desc(A.pk, 4, n_el);
#pragma unroll
                for (int m = 0; m < 4; ++m) {
                    const unsigned s = row(cc, m) * 4u;
                    BufRaw<4>::st(__builtin_bit_cast(unsigned, L.Res[0][4 * ws + m][lane_s] * f1[m]), rpr, lane_s * 4u, s);
                    BufRaw<4>::st(__builtin_bit_cast(unsigned, L.Res[1][4 * ws + m][lane_s] * f1[m]), rpk, lane_s * 4u, s);
                }
            } else {
                const f32x4 dg = *reinterpret_cast<const f32x4*>(&L.Diag[4 * ws]);
                const __amdgpu_buffer_rsrc_t rgr = desc(A.gr, A.out16 ? ES : 4u, n_el), rgk = desc(A.gk, A.out16 ? ES : 4u, n_el);
                float run = 0.f;
#pragma unroll
                for (int m = 0; m < 4; ++m) {
                    const float r1 = cvt(rc[m]), k1 = cvt(kc[m]), ud = uu * dg[m];
                    const float grd = L.Res[0][4 * ws + m][lane_s] * f1[m], gkd = L.Res[1][4 * ws + m][lane_s] * f1[m];
                    hq[m] = run - (k1 * gkd + r1 * grd);
                    run += r1 * (upr[m] - grd) + k1 * (upk[m] - gkd);
                    gu = fmaf(r1 * k1, dg[m], gu);
                    const unsigned s = row(cc, m);
                    put_out(fmaf(ud, k1, upr[m] + grd), rgr, A.out16, IO{}, lane_s, s);
                    put_out(fmaf(ud, r1, upk[m] + gkd), rgk, A.out16, IO{}, lane_s, s);
                }
                L.Q[ws][lane_s] = run;
            }
        }
        if (dn && !bail) {
            lds_barrier();
            put_gw(chunk_of(nchunk - 1));
        }
        if (bail) break;
    }
    if (!bail) {
        __syncthreads();
        L.Q[w8][lane] = gu;
        __syncthreads();
        if (threadIdx.x < HN) {
            float s = 0.f;
#pragma unroll
            for (int g = 0; g < 8; ++g) s += L.Q[g][threadIdx.x];
            gu_out[threadIdx.x] = s;
        }
        return;
    }
    }
    // Some chunk decays faster than the factors can represent: the whole sequence with the sequential sweeps, which add into fp32
    // buffers; 16-bit results are rounded from those afterwards.  The sweeps are four waves wide and a chain over the tokens, so
    // two run side by side: waves 0..3 gr of both passes and then half of gv, waves 4..7 the other half of gv and then gk and gw,
    // which need gr's `a` of the same pass (768 sequences of 196 tokens, bf16: 1140 us; one after the other 2010).
    __syncthreads();
    float* const stage = reinterpret_cast<float*>(&L) + (w8 >> 2) * SEQ_STAGE_FLOATS;
    const IO *r = static_cast<const IO*>(A.r), *k = static_cast<const IO*>(A.k), *v = static_cast<const IO*>(A.v);
    const WT* w = static_cast<const WT*>(A.w);
    float* const gu_row = A.gu_part + (size_t)b * nseg * C + h * HN;
    if (w8 < 4) seq_sweep_s<IO, WT, 1, W_IS_EW>(bh, r, k, v, w, A.u, A.gy, A.pr, A.a, gu_row, stage, T, C, A.H);
    else seq_sweep_v<IO, WT, 1, W_IS_EW>(bh, r, k, w, A.u, A.gy, A.pv, stage, T, C, A.H);
    __syncthreads();
    if (w8 < 4) seq_sweep_s<IO, WT, 0, W_IS_EW>(bh, r, k, v, w, A.u, A.gy, A.pr, A.a + A.a_size, gu_row, stage, T, C, A.H);
    else seq_sweep_g<IO, WT, 1, W_IS_EW>(bh, r, k, v, w, A.u, A.gy, A.a, A.pk, A.pw, stage, T, C, A.H);
    __syncthreads();
    if (w8 < 4) seq_sweep_v<IO, WT, 0, W_IS_EW>(bh, r, k, w, A.u, A.gy, A.pv, stage, T, C, A.H);
    else seq_sweep_g<IO, WT, 0, W_IS_EW>(bh, r, k, v, w, A.u, A.gy, A.a + A.a_size, A.pk, A.pw, stage, T, C, A.H);
    if ((ES == 2 && A.out16) || (WS == 2 && A.w16)) {
        __syncthreads();
        for (size_t q = threadIdx.x; q < (size_t)T * HN; q += 512) {
            const size_t o = base + (q >> 6) * C + (q & 63);
            if (ES == 2 && A.out16) {
                static_cast<IO*>(A.gr)[o] = from_f32<IO>(A.pr[o]);
                static_cast<IO*>(A.gk)[o] = from_f32<IO>(A.pk[o]);
                static_cast<IO*>(A.gv)[o] = from_f32<IO>(A.pv[o]);
            }
            if (WS == 2 && A.w16) static_cast<WT*>(A.gw)[o] = from_f32<WT>(A.pw[o]);
        }
    }
}

template <typename IO, typename WT, bool W_IS_EW>
__global__ __launch_bounds__(512, 4)                 // four waves per SIMD: at most 128 registers
void wkv6_bwd_sweep_kernel(BwdArgs A)
{
    __shared__ BwdLds<!__is_same(IO, __hip_bfloat16)> L;
    __shared__ int sFlag;
    int bh = blockIdx.x, seg = 0;
    if (A.nseg > 1) {
        seg_of_block(blockIdx.x, A.nseg, bh, seg);
        if (bh >= A.sequences) return;
    }
    bwd_sweep_sequence<IO, WT, W_IS_EW>(A, L, sFlag, bh, seg);
}

}  // namespace wkv6_detail
}  // namespace vrwkv
