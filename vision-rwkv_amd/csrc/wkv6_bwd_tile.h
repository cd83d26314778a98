// wkv6 backward, sequences of up to 256 tokens (or segments of up to 128) as one or two matrix products (gfx950, bf16 MFMA, fp32 accumulate).
//
// Both passes of the scan at once, as in wkv6_fwd_tile.h, with the same factors in a part of up to 128 tokens:
//   e1_t = 2^(Pex_t - c), e2_t = 2^(c - P_t), c = P_end / 2;   rf = r e1, kf = k e2 (i < t);   rb = r e2, kb = k e1 (i > t)
//   A[t][i] = rf_t . kf_i  (i < t),  rb_t . kb_i  (i > t),  sum_j r u k  (i = t);      D[t][i] = gy_t . v_i
//   gv_i = sum_t A[t][i] gy_t
//   gr_t = e1_t sum_{i<t} D[t][i] kf_i  +  e2_t sum_{i>t} D[t][i] kb_i  +  u k_t D[t][t]        (gr_up, gr_dn: from tokens before, behind)
//   gk_i = e2_i sum_{t>i} D[t][i] rf_t  +  e1_i sum_{t<i} D[t][i] rb_t  +  u r_i D[i][i]        (gk_dn, gk_up)
//   gw_n = ld_n (X + sum_{m>n} q_m - t_n),  q = r (gr_up - gr_dn) + k (gk_up - gk_dn),  t = k gk_dn + r gr_dn
// (X: the same sum over the tokens behind the part; formulas of classification/mmcls_custom/models/backbones/cuda_v6/wkv6_cuda.cu:99-346).
// Across parts, S = sum_i k_i v_i^T and G = sum_t r_t gy_t^T, decayed to the border, stand for the other part's tokens:
//   from the front   gr += e1 (2^c S gy),  gk += e1 (2^c G v),  gv += (2^c G)^T kb;      from behind   e2, e2 and kf in their place.
// Two parts are three steps: S and G of the first part; the second part with those; the first part with what the second one leaves in front of it.
//
// Against the sweeps of wkv6_bwd_sweep.h no partial gradient goes through memory (0.61 GB there at 64 x 196 x 768, 0.19 GB are the inputs and results), the
// 64 x 64 states are scaled and split once per part and not once per 32 tokens, and a token's factors are formed once and not once per sweep.
//
// A workgroup of eight waves holds a part, one on a compute unit (156 KB of LDS, 256 registers); a wave owns 16 tokens as i (gv, gk: rf, rb and gy of
// the others from LDS) and then as t (gr: kf, kb and v of the others from LDS).  Operands lie in rows of a token's 64 channels; the tiles of gr and gk take
// the channels in the order in which a lane holds its token's rows (token c16, channels 32 kb + 8 g4 .. + 7), so that the results meet r, k and the factors
// there and gw is summed along the rows of 16 lanes.  Computed operands are split into bf16 head + tail as in the sweeps, tail x tail included for gr and gk.
//
// Bound by latency and vector work: two waves a SIMD issue 6 200 vector instructions, 730 products and 970 LDS accesses each at 64 x 196 x 768, matrix cores
// busy 19 %, LDS 25 %, vector ALUs 40 %; of a full part's 42 000 cycles 6 500 wait for its rows, 4 500 form operands, 11 000 + 7 000 are products and 8 000 the
// results.  us there, sweeps -> here: bf16 195 -> 152, fp32 207 -> 186; one sequence 79 -> 49.  Measured and left out: rows brought into the L2s ahead
// (166 -> 172), pieces of four channels (the loads' halves have to be moved: 166 -> 188), places in LDS with twice the bank conflicts (166 -> 167).
//
// Range: |P_end| <= 200 in a part, less for rows of unusual size (PART_FREE in wkv6_segment.h), and 60 nats over 32 tokens as in the sweeps (gw is a
// difference of sums whose neighbouring tokens do not decay: the more the others do, the less of it is left).  Sequences beyond go through the sweeps' code,
// which leaves the latter to the sequential sweeps.
#pragma once
#include "wkv6_bwd_sweep.h"

namespace vrwkv {
namespace wkv6_detail {

constexpr int BWD_TILE_TOKENS = 2 * PART;            // most tokens of an uncut sequence; a segment has PART

// 32 rows (from row0) of an operand array (row_chunk) x 16 columns, 16 ct + c16, as an operand; slot (g4, e) is row 4 g4 + e (e < 4), 16 + 4 g4 + e - 4 (e >= 4)
__device__ __forceinline__ bf16x8 tile_across(const unsigned char* arr, unsigned row0, int ct, int lane) {
    const int g4 = lane >> 4, c16 = lane & 15;
    const unsigned char* p = arr + row_chunk(4 * g4 + (c16 >> 2), 2 * ct + ((c16 >> 1) & 1)) + 8 * (c16 & 1) + 128u * row0;
    return cat8(lds_read_tr4(reinterpret_cast<const __bf16*>(p)), lds_read_tr4(reinterpret_cast<const __bf16*>(p + 2048)));
}
// ... the columns in the order of a lane's rows: 32 kb + 8 (c16 >> 2) + 4 hf + (c16 & 3)
__device__ __forceinline__ bf16x8 tile_across_owned(const unsigned char* arr, unsigned row0, int kb, int hf, int lane) {
    const int g4 = lane >> 4, c16 = lane & 15;
    const unsigned char* p = arr + row_chunk(4 * g4 + (c16 >> 2), 4 * kb + (c16 & 3)) + 8 * hf + 128u * row0;
    return cat8(lds_read_tr4(reinterpret_cast<const __bf16*>(p)), lds_read_tr4(reinterpret_cast<const __bf16*>(p + 2048)));
}

// SEG: segments of cut sequences (a kernel of its own: either path's registers would hold the other back, 155 -> 176 us uncut).  LOOSE: 16-bit rows that do
// not lie on 4 bytes, fetched element by element.
template <typename IO, typename WT, bool W_IS_EW, bool SEG, bool LOOSE = false>
__global__ __launch_bounds__(64 * PART_WAVES, 2)
void wkv6_bwd_tile_kernel(BwdArgs A)
{
    constexpr bool VSPLIT = !__is_same(IO, __hip_bfloat16);
    constexpr unsigned ES = (unsigned)sizeof(IO), WS = (unsigned)sizeof(WT), ARR = PART * 128u;
    // while a wave's tokens are i / t / while a part's states are formed
    constexpr unsigned RFH = 0, RFL = ARR, RBH = 2 * ARR, RBL = 3 * ARR, GYH = 4 * ARR, GYL = 5 * ARR;
    constexpr unsigned KFH = 0, KFL = ARR, KBH = 2 * ARR, KBL = 3 * ARR, VH = 4 * ARR, VL = 5 * ARR;
    constexpr unsigned LVH = 6 * ARR, LVL = 7 * ARR;                      // (KFH, KFL, RBH, RBL, GYH, GYL beside them)
    // scaled states, row j: 64 value channels, head and tail; apart the G that is formed or waits while the other is read
    constexpr unsigned ZS = 6 * ARR, ZG = 7 * ARR, ZG_BEHIND = 8 * ARR, ZG_FRONT = ZG_BEHIND, ZTAIL = ARR / 2, TAB = 9 * ARR;
    struct Tables { float Tot[PART_WAVES][HN], Before[PART_WAVES][2][HN], Q[PART_WAVES][HN], X[2][HN], Max[PART_WAVES][4]; };
    __shared__ __attribute__((aligned(16))) unsigned char lds[TAB + sizeof(Tables)];
    __shared__ int sFlag;
    using Sweep = BwdLds<VSPLIT>;
    static_assert(sizeof(lds) >= sizeof(Sweep), "the sweeps' operands must fit");
    Tables& L = *reinterpret_cast<Tables*>(lds + TAB);

    // (Addresses are formed anew in every stage, from an opaque copy of the lane number: kept from the kernel's start they would take more registers than
    // there are.)
    int lane = threadIdx.x & 63, g4 = lane >> 4, c16 = lane & 15;
    auto renew = [&]() {
        __builtin_amdgcn_sched_barrier(0);
        lane = threadIdx.x & 63;
        asm volatile("" : "+v"(lane));
        g4 = lane >> 4;
        c16 = lane & 15;
    };
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int T = A.T, C = A.C, nseg = SEG ? A.nseg : 1;
    int bh = blockIdx.x, seg = 0;
    bool bail = false;
    if constexpr (SEG) {
        seg_of_block(blockIdx.x, nseg, bh, seg);
        if (bh >= A.sequences) return;
        const int f = lane < nseg ? A.seg_flags[(size_t)bh * nseg + lane] : 0;
        bail = __builtin_amdgcn_ballot_w64(f != 0) != 0ull;               // the whole sequence is left to its first segment
    }
    const int b = bh / A.H, h = bh % A.H;
    const size_t base = (size_t)b * T * C + (size_t)h * HN;
    const unsigned n_el = (unsigned)((size_t)(T - 1) * C + HN);          // elements from the block's first to its last
    const int nchunk = (T + LC - 1) / LC, cps = (nchunk + nseg - 1) / nseg;
    const int first = seg * cps * LC, n = min(cps * LC, T - first);
    const bool two = !SEG && n > PART;
    const int n1 = two ? (n - PART + LC - 1) / LC * LC : n;              // tokens of the first part

    constexpr int PI = (int)ES / 2, PW = (int)WS / 2;
    auto desc = [&](const void* p, unsigned es) { return make_rsrc(static_cast<const char*>(p) + base * es, n_el * es); };
    // eight channels 32 kb + 8 g4 .. + 7 of the wave's token c16, packed as they lie; rows past T lie outside the descriptors and read 0, which switches
    // such a token off (its decay is set to 1 below)
    auto fetch = [&](const void* p, int t0, auto& raw, unsigned es) {
        const __amdgpu_buffer_rsrc_t rs = desc(p, es);
        constexpr int pieces = sizeof(raw[0]) / 16;
        const unsigned vo = ((unsigned)c16 * C + 8 * g4) * es, so = (unsigned)(t0 + 16 * wave) * C * es;
#pragma unroll
        for (int kb = 0; kb < 2; ++kb) {
            if constexpr (LOOSE && pieces == 1) {
                unsigned e8[8];
#pragma unroll
                for (int e = 0; e < 8; ++e) e8[e] = (unsigned short)BufRaw<2>::ld(rs, vo + 64u * kb + 2u * e, so);
#pragma unroll
                for (int i = 0; i < 4; ++i) raw[kb][0][i] = e8[2 * i] | e8[2 * i + 1] << 16;
            } else {
#pragma unroll
                for (int i = 0; i < pieces; ++i) raw[kb][i] = BufRaw<16>::ld(rs, vo + 32u * kb * es + 16u * i, so);
            }
        }
    };
    // `count` neighbouring results of the wave's token c16 from channel ch on
    auto put_out = [&](void* p, bool narrow, auto type, const float* x, auto count, unsigned ch, int t0) {
        using OT = decltype(type);
        constexpr int N_OUT = decltype(count)::value;
        const unsigned el = (unsigned)c16 * C + ch, so = (unsigned)(t0 + 16 * wave) * C;
        if (sizeof(OT) == 2 && narrow) {
            OT q[N_OUT];
#pragma unroll
            for (int e = 0; e < N_OUT; ++e) q[e] = from_f32<OT>(x[e]);
            typename BufRaw<2 * N_OUT>::type raw;
            __builtin_memcpy(&raw, q, 2 * N_OUT);
            BufRaw<2 * N_OUT>::st(raw, desc(p, 2), el * 2u, so * 2u);
        } else {
            const __amdgpu_buffer_rsrc_t rs = desc(p, 4);
#pragma unroll
            for (int i = 0; i < N_OUT / 4; ++i)
                BufRaw<16>::st(__builtin_bit_cast(typename BufRaw<16>::type, f32x4{x[4 * i], x[4 * i + 1], x[4 * i + 2], x[4 * i + 3]}), rs, el * 4u + 16u * i, so * 4u);
        }
    };

    // A wave's share of the states: column j = 16 jt + c16, rows (value channels) 16 (ct0 + q) + 4 g4 + r
    const int jt = wave & 3, ct0 = 2 * (wave >> 2);
    // a state times 2^c as an operand into LDS
    auto put_state = [&](float c, const f32x4 (&X)[2], unsigned to) {
        const float f = fast_exp2(0.5f * __shfl(c, 16 * jt + c16));       // (c down to -200: in two halves)
#pragma unroll
        for (int q = 0; q < 2; ++q) {
            const unsigned at = to + row_chunk(16 * jt + c16, 2 * (ct0 + q) + (g4 >> 1)) + 8 * (g4 & 1);
            const f32x4 x = X[q] * f * f;
            const unsigned h0 = pack_bf16(x[0], x[1]), h1 = pack_bf16(x[2], x[3]);
            *reinterpret_cast<uint2*>(lds + at) = make_uint2(h0, h1);
            *reinterpret_cast<uint2*>(lds + ZTAIL + at) = make_uint2(tail_bf16(x[0], x[1], h0), tail_bf16(x[2], x[3], h1));
        }
    };
    // sum over the part's tokens of (kh + kl)[j] (vh + vl)[c]
    auto form_state = [&](unsigned kh, unsigned kl, unsigned vh, unsigned vl, auto split, int nb, f32x4 (&X)[2]) {
        X[0] = X[1] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll 1
        for (int q = 0; q < nb; ++q) {
            const bf16x8 bh8 = tile_across(lds + kh, 32 * q, jt, lane), bl8 = tile_across(lds + kl, 32 * q, jt, lane);
#pragma unroll
            for (int i = 0; i < 2; ++i) {
                const bf16x8 ah8 = tile_across(lds + vh, 32 * q, ct0 + i, lane);
                X[i] = mfma(ah8, bh8, X[i]);
                X[i] = mfma(ah8, bl8, X[i]);
                if constexpr (decltype(split)::value) X[i] = mfma(tile_across(lds + vl, 32 * q, ct0 + i, lane), bh8, X[i]);
            }
        }
    };
    constexpr std::integral_constant<bool, VSPLIT> v_split{};
    constexpr std::true_type is_split{};
    // The states that enter the segment from the front (up) or from behind: those that the segments there leave by themselves, each over the decay of the
    // segments in between.  (A launch that folds them first costs 11 us at 48 sequences of five segments.)
    auto local_state = [&](int s, int m, f32x4 (&X)[2]) {
        const float* const p = A.seg_ws + ((size_t)bh * nseg + s) * BWD_SEG_FLOATS + m * SEG_STATE;
#pragma unroll
        for (int q = 0; q < 2; ++q) X[q] = *reinterpret_cast<const f32x4*>(p + seg_frag(jt, ct0 + q, lane));
    };
    auto segment_decay = [&](int s) { return A.seg_ws[((size_t)bh * nseg + s) * BWD_SEG_FLOATS + 4 * SEG_STATE + 16 * jt + c16]; };
    auto entering = [&](bool up, f32x4 (&S)[2], f32x4 (&G)[2]) {
        S[0] = S[1] = G[0] = G[1] = f32x4{0.f, 0.f, 0.f, 0.f};
        const int count = up ? seg : nseg - 1 - seg, m = up ? 0 : 2;
        constexpr int U = 4;
#pragma unroll 1
        for (int q = 0; q < count; q += U) {
            f32x4 ls[U][2], lg[U][2];
            float d[U];
#pragma unroll
            for (int i = 0; i < U; ++i)
                if (q + i < count) {
                    const int s = up ? q + i : nseg - 1 - q - i;
                    local_state(s, m, ls[i]);
                    local_state(s, m + 1, lg[i]);
                    d[i] = segment_decay(s);
                }
#pragma unroll
            for (int i = 0; i < U; ++i)
                if (q + i < count) {
#pragma unroll
                    for (int e = 0; e < 2; ++e) {
                        S[e] = S[e] * d[i] + ls[i][e];
                        G[e] = G[e] * d[i] + lg[i][e];
                    }
                }
        }
    };

    const float uj = A.u[h * HN + lane];
    float xrun = 0.f, c_both = 0.f, gu = 0.f;        // of channel `lane`: the sum of q behind the part; c of both parts; gu of channel gu_at
    int gu_at = 0;
    f32x4 XS[2], XG[2];
#pragma unroll 1
    for (int step = two ? 0 : 2; step < 3 && !bail; ++step) {
        const int part = step == 1 ? 1 : 0, t0 = first + (part ? n1 : 0), np = part ? n - n1 : n1, nb = (np + LC - 1) / LC;
        const bool mine = wave < 2 * nb;             // the wave has tokens, or rows of zeros that another one reads
        renew();
        u32x4 wraw[2][PW], rraw[2][PI], kraw[2][PI], vraw[2][PI], graw[2][2];
        fetch(A.w, t0, wraw, WS);
        fetch(A.k, t0, kraw, ES);
        fetch(A.r, t0, rraw, ES);
        fetch(A.gy, t0, graw, 4u);
        fetch(A.v, t0, vraw, ES);
        f32x4 XD[2], YD[2], XU[2], YU[2];            // S and G that enter a segment from behind and from the front
        if constexpr (SEG) {
            entering(false, XD, YD);
            entering(true, XU, YU);
            // X at the segment's end: sum over the value channels of S G of both passes
            f32x4 ls[2], lg[2];
            local_state(seg, 0, ls);
            local_state(seg, 1, lg);
            const float d = segment_decay(seg);
            float x = 0.f;
#pragma unroll
            for (int q = 0; q < 2; ++q)
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    x = fmaf(fmaf(XU[q][e], d, ls[q][e]), YD[q][e], x);
                    x = fmaf(fmaf(YU[q][e], d, lg[q][e]), XD[q][e], x);
                }
            x += __shfl_xor(x, 16);
            x += __shfl_xor(x, 32);
            if (lane < 16) L.X[wave >> 2][16 * jt + lane] = x;
        }
        const bool past = 16 * wave + c16 >= np;
        float x[2][8];                               // log2 decays summed over the wave's tokens, channel 32 kb + 8 g4 + e
        float c_part;
        {
#pragma unroll
            for (int kb = 0; kb < 2; ++kb) {
                summed_decays<WT, W_IS_EW>(wraw[kb], past, x[kb]);
                if (c16 == 15) {
#pragma unroll
                    for (int hf = 0; hf < 2; ++hf)
                        *reinterpret_cast<f32x4*>(&L.Tot[wave][32 * kb + 8 * g4 + 4 * hf]) = f32x4{x[kb][4 * hf], x[kb][4 * hf + 1], x[kb][4 * hf + 2], x[kb][4 * hf + 3]};
                }
            }
            lds_barrier();
            float s = 0.f, total = 0.f, t[PART_WAVES];
#pragma unroll
            for (int g = 0; g < PART_WAVES; ++g) {
                t[g] = L.Tot[g][lane];
                s += g < wave ? t[g] : 0.f;
                total += t[g];
            }
            c_part = 0.5f * total;
            bool in_range = total >= -PART_RANGE;
#pragma unroll
            for (int g = 0; g < PART_WAVES; g += 2) in_range &= t[g] + t[g + 1] >= -SAFE_DECAY * LOG2E;
            if (__builtin_amdgcn_ballot_w64(!in_range) != 0ull) { bail = true; break; }                       // the same in every wave
            if (__builtin_amdgcn_ballot_w64(!(total >= -PART_FREE)) != 0ull) {                                // ... and this
                const float mr = largest_of_wave(mine ? largest16<IO>(rraw[0], rraw[1]) : 0.f), mk = largest_of_wave(mine ? largest16<IO>(kraw[0], kraw[1]) : 0.f),
                            mv = largest_of_wave(mine ? largest16<IO>(vraw[0], vraw[1]) : 0.f), mg = largest_of_wave(mine ? largest16<float>(graw[0], graw[1]) : 0.f);
                if (lane == 0) *reinterpret_cast<f32x4*>(L.Max[wave]) = f32x4{mr, mk, mv, mg};
                lds_barrier();
                f32x4 m = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
                for (int g = 0; g < PART_WAVES; ++g) {
                    const f32x4 x = *reinterpret_cast<const f32x4*>(L.Max[g]);
#pragma unroll
                    for (int e = 0; e < 4; ++e) m[e] = fmaxf(m[e], x[e]);
                }
                const float lr = log2_of_largest(m[0]), lk = log2_of_largest(m[1]), lv = log2_of_largest(m[2]), lg = log2_of_largest(m[3]);
                const float lo = fminf(lr, lk), hi = fmaxf(lr, lk);
                const float smallest = fminf(fminf(lo, lo + lg + lv), fminf(lk + lv, lr + lg)), largest = fmaxf(fmaxf(hi, hi + lg + lv), fmaxf(lk + lv, lr + lg));
                if (__builtin_amdgcn_ballot_w64(!(total >= -part_decay(smallest, largest))) != 0ull) { bail = true; break; }
            }
            L.Before[wave][0][lane] = s - c_part;
            L.Before[wave][1][lane] = uj;
        }
        // (formed twice, before the products and after them: kept they would take 32 registers)
        auto factors = [&](int kb, float (&e1)[8], float (&e2)[8]) {
#pragma unroll
            for (int hf = 0; hf < 2; ++hf) {
                const f32x4 before = *reinterpret_cast<const f32x4*>(&L.Before[wave][0][32 * kb + 8 * g4 + 4 * hf]);
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const float d = x[kb][4 * hf + e];
                    e1[4 * hf + e] = fast_exp2(before[e] + dpp_get<0x111>(d));
                    e2[4 * hf + e] = fast_exp2(-(before[e] + d));
                }
            }
        };
        auto times = [&](const u32x4* raw, const float* f, bf16x8& hi, bf16x8& lo) {
            float o8[8];
            widen8<IO>(raw, o8);
#pragma unroll
            for (int e = 0; e < 8; ++e) o8[e] *= f[e];
            split8<true>(o8, hi, lo);
        };
        auto store = [&](unsigned hi, unsigned lo, int kb, const bf16x8& xh, const bf16x8& xl) {
            const unsigned at = row_chunk(16 * wave + c16, 4 * kb + g4);
            *reinterpret_cast<bf16x8*>(lds + hi + at) = xh;
            *reinterpret_cast<bf16x8*>(lds + lo + at) = xl;
        };
        bf16x8 KF[2][2], KB[2][2], GY[2][2], V[2][2];          // [kb][head, tail], slot (g4, e): channel 32 kb + 8 g4 + e
        float bonus = 0.f, dd = 0.f;
#pragma unroll
        for (int kb = 0; kb < 2; ++kb) {
            bf16x8 hi, lo;
            float g8[8], e1[8], e2[8];
            factors(kb, e1, e2);
            widen8<float>(graw[kb], g8);
            split8<true>(g8, GY[kb][0], GY[kb][1]);
            store(GYH, GYL, kb, GY[kb][0], GY[kb][1]);
            times(rraw[kb], e2, hi, lo);
            store(RBH, RBL, kb, hi, lo);
            times(kraw[kb], e2, KF[kb][0], KF[kb][1]);
            float v8[8];
            widen8<IO>(vraw[kb], v8);
            if constexpr (VSPLIT) split8<true>(v8, V[kb][0], V[kb][1]);
            else V[kb][0] = __builtin_bit_cast(bf16x8, vraw[kb][0]);
            if (step == 0) {
                const unsigned at = row_chunk(16 * wave + c16, 4 * kb + g4);
                store(KFH, KFL, kb, KF[kb][0], KF[kb][1]);
                *reinterpret_cast<bf16x8*>(lds + LVH + at) = V[kb][0];
                if constexpr (VSPLIT) *reinterpret_cast<bf16x8*>(lds + LVL + at) = V[kb][1];
                continue;
            }
            times(rraw[kb], e1, hi, lo);
            store(RFH, RFL, kb, hi, lo);
            times(kraw[kb], e1, KB[kb][0], KB[kb][1]);
            float r8[8], k8[8];
            widen8<IO>(rraw[kb], r8);
            widen8<IO>(kraw[kb], k8);
#pragma unroll
            for (int hf = 0; hf < 2; ++hf) {
                const f32x4 uu = *reinterpret_cast<const f32x4*>(&L.Before[wave][1][32 * kb + 8 * g4 + 4 * hf]);
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    bonus = fmaf(r8[4 * hf + e] * uu[e], k8[4 * hf + e], bonus);
                    dd = fmaf(g8[4 * hf + e], v8[4 * hf + e], dd);
                }
            }
        }
        if (step == 0) {                             // what the first part leaves behind it
            lds_barrier();
            form_state(KFH, KFL, LVH, LVL, v_split, nb, XS);
            form_state(RBH, RBL, GYH, GYL, is_split, nb, XG);
            c_both = c_part;
            continue;
        }
        bonus += __shfl_xor(bonus, 16);
        bonus += __shfl_xor(bonus, 32);
        dd += __shfl_xor(dd, 16);
        dd += __shfl_xor(dd, 32);
        dd = mine ? dd : 0.f;
        if (step == 1) {
            c_both += c_part;
            put_state(c_both, XS, ZS);
            put_state(c_both, XG, ZG);
#pragma unroll
            for (int q = 0; q < 2; ++q) {            // (not kept beyond)
                XS[q] = __builtin_nondeterministic_value(XS[q]);
                XG[q] = __builtin_nondeterministic_value(XG[q]);
            }
        } else if constexpr (SEG) {
            put_state(c_part, XD, ZS);
            put_state(c_part, YD, ZG);
            put_state(c_part, YU, ZG_FRONT);
        }
        lds_barrier();

        // ---- the wave's tokens as i: gv, gk ----
        renew();
        const f32x4 zero = {0.f, 0.f, 0.f, 0.f};
        f32x4 accV[4], gkd[4], gku[4], gru[4], grd[4];                    // gk, gr: entry 2 kb + hf: channels 32 kb + 8 g4 + 4 hf + r; gv: 16 ct + 4 g4 + r
#pragma unroll
        for (int i = 0; i < 4; ++i) accV[i] = gkd[i] = gku[i] = gru[i] = grd[i] = zero;
        const int own = wave >> 1, off = c16 - 4 * g4;                    // the block of 32 tokens with the wave's; the wave's token - register 0's token
        const bool odd = wave & 1;
        // 16 rows (tile tt) of an array x a register operand
        auto rows = [&](unsigned arr, int tt, int kb) { return *reinterpret_cast<const bf16x8*>(lds + arr + row_chunk(c16, 4 * kb + g4) + 2048u * tt); };
        auto product = [&](unsigned hi, unsigned lo, int tt, const bf16x8 (&B)[2][2], auto a_split, auto b_split) {
            f32x4 a = zero;
#pragma unroll
            for (int kb = 0; kb < 2; ++kb) {
                const bf16x8 ah = rows(hi, tt, kb);
                a = mfma(ah, B[kb][0], a);
                if constexpr (decltype(b_split)::value) a = mfma(ah, B[kb][1], a);
                if constexpr (decltype(a_split)::value) a = mfma(rows(lo, tt, kb), B[kb][0], a);
            }
            return a;
        };
        struct Pair { bf16x8 h, l; };
        auto pair = [&](const f32x4& a, const f32x4& c) {
            const float x[8] = {a[0], a[1], a[2], a[3], c[0], c[1], c[2], c[3]};
            Pair p;
            split8<true>(x, p.h, p.l);
            return p;
        };
        // acc[2 kb + hf] += sum over block q of (hi + lo)[channel] (p.h + p.l)
        auto gather = [&](unsigned hi, unsigned lo, int q, const Pair& p, f32x4 (&acc)[4]) {
            bf16x8 ah[4], al[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                ah[i] = tile_across_owned(lds + hi, 32 * q, i >> 1, i & 1, lane);
                al[i] = tile_across_owned(lds + lo, 32 * q, i >> 1, i & 1, lane);
            }
#pragma unroll
            for (int i = 0; i < 4; ++i) acc[i] = mfma(ah[i], p.h, acc[i]);
#pragma unroll
            for (int i = 0; i < 4; ++i) acc[i] = mfma(ah[i], p.l, acc[i]);
#pragma unroll
            for (int i = 0; i < 4; ++i) acc[i] = mfma(al[i], p.h, acc[i]);
#pragma unroll
            for (int i = 0; i < 4; ++i) acc[i] = mfma(al[i], p.l, acc[i]);
        };
        auto gather_gy = [&](int q, const Pair& p) {
            bf16x8 ah[4], al[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                ah[i] = tile_across(lds + GYH, 32 * q, i, lane);
                al[i] = tile_across(lds + GYL, 32 * q, i, lane);
            }
#pragma unroll
            for (int i = 0; i < 4; ++i) accV[i] = mfma(ah[i], p.h, accV[i]);
#pragma unroll
            for (int i = 0; i < 4; ++i) accV[i] = mfma(ah[i], p.l, accV[i]);
#pragma unroll
            for (int i = 0; i < 4; ++i) accV[i] = mfma(al[i], p.h, accV[i]);
        };
        auto d_tile = [&](int tt) { return product(GYH, GYL, tt, V, is_split, v_split); };              // D[t][i], t the rows
        if (mine) {
            auto block = [&](int q, unsigned hi, unsigned lo, const bf16x8 (&K)[2][2], f32x4 (&acc)[4]) {
                gather_gy(q, pair(product(hi, lo, 2 * q, K, is_split, is_split), product(hi, lo, 2 * q + 1, K, is_split, is_split)));
                gather(hi, lo, q, pair(d_tile(2 * q), d_tile(2 * q + 1)), acc);
            };
#pragma unroll 1
            for (int q = 0; q < own; ++q) block(q, RBH, RBL, KB, gku);
            {
                const f32x4 f = product(RFH, RFL, wave, KF, is_split, is_split), g = product(RBH, RBL, wave, KB, is_split, is_split);
                const f32x4 o = odd ? product(RBH, RBL, wave - 1, KB, is_split, is_split) : product(RFH, RFL, wave + 1, KF, is_split, is_split);
                f32x4 a;
#pragma unroll
                for (int e = 0; e < 4; ++e) a[e] = e > off ? f[e] : e < off ? g[e] : bonus;
                gather_gy(own, odd ? pair(o, a) : pair(a, o));
                const f32x4 d = d_tile(wave), m = d_tile(odd ? wave - 1 : wave + 1);
                f32x4 up, dn;
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    up[e] = e < off ? d[e] : 0.f;
                    dn[e] = e > off ? d[e] : 0.f;
                }
                gather(RBH, RBL, own, odd ? pair(m, up) : pair(up, zero), gku);
                gather(RFH, RFL, own, odd ? pair(zero, dn) : pair(dn, m), gkd);
            }
#pragma unroll 1
            for (int q = own + 1; q < nb; ++q) block(q, RFH, RFL, KF, gkd);
        }
        if (step == 1) {
            f32x4 X[2];
            form_state(RFH, RFL, GYH, GYL, is_split, nb, X);
            put_state(c_both, X, ZG_BEHIND);
        }
        lds_barrier();                               // the operands' place is written below
        // ---- the states' share ----
        renew();
        auto state_rows = [&](unsigned z, int i, int kb) {                // rows in the order of gr and gk
            return reinterpret_cast<const bf16x8*>(lds + z + row_chunk(32 * (i >> 1) + 8 * (c16 >> 2) + 4 * (i & 1) + (c16 & 3), 4 * kb + g4));
        };
        auto state_gr = [&](f32x4 (&gr)[4]) {
#pragma unroll
            for (int i = 0; i < 4; ++i) {
#pragma unroll
                for (int kb = 0; kb < 2; ++kb) {
                    const bf16x8 sh = *state_rows(ZS, i, kb), sl = *state_rows(ZS + ZTAIL, i, kb);
                    gr[i] = mfma(sh, GY[kb][0], gr[i]);
                    gr[i] = mfma(sh, GY[kb][1], gr[i]);
                    gr[i] = mfma(sl, GY[kb][0], gr[i]);
                    gr[i] = mfma(sl, GY[kb][1], gr[i]);
                }
                __builtin_amdgcn_sched_barrier(0);
            }
        };
        auto state_gkv = [&](unsigned z, const bf16x8 (&K)[2][2], f32x4 (&gk)[4]) {
#pragma unroll
            for (int i = 0; i < 4; ++i)
#pragma unroll
                for (int kb = 0; kb < 2; ++kb) {
                    const bf16x8 gh = *state_rows(z, i, kb), gl = *state_rows(z + ZTAIL, i, kb);
                    gk[i] = mfma(gh, V[kb][0], gk[i]);
                    gk[i] = mfma(gl, V[kb][0], gk[i]);
                    if constexpr (VSPLIT) {
                        gk[i] = mfma(gh, V[kb][1], gk[i]);
                        gk[i] = mfma(gl, V[kb][1], gk[i]);
                    }
                    // value channels 16 i .. + 15, slot (g4, e): row 32 kb + 8 g4 + e
                    auto across = [&](unsigned arr) {
                        const unsigned ch = 2 * i + ((c16 >> 1) & 1), row = 32 * kb + 8 * g4 + (c16 >> 2);
                        return cat8(lds_read_tr4(reinterpret_cast<const __bf16*>(lds + arr + row_chunk(row, ch) + 8 * (c16 & 1))),
                                    lds_read_tr4(reinterpret_cast<const __bf16*>(lds + arr + row_chunk(row + 4, ch) + 8 * (c16 & 1))));
                    };
                    const bf16x8 th = across(z), tl = across(z + ZTAIL);
                    accV[i] = mfma(th, K[kb][0], accV[i]);
                    accV[i] = mfma(th, K[kb][1], accV[i]);
                    accV[i] = mfma(tl, K[kb][0], accV[i]);
                    __builtin_amdgcn_sched_barrier(0);
                }
        };
        if (step == 1) {
            state_gkv(ZG, KB, gku);
        } else if (two) {
            state_gkv(ZG_BEHIND, KF, gkd);
        } else if constexpr (SEG) {
            state_gkv(ZG, KF, gkd);
            state_gkv(ZG_FRONT, KB, gku);
            state_gr(grd);
            lds_barrier();                           // (S from behind is read)
            put_state(c_part, XU, ZS);
        }
#pragma unroll
        for (int kb = 0; kb < 2; ++kb) {
            store(KFH, KFL, kb, KF[kb][0], KF[kb][1]);
            store(KBH, KBL, kb, KB[kb][0], KB[kb][1]);
            const unsigned at = row_chunk(16 * wave + c16, 4 * kb + g4);
            *reinterpret_cast<bf16x8*>(lds + VH + at) = V[kb][0];
            if constexpr (VSPLIT) *reinterpret_cast<bf16x8*>(lds + VL + at) = V[kb][1];
        }
        if (mine) {
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const float x[4] = {accV[i][0], accV[i][1], accV[i][2], accV[i][3]};
                put_out(A.gv, A.out16, IO{}, x, std::integral_constant<int, 4>{}, 16 * i + 4 * g4, t0);
            }
        }
        lds_barrier();

        // ---- the wave's tokens as t: gr ----
        renew();
        fetch(A.r, t0, rraw, ES);                    // once more, for the results
        fetch(A.k, t0, kraw, ES);
        fetch(A.w, t0, wraw, WS);
        if (mine) {
            auto dt_tile = [&](int tt) { return product(VH, VL, tt, GY, v_split, is_split); };          // D[t][i], i the rows
#pragma unroll 1
            for (int q = 0; q < own; ++q) gather(KFH, KFL, q, pair(dt_tile(2 * q), dt_tile(2 * q + 1)), gru);
            {
                const f32x4 d = dt_tile(wave), m = dt_tile(odd ? wave - 1 : wave + 1);
                f32x4 up, dn;
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    up[e] = e < off ? d[e] : 0.f;
                    dn[e] = e > off ? d[e] : 0.f;
                }
                gather(KFH, KFL, own, odd ? pair(m, up) : pair(up, zero), gru);
                gather(KBH, KBL, own, odd ? pair(zero, dn) : pair(dn, m), grd);
            }
#pragma unroll 1
            for (int q = own + 1; q < nb; ++q) gather(KBH, KBL, q, pair(dt_tile(2 * q), dt_tile(2 * q + 1)), grd);
        }
        if (two && step == 2) state_gr(grd);
        else if (SEG || step == 1) state_gr(gru);
        if (step == 1) {
            f32x4 X[2];
            form_state(KBH, KBL, VH, VL, v_split, nb, X);
            lds_barrier();                           // (S from the front is read)
            put_state(c_both, X, ZS);
        }

        // ---- results: gr, gk, and gw from the sums over the tokens behind ----
        renew();
        float sx[16], tt[16], gu16[16];              // q summed over the wave's tokens behind c16; t; gu token by token
#pragma unroll
        for (int kb = 0; kb < 2; ++kb) {
            float r8[8], k8[8], o8[8], p8[8], e1[8], e2[8];
            factors(kb, e1, e2);
            widen8<IO>(rraw[kb], r8);
            widen8<IO>(kraw[kb], k8);
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                const int x = 8 * kb + e, i = 2 * kb + (e >> 2), m = e & 3;
                const float uu = L.Before[wave][1][32 * kb + 8 * g4 + e] * dd;
                const float ru = gru[i][m] * e1[e], rd = grd[i][m] * e2[e], ku = gku[i][m] * e1[e], kd = gkd[i][m] * e2[e];
                tt[x] = k8[e] * kd + r8[e] * rd;
                float q = r8[e] * (ru - rd) + k8[e] * (ku - kd);
                o8[e] = fmaf(uu, k8[e], ru + rd);
                p8[e] = fmaf(uu, r8[e], ku + kd);
                gu16[x] = r8[e] * k8[e] * dd;
                q = mine ? q : 0.f;
                q += dpp_get<0x101>(q);              // row_shl:1, 2, 4, 8
                q += dpp_get<0x102>(q);
                q += dpp_get<0x104>(q);
                q += dpp_get<0x108>(q);
                if (c16 == 0) L.Q[wave][32 * kb + 8 * g4 + e] = q;
                sx[x] = dpp_get<0x101>(q);
            }
            if (mine) {
                put_out(A.gr, A.out16, IO{}, o8, std::integral_constant<int, 8>{}, 32 * kb + 8 * g4, t0);
                put_out(A.gk, A.out16, IO{}, p8, std::integral_constant<int, 8>{}, 32 * kb + 8 * g4, t0);
            }
        }
        gu += row_sums16(gu16, lane, gu_at);
        lds_barrier();
        {
            if constexpr (SEG) xrun = L.X[0][lane] + L.X[1][lane];
            float after = 0.f, total = 0.f;
#pragma unroll
            for (int g = 0; g < PART_WAVES; ++g) {
                const float t = L.Q[g][lane];
                after += g > wave ? t : 0.f;
                total += t;
            }
            L.Before[wave][0][lane] = xrun + after;
            xrun += total;
        }
        if (mine) {
#pragma unroll
            for (int kb = 0; kb < 2; ++kb) {
                float w8[8], o8[8];
                widen8<WT>(wraw[kb], w8);
#pragma unroll
                for (int hf = 0; hf < 2; ++hf) {
                    const f32x4 behind = *reinterpret_cast<const f32x4*>(&L.Before[wave][0][32 * kb + 8 * g4 + 4 * hf]);
#pragma unroll
                    for (int m = 0; m < 4; ++m) {
                        const int e = 4 * hf + m, x = 8 * kb + e;
                        const float ld = W_IS_EW ? w8[e] : -fast_exp2(fmaf(w8[e], LOG2E, LOG2_LOG2E)) * (1.0f / LOG2E);
                        o8[e] = ld * ((behind[m] + sx[x]) - tt[x]);
                    }
                }
                put_out(A.gw, A.w16, WT{}, o8, std::integral_constant<int, 8>{}, 32 * kb + 8 * g4, t0);
            }
        }
    }
    if (bail) {
        if constexpr (SEG) {
            // the sweeps take the states that enter the segment from memory
            float* const own = A.seg_own + ((size_t)bh * nseg + seg) * BWD_SEG_FLOATS;
#pragma unroll 1
            for (int m = 0; m < 4; m += 2) {
                f32x4 S[2], G[2];
                entering(m == 0, S, G);
#pragma unroll
                for (int q = 0; q < 2; ++q) {
                    *reinterpret_cast<f32x4*>(own + m * SEG_STATE + seg_frag(jt, ct0 + q, lane)) = S[q];
                    *reinterpret_cast<f32x4*>(own + (m + 1) * SEG_STATE + seg_frag(jt, ct0 + q, lane)) = G[q];
                }
            }
            A.seg_ws = A.seg_own;
        }
        __syncthreads();
        bwd_sweep_sequence<IO, WT, W_IS_EW>(A, *reinterpret_cast<Sweep*>(lds), sFlag, bh, seg);
        return;
    }
    lds_barrier();
    L.Q[wave][32 * (gu_at >> 3) + 8 * g4 + (gu_at & 7)] = gu;
    lds_barrier();
    if (threadIdx.x < HN) {
        float x = 0.f;
#pragma unroll
        for (int g = 0; g < PART_WAVES; ++g) x += L.Q[g][threadIdx.x];
        A.gu_part[((size_t)b * nseg + seg) * C + h * HN + threadIdx.x] = x;
    }
}

// What every segment of up to 128 tokens leaves behind it in both directions by itself, S (k, v) and G (r, gy), with its decay and whether it is out of range:
// wkv6_bwd_seg_state_kernel's results, a part at a time (two pairs of barriers in place of two for every 32 tokens; the up states' factors first, then, in
// their place, the down states').  All exponents are <= 0.  One workgroup on a compute unit (136 KB of LDS), for calls that do not have more.
template <typename IO, typename WT, bool W_IS_EW>
__global__ __launch_bounds__(64 * PART_WAVES, 2)
void wkv6_bwd_part_state_kernel(const void* r_, const void* k_, const void* v_, const void* w_, const float* gy_, float* ws, int* flags, int T, int C, int H,
                                int sequences, int nseg)
{
    constexpr bool VSPLIT = !__is_same(IO, __hip_bfloat16);
    constexpr unsigned ES = (unsigned)sizeof(IO), WS = (unsigned)sizeof(WT), ARR = PART * 128u;
    constexpr unsigned KH = 0, KL = ARR, RH = 2 * ARR, RL = 3 * ARR, GYH = 4 * ARR, GYL = 5 * ARR, VH = 6 * ARR, VL = 7 * ARR, TAB = (VSPLIT ? 8 : 7) * ARR;
    struct Tables { float Tot[PART_WAVES][HN], Before[PART_WAVES][2][HN]; };
    __shared__ __attribute__((aligned(16))) unsigned char lds[TAB + sizeof(Tables)];
    Tables& L = *reinterpret_cast<Tables*>(lds + TAB);
    const int lane = threadIdx.x & 63, g4 = lane >> 4, c16 = lane & 15;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    int bh, seg;
    seg_of_block(blockIdx.x, nseg, bh, seg);
    if (bh >= sequences) return;
    const size_t base = (size_t)(bh / H) * T * C + (size_t)(bh % H) * HN;
    const unsigned n_el = (unsigned)((size_t)(T - 1) * C + HN);
    const int nchunk = (T + LC - 1) / LC, cps = (nchunk + nseg - 1) / nseg;
    const int first = seg * cps * LC, n = min(cps * LC, T - first), nb = (n + LC - 1) / LC;
    auto fetch = [&](const void* p, auto& raw, unsigned es) {
        const __amdgpu_buffer_rsrc_t rs = make_rsrc(static_cast<const char*>(p) + base * es, n_el * es);
        constexpr int pieces = sizeof(raw[0]) / 16;
        const unsigned vo = ((unsigned)c16 * C + 8 * g4) * es, so = (unsigned)(first + 16 * wave) * C * es;
#pragma unroll
        for (int kb = 0; kb < 2; ++kb)
#pragma unroll
            for (int i = 0; i < pieces; ++i) raw[kb][i] = BufRaw<16>::ld(rs, vo + 32u * kb * es + 16u * i, so);
    };
    u32x4 wraw[2][WS / 2], rraw[2][ES / 2], kraw[2][ES / 2], vraw[2][ES / 2], graw[2][2];
    fetch(w_, wraw, WS);
    fetch(k_, kraw, ES);
    fetch(r_, rraw, ES);
    fetch(v_, vraw, ES);
    fetch(gy_, graw, 4u);
    float x[2][8];
#pragma unroll
    for (int kb = 0; kb < 2; ++kb) {
        summed_decays<WT, W_IS_EW>(wraw[kb], 16 * wave + c16 >= n, x[kb]);
        if (c16 == 15) {
#pragma unroll
            for (int hf = 0; hf < 2; ++hf)
                *reinterpret_cast<f32x4*>(&L.Tot[wave][32 * kb + 8 * g4 + 4 * hf]) = f32x4{x[kb][4 * hf], x[kb][4 * hf + 1], x[kb][4 * hf + 2], x[kb][4 * hf + 3]};
        }
    }
    auto store = [&](unsigned arr, int kb, const bf16x8& o) { *reinterpret_cast<bf16x8*>(lds + arr + row_chunk(16 * wave + c16, 4 * kb + g4)) = o; };
#pragma unroll
    for (int kb = 0; kb < 2; ++kb) {
        float o8[8];
        bf16x8 hi, lo;
        widen8<float>(graw[kb], o8);
        split8<true>(o8, hi, lo);
        store(GYH, kb, hi);
        store(GYL, kb, lo);
        if constexpr (VSPLIT) {
            widen8<IO>(vraw[kb], o8);
            split8<true>(o8, hi, lo);
            store(VH, kb, hi);
            store(VL, kb, lo);
        } else {
            store(VH, kb, __builtin_bit_cast(bf16x8, vraw[kb][0]));
        }
    }
    lds_barrier();
    float before = 0.f, total = 0.f, t[PART_WAVES];
#pragma unroll
    for (int g = 0; g < PART_WAVES; ++g) {
        t[g] = L.Tot[g][lane];
        before += g < wave ? t[g] : 0.f;
        total += t[g];
    }
    bool out_of_range = false;
#pragma unroll
    for (int g = 0; g < PART_WAVES; g += 2) out_of_range |= !(t[g] + t[g + 1] >= -SAFE_DECAY * LOG2E);        // a 32-token chunk
    L.Before[wave][0][lane] = before;
    L.Before[wave][1][lane] = total - before;
    float* const out = ws + ((size_t)bh * nseg + seg) * BWD_SEG_FLOATS;
    if (wave == 0) {                                                      // every wave saw all totals
        out[4 * SEG_STATE + lane] = fast_exp2(total);
        const bool any = __builtin_amdgcn_ballot_w64(out_of_range) != 0ull;
        if (lane == 0) flags[(size_t)bh * nseg + seg] = any ? 1 : 0;
    }
    const int jt = wave & 3, ct0 = 2 * (wave >> 2);                       // column j = 16 jt + c16, rows (value channels) 16 (ct0 + q) + 4 g4 + r
#pragma unroll
    for (int dn = 0; dn < 2; ++dn) {
#pragma unroll
        for (int kb = 0; kb < 2; ++kb) {
            float f[8];
#pragma unroll
            for (int hf = 0; hf < 2; ++hf) {
                const f32x4 b = *reinterpret_cast<const f32x4*>(&L.Before[wave][1 - dn][32 * kb + 8 * g4 + 4 * hf]);
#pragma unroll
                for (int e = 0; e < 4; ++e) f[4 * hf + e] = fast_exp2(dn ? b[e] + dpp_get<0x111>(x[kb][4 * hf + e]) : b[e] - x[kb][4 * hf + e]);
            }
            auto times = [&](const u32x4* raw, unsigned h, unsigned l) {
                float o8[8];
                bf16x8 hi, lo;
                widen8<IO>(raw, o8);
#pragma unroll
                for (int e = 0; e < 8; ++e) o8[e] *= f[e];
                split8<true>(o8, hi, lo);
                store(h, kb, hi);
                store(l, kb, lo);
            };
            times(kraw[kb], KH, KL);
            times(rraw[kb], RH, RL);
        }
        lds_barrier();
        f32x4 S[2], G[2];
        S[0] = S[1] = G[0] = G[1] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll 1
        for (int q = 0; q < nb; ++q) {
            const bf16x8 kh = tile_across(lds + KH, 32 * q, jt, lane), kl = tile_across(lds + KL, 32 * q, jt, lane);
            const bf16x8 rh = tile_across(lds + RH, 32 * q, jt, lane), rl = tile_across(lds + RL, 32 * q, jt, lane);
#pragma unroll
            for (int i = 0; i < 2; ++i) {
                const bf16x8 vh = tile_across(lds + VH, 32 * q, ct0 + i, lane), gh = tile_across(lds + GYH, 32 * q, ct0 + i, lane),
                             gl = tile_across(lds + GYL, 32 * q, ct0 + i, lane);
                S[i] = mfma(vh, kh, S[i]);
                G[i] = mfma(gh, rh, G[i]);
                S[i] = mfma(vh, kl, S[i]);
                G[i] = mfma(gh, rl, G[i]);
                if constexpr (VSPLIT) S[i] = mfma(tile_across(lds + VL, 32 * q, ct0 + i, lane), kh, S[i]);
                G[i] = mfma(gl, rh, G[i]);
            }
        }
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            *reinterpret_cast<f32x4*>(out + 2 * dn * SEG_STATE + seg_frag(jt, ct0 + i, lane)) = S[i];
            *reinterpret_cast<f32x4*>(out + (2 * dn + 1) * SEG_STATE + seg_frag(jt, ct0 + i, lane)) = G[i];
        }
        if (dn == 0) lds_barrier();                                       // the operands' place is written next
    }
}

}  // namespace wkv6_detail
}  // namespace vrwkv
