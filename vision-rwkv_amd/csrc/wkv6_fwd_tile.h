// wkv6 forward, sequences (or segments) of up to 256 tokens as one or two matrix products (gfx950, bf16 MFMA, fp32 accumulate).
//
// Both passes of the scan at once.  In a part of up to 128 tokens, with P_t the cumulative log2 decay up to and with token t, Pex_t = P_(t-1),
//   y_t = sum_i A[t][i] v_i,   A[t][i] = sum_j r_t[j] k_i[j] 2^(Pex_t - P_i)[j]   i < t   (ascending pass)
//                                        sum_j r_t[j] k_i[j] 2^(Pex_i - P_t)[j]   i > t   (descending pass)
//                                        sum_j r_t[j] u[j] k_t[j]                 i = t   (bonus)
// and one reference exponent per channel, c = P_end / 2, the factors of A take two exponentials a token and channel:
//   e1_t = 2^(Pex_t - c), e2_t = 2^(c - P_t);   rf = r e1, kf = k e2 (i < t);   rb = r e2, kb = k e1 (i > t).
// States that enter a part from the front (S_up) and from behind (S_down) add rf (2^c S_up) + rb (2^c S_down); what it leaves behind is
// 2^c sum_i kf_i v_i in front of the next part and 2^c sum_i kb_i v_i behind the last one.  A longer sequence is two parts: the second one first, which
// keeps its rf, then the first one with the state from behind, then the second one's share of the state from the front.  A segment of a cut sequence
// starts from the states that wkv6_segment.h provides.
//
// Against the chunked kernel (two passes of 32-token chunks) a token and channel is prepared once and not twice, with three exponentials instead of
// six, the 64 x 64 states are scaled and split once per part and not once per chunk, and y is not fetched again.
//
// A workgroup of eight waves holds a part, two (fp16 and fp32, whose v is split: one) share a compute unit; a wave owns 16 tokens.  Element-wise stage: lane = (token c16, eight
// channels of each half), the layout of the matrix operands, so rf and rb stay in registers and kf, kb, v (head and tail) leave for LDS in 16-byte pieces;
// the decays are summed along a row of 16 lanes, then over the waves.  Matrix stage, no barrier inside: the wave walks the 32-token blocks of the part's
// tokens i, A^T leaves its accumulators as the next product's operand, v is read across with ds_read_b64_tr_b16, y is transposed in accumulators.
// Computed operands are split into bf16 head + tail, products head*head + head*tail + tail*head, as in the chunked kernel.
//
// Bound by latency: the workgroups of a compute unit spend a third of their time on rows on their way, each part is a chain of an element-wise and a
// matrix stage, and 768 sequences are one and a half rounds.  us, chunked kernel -> here, bf16 / fp32: 768 sequences of 196 tokens 62 -> 46 / 80 -> 67,
// of 128 36 -> 22 / 51 -> 35, of 49 22 -> 15 / 31 -> 22; 3 sequences of 196 23.0 -> 16.9 / 23.6 -> 18.7.
//
// Range: |P_end| <= 200 in a part (e^-138 over it), less for rows of unusual size (PART_FREE in wkv6_segment.h).  Sequences beyond go through the chunked
// kernel's code (range per 32 tokens, the sequential recurrence beyond that).
#pragma once
#include "wkv6_fwd_chunk.h"

namespace vrwkv {
namespace wkv6_detail {

constexpr int TILE_TOKENS = 2 * PART;               // most tokens of a sequence or segment
static_assert(PART_WAVES == FW_WAVES, "the chunked kernel's code runs on the same workgroup");

struct FwdTileArgs {
    const void *r, *k, *v, *w;
    const float* u;
    float* y;
    int T, C, H, sequences, nseg;
    const float* seg_ws;                             // the segments' states
    const int* seg_flags;
    float* seg_own;                                  // SEGMENTS 2: room for the states that enter the segments
};

// SEGMENTS: of cut sequences, 1 with the states that enter them, 2 with those that they leave by themselves (of one part; in a kernel of its own, for the
// registers).  LOOSE: 16-bit rows that do not lie on 4 bytes, fetched element by element (the same results, in a kernel of its own: the packing takes registers).
template <typename IO, typename WT, bool W_IS_EW, int SEGMENTS, bool LOOSE = false>
__global__ __launch_bounds__(64 * PART_WAVES, 4)
void wkv6_fwd_tile_kernel(FwdTileArgs A)
{
    constexpr bool VSPLIT = !__is_same(IO, __hip_bfloat16);
    constexpr bool SEG = SEGMENTS != 0, FOLD = SEGMENTS == 2;
    constexpr unsigned ES = (unsigned)sizeof(IO), WS = (unsigned)sizeof(WT), ARR = PART * 128u;
    constexpr unsigned KFH = 0, KFL = ARR, KBH = 2 * ARR, KBL = 3 * ARR, VH = 4 * ARR, VL = 5 * ARR;
    __shared__ __attribute__((aligned(16))) unsigned char lds[(VSPLIT ? 6 : 5) * ARR];
    static_assert(sizeof(lds) >= sizeof(FwdLds<VSPLIT>) * 2 + 16, "the chunked kernel's operands must fit");
    // The waves' decay sums lie where the first factors of k go afterwards (a barrier apart), the sums in front of a wave and u in its own rows of the
    // second ones, a scaled state (head, tail) where v goes.
    constexpr unsigned ZH = VH, ZL = VH + ARR / 2, OWN = 16 * 128;

    // (Addresses are formed anew in every stage, from an opaque copy of the lane number: kept from the kernel's start they would take more registers than
    // there are.)
    int lane = threadIdx.x & 63, g4 = lane >> 4, c16 = lane & 15;
    auto renew = [&]() {
        lane = threadIdx.x & 63;
        asm volatile("" : "+v"(lane));
        g4 = lane >> 4;
        c16 = lane & 15;
    };
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int T = A.T, C = A.C, nseg = SEG ? A.nseg : 1;
    const int nchunk = (T + LC - 1) / LC, cps = (nchunk + nseg - 1) / nseg;
    int bh = blockIdx.x, seg = 0;
    bool bail = false;
    if constexpr (SEG) {
        seg_of_block(blockIdx.x, nseg, bh, seg);
        if (bh >= A.sequences) return;
        const int f = lane < nseg ? A.seg_flags[(size_t)bh * nseg + lane] : 0;
        if (__builtin_amdgcn_ballot_w64(f != 0) != 0ull) {               // the whole sequence is left to its first segment
            if (seg != 0) return;
            bail = true;
        }
    }
    const int b = bh / A.H, h = bh % A.H;
    const size_t base = (size_t)b * T * C + (size_t)h * HN;
    const int first = seg * cps * LC, n = min(cps * LC, T - first);
    const bool two = !FOLD && n > PART;
    const int n1 = two ? ((n + LC - 1) / LC + 1) / 2 * LC : n;           // tokens of the first part

    // eight channels 32 kb + 8 g4 .. + 7 of a row, packed as they lie, in 16-byte pieces
    constexpr int PI = (int)ES / 2, PW = (int)WS / 2;
    auto desc = [&](const void* p, unsigned es) {
        return make_rsrc(static_cast<const char*>(p) + base * es, (unsigned)(((size_t)(T - 1) * C + HN) * es));
    };
    // Rows past T lie outside the descriptors and read 0: k = r = 0 switches such a token off, its decay is set to 1 below.
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
    // y of the wave's tokens: value channels 16 vt + 4 g4 .. + 3 of token c16
    auto y_lane = [&]() { return ((unsigned)c16 * C + 4 * g4) * 4u; };
    auto y_row = [&](int t0) { return (unsigned)(t0 + 16 * wave) * C * 4u; };

    // X: a wave's part of a 64 x 64 state, as the accumulators hold it: tile jt = 2 (wave / 4) + q has rows j = 16 jt + 4 g4 + r, column 16 (wave & 3) + c16
    f32x4v X[2];
    const int jt0 = 2 * (wave >> 2), it0 = wave & 3;
    bf16x8 Hh[2], Hl[2];                             // rf of the second part
    float c_first = 0.f, c_second = 0.f;             // c of the parts, of channel `lane`

    // X times 2^c (c of one or two parts, down to -200: in two halves) as operands into LDS: rows are value channels
    auto put_state = [&](float c) {
#pragma unroll
        for (int q = 0; q < 2; ++q) {
            const int jt = jt0 + q;
            float x[4];
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const float f = fast_exp2(0.5f * __shfl(c, 16 * jt + 4 * g4 + e));
                x[e] = X[q][e] * f * f;
            }
            if constexpr (SEG) X[q] = f32x4v{x[0], x[1], x[2], x[3]};
            unsigned xh[2], xl[2];
            split4(x, xh, xl);
            const unsigned at = row_chunk(16 * it0 + c16, 2 * jt + (g4 >> 1)) + 8 * (g4 & 1);
            *reinterpret_cast<uint2*>(lds + ZH + at) = make_uint2(xh[0], xh[1]);
            *reinterpret_cast<uint2*>(lds + ZL + at) = make_uint2(xl[0], xl[1]);
        }
    };
    auto add_state = [&](const bf16x8 (&Rh)[2], const bf16x8 (&Rl)[2], f32x4v (&y)[4]) {
#pragma unroll
        for (int vt = 0; vt < 4; ++vt)
#pragma unroll
            for (int kb = 0; kb < 2; ++kb) {
                const unsigned at = row_chunk(16 * vt + c16, 4 * kb + g4);
                const bf16x8 zh = *reinterpret_cast<const bf16x8*>(lds + ZH + at), zl = *reinterpret_cast<const bf16x8*>(lds + ZL + at);
                y[vt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(zh, Rh[kb], y[vt], 0, 0, 0);
                y[vt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(zl, Rh[kb], y[vt], 0, 0, 0);
                y[vt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(zh, Rl[kb], y[vt], 0, 0, 0);
            }
    };
    auto load_state = [&](bool down) {
        const float* in = A.seg_ws + ((size_t)bh * nseg + seg) * SEG_FLOATS + (down ? SEG_STATE : 0);
#pragma unroll
        for (int q = 0; q < 2; ++q) X[q] = *reinterpret_cast<const f32x4v*>(in + seg_frag(it0, jt0 + q, lane));
    };
    // the same from the states that the segments in front of this one, or behind it, leave by themselves, each over the decays in between
    auto fold_states = [&](bool down, f32x4v (&S)[2]) {
        constexpr int U = 4;
        const int count = down ? nseg - 1 - seg : seg;
        S[0] = S[1] = f32x4v{0.f, 0.f, 0.f, 0.f};
#pragma unroll 1
        for (int i0 = 0; i0 < count; i0 += U) {
            f32x4v l[U][2], d[U][2];
#pragma unroll
            for (int i = 0; i < U; ++i)
                if (i0 + i < count) {
                    const float* p = A.seg_ws + ((size_t)bh * nseg + (down ? nseg - 1 - i0 - i : i0 + i)) * SEG_FLOATS;
#pragma unroll
                    for (int q = 0; q < 2; ++q) {
                        l[i][q] = *reinterpret_cast<const f32x4v*>(p + (down ? SEG_STATE : 0) + seg_frag(it0, jt0 + q, lane));
                        d[i][q] = *reinterpret_cast<const f32x4v*>(p + 2 * SEG_STATE + 16 * (jt0 + q) + 4 * g4);
                    }
                }
#pragma unroll
            for (int i = 0; i < U; ++i)
                if (i0 + i < count) {
                    S[0] = S[0] * d[i][0] + l[i][0];
                    S[1] = S[1] * d[i][1] + l[i][1];
                }
        }
    };
    auto across = [&](unsigned arr, int q, int ct) { return read_across(lds + arr, q, ct, lane); };

    u32x4 wraw[2][PW];
    X[0] = X[1] = f32x4v{0.f, 0.f, 0.f, 0.f};
    const float uj = A.u[h * HN + lane];
#pragma unroll 1
    for (int part = two ? 1 : 0; part >= 0 && !bail; --part) {
        renew();
        const int t0 = first + (part ? n1 : 0), np = part ? n - n1 : n1, nb = (np + LC - 1) / LC;
        const bool mine = wave < 2 * nb;             // the wave has tokens, or rows of zeros that another one reads
        u32x4 rraw[2][PI], kraw[2][PI], vraw[2][PI];
        if (part == 1 || !two) fetch(A.w, t0, wraw, WS);
        fetch(A.r, t0, rraw, ES);
        fetch(A.k, t0, kraw, ES);
        fetch(A.v, t0, vraw, ES);
        f32x4v XF[2];                                // the state from the front, where it is folded here
        if constexpr (FOLD) {                        // (of one part)
            fold_states(true, X);
            fold_states(false, XF);
        }
        float x[2][8];                               // log2 decays summed over the wave's tokens
        const bool past = 16 * wave + c16 >= np;
#pragma unroll
        for (int kb = 0; kb < 2; ++kb) {
            summed_decays<WT, W_IS_EW>(wraw[kb], past, x[kb]);
            if (c16 == 15) {
#pragma unroll
                for (int hf = 0; hf < 2; ++hf)
                    *reinterpret_cast<f32x4*>(lds + KFH + 256 * wave + 128 * kb + 32 * g4 + 16 * hf) =
                        f32x4{x[kb][4 * hf], x[kb][4 * hf + 1], x[kb][4 * hf + 2], x[kb][4 * hf + 3]};
            }
        }
        lds_barrier();
        renew();
        float total = 0.f;
        {
            float s = 0.f;
#pragma unroll
            for (int g = 0; g < PART_WAVES; ++g) {
                const float t = *reinterpret_cast<const float*>(lds + KFH + 256 * g + 4 * lane);
                s += g < wave ? t : 0.f;
                total += t;
            }
            (part ? c_second : c_first) = 0.5f * total;
            float* const own = reinterpret_cast<float*>(lds + KFL + OWN * wave);
            own[lane] = s - 0.5f * total;
            own[HN + lane] = uj;
        }
        if (__builtin_amdgcn_ballot_w64(!(total >= -PART_FREE)) != 0ull) {       // the same in every wave
            const float mr = largest_of_wave(mine ? largest16<IO>(rraw[0], rraw[1]) : 0.f), mk = largest_of_wave(mine ? largest16<IO>(kraw[0], kraw[1]) : 0.f),
                        mv = largest_of_wave(mine ? largest16<IO>(vraw[0], vraw[1]) : 0.f);
            if (lane == 0) *reinterpret_cast<f32x4*>(lds + KFH + 2048 + 16 * wave) = f32x4{mr, mk, mv, 0.f};      // (behind the decay sums)
            lds_barrier();
            f32x4 m = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int g = 0; g < PART_WAVES; ++g) {
                const f32x4 x = *reinterpret_cast<const f32x4*>(lds + KFH + 2048 + 16 * g);
#pragma unroll
                for (int e = 0; e < 3; ++e) m[e] = fmaxf(m[e], x[e]);
            }
            const float lr = log2_of_largest(m[0]), lk = log2_of_largest(m[1]), lkv = lk + log2_of_largest(m[2]);
            if (__builtin_amdgcn_ballot_w64(!(total >= -part_decay(fminf(fminf(lr, lk), lkv), fmaxf(fmaxf(lr, lk), lkv)))) != 0ull) { bail = true; break; }
        }
        lds_barrier();                               // the sums are read: their place is written below
        // bonus: sum_j r_t[j] u[j] k_t[j] of the lane's token, over the four lanes that share it
        f32x4 before[2][2];
        float bonus = 0.f;
#pragma unroll
        for (int kb = 0; kb < 2; ++kb) {
            float r8[8], k8[8];
            widen8<IO>(rraw[kb], r8);
            widen8<IO>(kraw[kb], k8);
#pragma unroll
            for (int hf = 0; hf < 2; ++hf) {
                const unsigned char* own = lds + KFL + OWN * wave + 128 * kb + 32 * g4 + 16 * hf;
                before[kb][hf] = *reinterpret_cast<const f32x4*>(own);
                const f32x4 uu = *reinterpret_cast<const f32x4*>(own + 256);
#pragma unroll
                for (int e = 0; e < 4; ++e) bonus = fmaf(r8[4 * hf + e] * uu[e], k8[4 * hf + e], bonus);
            }
            // (widened again where they are used next: kept so they would take twice the registers)
#pragma unroll
            for (int i = 0; i < PI; ++i) asm volatile("" : "+v"(rraw[kb][i]), "+v"(kraw[kb][i]));
        }
        bonus += __shfl_xor(bonus, 16);
        bonus += __shfl_xor(bonus, 32);
        renew();
        f32x4v accY[4];                              // y^T: value channels 16 vt + 4 g4 + r of token c16
#pragma unroll
        for (int vt = 0; vt < 4; ++vt) accY[vt] = f32x4v{0.f, 0.f, 0.f, 0.f};
        bf16x8 RFh[2], RFl[2], RBh[2], RBl[2];       // slot (g4, e) of half kb: channel 32 kb + 8 g4 + e
#pragma unroll
        for (int kb = 0; kb < 2; ++kb) {
            const unsigned at = row_chunk(16 * wave + c16, 4 * kb + g4);
            float e1[8], e2[8];
#pragma unroll
            for (int hf = 0; hf < 2; ++hf)
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const float s = before[kb][hf][e], d = x[kb][4 * hf + e];
                    e1[4 * hf + e] = fast_exp2(s + dpp_get<0x111>(d));
                    e2[4 * hf + e] = fast_exp2(-(s + d));
                }
            auto times = [&](const u32x4* raw, const float (&f)[8], bf16x8& hi, bf16x8& lo) {
                float o8[8];
                widen8<IO>(raw, o8);
#pragma unroll
                for (int e = 0; e < 8; ++e) o8[e] *= f[e];
                split8<true>(o8, hi, lo);
                __builtin_amdgcn_sched_barrier(0);
            };
            bf16x8 hi, lo;
            times(kraw[kb], e2, hi, lo);
            *reinterpret_cast<bf16x8*>(lds + KFH + at) = hi;
            *reinterpret_cast<bf16x8*>(lds + KFL + at) = lo;
            times(kraw[kb], e1, hi, lo);
            *reinterpret_cast<bf16x8*>(lds + KBH + at) = hi;
            *reinterpret_cast<bf16x8*>(lds + KBL + at) = lo;
            times(rraw[kb], e1, RFh[kb], RFl[kb]);
            times(rraw[kb], e2, RBh[kb], RBl[kb]);
        }
        renew();
        // states that enter the part: from behind (the second part's, or the segment's), from the front (the segment's, of a first part)
        if (SEG || (two && part == 0)) {
            if constexpr (SEG) {
                if (!FOLD && (part == 1 || !two)) load_state(true);
            }
            put_state(part ? c_second : two ? c_first + c_second : c_first);
            lds_barrier();
            add_state(RBh, RBl, accY);
            lds_barrier();
            if constexpr (SEG) {
                if (part == 0) {
                    if constexpr (FOLD) { X[0] = XF[0]; X[1] = XF[1]; }
                    else load_state(false);
                    put_state(c_first);
                    lds_barrier();
                    add_state(RFh, RFl, accY);
                    lds_barrier();
                }
            }
        }
#pragma unroll
        for (int kb = 0; kb < 2; ++kb) {
            const unsigned at = row_chunk(16 * wave + c16, 4 * kb + g4);
            if constexpr (!VSPLIT) {
                *reinterpret_cast<u32x4*>(lds + VH + at) = vraw[kb][0];
            } else {
                float v8[8];
                bf16x8 hi, lo;
                widen8<IO>(vraw[kb], v8);
                split8<true>(v8, hi, lo);
                *reinterpret_cast<bf16x8*>(lds + VH + at) = hi;
                *reinterpret_cast<bf16x8*>(lds + VL + at) = lo;
            }
        }
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");     // (v was the last to be fetched; the second part's y rows are stored by then)
        lds_barrier();
        renew();
        if (part == 1) fetch(A.w, first, wraw, WS);  // the first part's decays, behind the products
        if (mine) {
            // A^T tile (16 tokens i, the wave's tokens t)
            auto tile = [&](unsigned hi, unsigned lo, int it, const bf16x8 (&Rh)[2], const bf16x8 (&Rl)[2], f32x4v& a) {
#pragma unroll
                for (int kb = 0; kb < 2; ++kb) {
                    const unsigned at = row_chunk(c16, 4 * kb + g4) + 2048 * it;
                    const bf16x8 kh = *reinterpret_cast<const bf16x8*>(lds + hi + at), kl = *reinterpret_cast<const bf16x8*>(lds + lo + at);
                    a = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kh, Rh[kb], a, 0, 0, 0);
                    a = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kh, Rl[kb], a, 0, 0, 0);
                    a = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kl, Rh[kb], a, 0, 0, 0);
                }
            };
            auto words = [](const f32x4v& a, unsigned* hw, unsigned* lw) {
#pragma unroll
                for (int p = 0; p < 2; ++p) {
                    hw[p] = pack_bf16(a[2 * p], a[2 * p + 1]);
                    lw[p] = tail_bf16(a[2 * p], a[2 * p + 1], hw[p]);
                }
            };
            // y^T += v^T A^T over the tokens of block q
            auto values = [&](int q, const unsigned (&hw)[4], const unsigned (&lw)[4]) {
                const bf16x8 ah = words8(hw[0], hw[1], hw[2], hw[3]), al = words8(lw[0], lw[1], lw[2], lw[3]);
#pragma unroll
                for (int vt = 0; vt < 4; ++vt) {
                    const bf16x8 vv = across(VH, q, vt);
                    accY[vt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(vv, ah, accY[vt], 0, 0, 0);
                    accY[vt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(vv, al, accY[vt], 0, 0, 0);
                    if constexpr (VSPLIT) accY[vt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(across(VL, q, vt), ah, accY[vt], 0, 0, 0);
                }
            };
            const int own = wave >> 1;               // the block of 32 tokens with the wave's
            auto block = [&](int q, unsigned hi, unsigned lo, const bf16x8 (&Rh)[2], const bf16x8 (&Rl)[2]) {
                f32x4v a0 = {0.f, 0.f, 0.f, 0.f}, a1 = {0.f, 0.f, 0.f, 0.f};
                tile(hi, lo, 2 * q, Rh, Rl, a0);
                tile(hi, lo, 2 * q + 1, Rh, Rl, a1);
                unsigned hw[4], lw[4];
                words(a0, hw, lw);
                words(a1, hw + 2, lw + 2);
                values(q, hw, lw);
            };
#pragma unroll 1
            for (int q = 0; q < own; ++q) block(q, KFH, KFL, RFh, RFl);
            {
                // the block with the wave's own tile: i < t, i > t and the bonus at i = t there, the block's other tile in front of it or behind
                f32x4v f = {0.f, 0.f, 0.f, 0.f}, g = {0.f, 0.f, 0.f, 0.f}, o = {0.f, 0.f, 0.f, 0.f};
                const bool odd = wave & 1;
                tile(KFH, KFL, wave, RFh, RFl, f);
                tile(KBH, KBL, wave, RBh, RBl, g);
                if (odd) tile(KFH, KFL, wave - 1, RFh, RFl, o);
                else tile(KBH, KBL, wave + 1, RBh, RBl, o);
                const int off = c16 - 4 * g4;                             // t - i of register 0
                f32x4v d;
#pragma unroll
                for (int e = 0; e < 4; ++e) d[e] = e < off ? f[e] : e > off ? g[e] : bonus;
                unsigned hw[4], lw[4];
                words(odd ? o : d, hw, lw);
                words(odd ? d : o, hw + 2, lw + 2);
                values(own, hw, lw);
            }
#pragma unroll 1
            for (int q = own + 1; q < nb; ++q) block(q, KBH, KBL, RBh, RBl);
            renew();
            const __amdgpu_buffer_rsrc_t rsy = desc(A.y, 4);
#pragma unroll
            for (int vt = 0; vt < 4; ++vt)
                BufRaw<16>::st(__builtin_bit_cast(typename BufRaw<16>::type, accY[vt]), rsy, y_lane() + 64u * vt, y_row(t0));
        }
        if (two) {
            renew();
            // what the part leaves behind: from behind for the first part, from the front for the second one
            if constexpr (!SEG) X[0] = X[1] = f32x4v{0.f, 0.f, 0.f, 0.f};      // (a segment's: on top of what entered on that side, scaled by put_state)
            const unsigned hi = part ? KBH : KFH, lo = part ? KBL : KFL;
#pragma unroll 1
            for (int q = 0; q < nb; ++q) {
                const bf16x8 vv = across(VH, q, it0);
                bf16x8 vl;
                if constexpr (VSPLIT) vl = across(VL, q, it0);
#pragma unroll
                for (int j = 0; j < 2; ++j) {
                    const bf16x8 kh = across(hi, q, jt0 + j), kl = across(lo, q, jt0 + j);
                    X[j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kh, vv, X[j], 0, 0, 0);
                    X[j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kl, vv, X[j], 0, 0, 0);
                    if constexpr (VSPLIT) X[j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kh, vl, X[j], 0, 0, 0);
                }
            }
            if (part == 1) {
#pragma unroll
                for (int kb = 0; kb < 2; ++kb) { Hh[kb] = RFh[kb]; Hl[kb] = RFl[kb]; }
            }
            lds_barrier();                           // the operands' place is written next
        }
    }
    if (two && !bail) {
        // the second part's share of the state from the front
        renew();
        const __amdgpu_buffer_rsrc_t rsy = desc(A.y, 4);
        f32x4v Y2[4];                                // its y, stored by the wave itself (the wait for v since then was one for every access before it)
#pragma unroll
        for (int vt = 0; vt < 4; ++vt) Y2[vt] = __builtin_bit_cast(f32x4v, BufRaw<16>::ld(rsy, y_lane() + 64u * vt, y_row(first + n1)));
        put_state(c_first + c_second);
        lds_barrier();
        if (16 * wave < n - n1) {
            add_state(Hh, Hl, Y2);
#pragma unroll
            for (int vt = 0; vt < 4; ++vt)
                BufRaw<16>::st(__builtin_bit_cast(typename BufRaw<16>::type, Y2[vt]), rsy, y_lane() + 64u * vt, y_row(first + n1));
        }
    }
    if (bail) {
        const float* states = A.seg_ws;
        if constexpr (FOLD) {                        // the chunked kernel's code takes the states that enter the segment from memory
            float* const own = A.seg_own + ((size_t)bh * nseg + seg) * SEG_FLOATS;
#pragma unroll 1
            for (int down = 0; down < 2; ++down) {
                fold_states(down, X);
#pragma unroll
                for (int q = 0; q < 2; ++q) *reinterpret_cast<f32x4v*>(own + down * SEG_STATE + seg_frag(it0, jt0 + q, lane)) = X[q];
            }
            states = A.seg_own;
        }
        __syncthreads();
        fwd_chunk_sequence<IO, WT, W_IS_EW>(reinterpret_cast<FwdLds<VSPLIT>*>(lds), reinterpret_cast<int*>(lds + sizeof(FwdLds<VSPLIT>) * 2), bh, seg,
                                            static_cast<const IO*>(A.r), static_cast<const IO*>(A.k), static_cast<const IO*>(A.v),
                                            static_cast<const WT*>(A.w), A.u, A.y, T, C, A.H, nseg, states, A.seg_flags);
    }
}

}  // namespace wkv6_detail
}  // namespace vrwkv
