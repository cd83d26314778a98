// wkv6 backward for gfx950: gr, gk, gv, gw (B,T,C) and gu (H,64) from gy.
// Replaces backward(B,T,C,H,r,k,v,ew,u,gy,gr,gk,gv,gw,gu)
// (classification/mmcls_custom/models/backbones/cuda_v6/wkv6_op.cpp:10-12, kernels
//  .../cuda_v6/wkv6_cuda.cu:99-346), without its T <= 256 limit (per-thread arrays of length _T_).
//
// The forward is the sum of two causal passes (DIR 0: tokens ascending, with the bonus u; DIR 1:
// descending, no bonus).  In a pass's own token order n, with S_n the state before token n,
//   y_n = r_n (diag(u) k_n v_n^T + S_n),   S_{n+1} = diag(d_n) S_n + k_n v_n^T,  d = exp(ew), ew = -exp(w)
// the gradients are, with the adjoint state G_n = r_n gy_n^T + diag(d_n) G_{n+1}:
//   gr_n[j] = u_j k_n[j] (v_n.gy_n) + (S_n gy_n)[j]
//   gk_n[j] = u_j r_n[j] (v_n.gy_n) + (G_{n+1} v_n)[j]
//   gv_n[i] = sum_j k_n[j] ( u_j r_n[j] gy_n[i] + G_{n+1}[j,i] )
//   gu[j]   = sum_n r_n[j] k_n[j] (v_n.gy_n)
//   gw_n[j] = ew_n[j] * ( sum_{m>n} (a_m[j] - b_m[j]) - b_n[j] ),
//             a_n = r_n[j] (S_n gy_n)[j],  b_n = k_n[j] (G_{n+1} v_n)[j]
// (the last line follows from X_n = sum_i S_n[j,i] G_n[j,i]:  d_n * dL/dd_n = X_n - a_n = X_{n+1} - b_n;
//  gw is the gradient w.r.t. the raw decay logit, as in wkv6_cuda.cu:248,277.)
#include "wkv6_bwd_tile.h"
#include <algorithm>
#include <cstdlib>
#include <type_traits>

namespace vrwkv {
namespace {

using namespace wkv6_detail;

// ---- sequential path: one sweep of one pass per launch ----
template <typename IO, typename WT, int DIR, bool W_IS_EW>
__global__ __launch_bounds__(256)
void wkv6_bwd_seq_s(const IO* r_, const IO* k_, const IO* v_, const WT* w_, const float* u_, const float* gy_,
                    float* gr_, float* a_, float* gu_part, int T, int C, int H) {
    __shared__ __attribute__((aligned(16))) float stage[SEQ_STAGE_FLOATS];
    seq_sweep_s<IO, WT, DIR, W_IS_EW>(blockIdx.x, r_, k_, v_, w_, u_, gy_, gr_, a_, gu_part + (size_t)(blockIdx.x / H) * C + (blockIdx.x % H) * HN, stage, T, C, H);
}
template <typename IO, typename WT, int DIR, bool W_IS_EW>
__global__ __launch_bounds__(256)
void wkv6_bwd_seq_g(const IO* r_, const IO* k_, const IO* v_, const WT* w_, const float* u_, const float* gy_,
                    const float* a_, float* gk_, float* gw_, int T, int C, int H) {
    __shared__ __attribute__((aligned(16))) float stage[SEQ_STAGE_FLOATS];
    seq_sweep_g<IO, WT, DIR, W_IS_EW>(blockIdx.x, r_, k_, v_, w_, u_, gy_, a_, gk_, gw_, stage, T, C, H);
}
template <typename IO, typename WT, int DIR, bool W_IS_EW>
__global__ __launch_bounds__(256)
void wkv6_bwd_seq_v(const IO* r_, const IO* k_, const WT* w_, const float* u_, const float* gy_,
                    float* gv_, int T, int C, int H) {
    __shared__ __attribute__((aligned(16))) float stage[SEQ_STAGE_FLOATS];
    seq_sweep_v<IO, WT, DIR, W_IS_EW>(blockIdx.x, r_, k_, w_, u_, gy_, gv_, stage, T, C, H);
}
// the fp32 sums of the sequential path rounded to 16-bit results
template <typename OT>
__global__ __launch_bounds__(256)
void round_kernel(const float* __restrict__ x, OT* __restrict__ y, size_t n) {
    for (size_t i = (size_t)blockIdx.x * 256 + threadIdx.x; i < n; i += (size_t)gridDim.x * 256) y[i] = from_f32<OT>(x[i]);
}

// Uncut sequences in one or two products (wkv6_bwd_tile.h).  By length and type alone, so that a sample's gradients do not depend on the batch.  Two parts
// are three steps whatever the second one holds, the sweeps a step of two barriers more for every 32 tokens: short ones stay with the sweeps for the calls that
// give every compute unit one to two sequences, where the sweeps run two at a time and the parts one.  us, sweeps -> products, 64 x 12 sequences: of 128 tokens
// bf16 119 -> 71, fp32 126 -> 84; of 196 bf16 195 -> 152, fp16 190 -> 160, fp32 207 -> 186; of 256 bf16 230 -> 164, fp16 224 -> 172, fp32 249 -> 206.  At the
// limits, 3 / 256 / 264 / 512 / 768 sequences: of 160 tokens bf16 60 -> 44, 65 -> 49, 87 -> 87, 92 -> 90, 146 -> 132, fp16 58 -> 45, 64 -> 51, 85 -> 91, 92 -> 94,
// 145 -> 137; of 192 fp32 64 -> 52, 74 -> 63, 98 -> 109, 122 -> 118, 190 -> 175; of 193 fp32 73 -> 55, 83 -> 65, 110 -> 114, 131 -> 124, 204 -> 186.  (257 to 384
// fp32 sequences of 193 to 224 tokens are 1 to 7 % behind the sweeps for it.)
bool bwd_tile_takes(int T, int rkv_dtype) {
    return T <= PART || (T > (rkv_dtype == VRWKV_F32 ? 192 : 160) && T <= BWD_TILE_TOKENS);
}

// Segments per sequence of a call (1: not cut); OPT_WKV6_SEGMENTS forces a number (testing).  parts: of 128 tokens, one part of wkv6_bwd_tile.h each.  Those
// take three launches and BWD_PARTS_US whatever the sequences' number and length, as long as every segment has a compute unit and there are not more than
// sixteen in a sequence (each folds the states of all others); the sweeps are ahead where they find short segments for all of them.  us, sweeps -> parts,
// bf16 / fp32: 48 sequences of 577 tokens 74 -> 43 / 76 -> 51, of 400 80 -> 41 / 82 -> 48, 24 of 1024 85 -> 43 / 90 -> 50, 12 of 1025 78 -> 42 / 81 -> 48 (the
// sweeps' estimate is too low there for fp32 to take it), 24 of 577 59 -> 41 / 61 -> 47 (fp32 likewise), 24 of 300 43 -> 39 / 43 -> 45, 3 of 577 41 -> 39 / 41 -> 44.
constexpr int BWD_TILE_SEGMENTS = 16;
constexpr double BWD_PARTS_US[3] = {59.5, 52., 55.};    // VRWKV_F32, VRWKV_BF16, VRWKV_F16
int segments(int B, int T, int H, int rkv_dtype, bool& parts) {
    const int nchunk = (T + LC - 1) / LC, forced = option(OPT_WKV6_SEGMENTS);
    const long long sequences = (long long)B * H;
    parts = false;
    if (forced > 0 && sequences <= SEG_SEQUENCES) {
        const int n = forced < nchunk ? forced : nchunk, cps = (nchunk + n - 1) / n, nseg = (nchunk + cps - 1) / cps;
        parts = nseg > 1 && nseg <= BWD_TILE_SEGMENTS && cps * LC <= PART;
        return nseg;
    }
    if (forced > 0) return 1;
    double us;
    const int nseg = wkv6_segments(sequences, nchunk, device_cus(), SEG_BWD, us), nparts = (nchunk + PART / LC - 1) / (PART / LC);
    parts = nchunk > 8 && nparts <= BWD_TILE_SEGMENTS && (sequences + 7) / 8 * 8 * nparts <= device_cus() && us > BWD_PARTS_US[rkv_dtype];
    return parts ? nparts : nseg;
}

// Workspace: [fp32 sums gr, gk, gv (16-bit results only)] [gw (16-bit decay logits only)] [a of both passes] [partial gu] [states] [flags]
struct Plan {
    bool out16, w16, parts;
    int nseg;
    size_t n, sums, states, bytes;                       // elements of a tensor; floats in front of `a`; bytes of the state block
};
Plan plan(int B, int T, int C, int H, int rkv_dtype, int w_dtype, int grad_dtypes_of_inputs, bool cut = true) {
    Plan p;
    p.out16 = grad_dtypes_of_inputs && rkv_dtype != VRWKV_F32;
    p.w16 = grad_dtypes_of_inputs && w_dtype != VRWKV_F32;
    p.nseg = 1;
    p.parts = false;
    if (cut) p.nseg = segments(B, T, H, rkv_dtype, p.parts);
    p.n = (size_t)B * T * C;
    p.sums = (p.out16 ? 3 * p.n : 0) + (p.w16 ? p.n : 0);
    p.states = seg_bytes((long long)B * H, p.nseg, BWD_SEG_FLOATS * (p.parts ? 2 : 1));
    p.bytes = ((p.sums + 2 * p.n + (size_t)B * p.nseg * C + 3) & ~(size_t)3) * sizeof(float) + p.states;
    return p;
}

template <typename IO, typename WT, bool EW>
int launch_all(const void* r, const void* k, const void* v, const void* w, const float* u, const float* gy,
               void* gr, void* gk, void* gv, void* gw, float* gu, float* ws, const Plan& p, int B, int T, int C, int H, hipStream_t st) {
    BwdArgs A;
    A.r = r; A.k = k; A.v = v; A.w = w; A.u = u; A.gy = gy;
    A.gr = gr; A.gk = gk; A.gv = gv; A.gw = gw;
    float* q = ws;
    auto take = [&](size_t floats) { float* x = q; q += floats; return x; };
    A.pr = p.out16 ? take(p.n) : static_cast<float*>(gr);
    A.pk = p.out16 ? take(p.n) : static_cast<float*>(gk);
    A.pv = p.out16 ? take(p.n) : static_cast<float*>(gv);
    A.pw = p.w16 ? take(p.n) : static_cast<float*>(gw);
    A.a = take(2 * p.n);
    A.a_size = p.n;
    A.gu_part = take((size_t)B * p.nseg * C);
    q = ws + (((size_t)(q - ws) + 3) & ~(size_t)3);      // states: 16-byte aligned
    // results leave the kernels in pieces of several channels; where 16-bit rows do not lie on 4 bytes, the sums are rounded afterwards
    const bool apart = p.out16 && (((uintptr_t)gr | (uintptr_t)gk | (uintptr_t)gv) & 3), w_apart = p.w16 && ((uintptr_t)gw & 3);
    if (apart) { A.gr = A.pr; A.gk = A.pk; A.gv = A.pv; }
    if (w_apart) A.gw = A.pw;
    A.T = T; A.C = C; A.H = H; A.sequences = B * H; A.nseg = p.nseg; A.out16 = p.out16 && !apart; A.w16 = p.w16 && !w_apart;
    A.seg_ws = q;
    A.seg_own = q + (size_t)A.sequences * p.nseg * BWD_SEG_FLOATS;
    int* flags = reinterpret_cast<int*>(p.parts ? A.seg_own + (A.seg_own - q) : A.seg_own);
    A.seg_flags = flags;
    const IO *rr = static_cast<const IO*>(r), *kk = static_cast<const IO*>(k), *vv = static_cast<const IO*>(v);
    const WT* ww = static_cast<const WT*>(w);
    int part_rows = B;
    const dim3 rg((unsigned)((p.n + 1023) / 1024 < 8192 ? (p.n + 1023) / 1024 : 8192));
    auto round_w = [&]() { hipLaunchKernelGGL((round_kernel<WT>), rg, dim3(256), 0, st, A.pw, static_cast<WT*>(gw), p.n); };
    auto round_rkv = [&]() {
        const dim3 block(256);
        hipLaunchKernelGGL((round_kernel<IO>), rg, block, 0, st, A.pr, static_cast<IO*>(gr), p.n);
        hipLaunchKernelGGL((round_kernel<IO>), rg, block, 0, st, A.pk, static_cast<IO*>(gk), p.n);
        hipLaunchKernelGGL((round_kernel<IO>), rg, block, 0, st, A.pv, static_cast<IO*>(gv), p.n);
    };
    if (!option(OPT_WKV6_BWD_SCALAR)) {                  // the option forces the sequential sweeps (testing)
        unsigned grid = (unsigned)A.sequences;
        if (p.nseg > 1) {
            grid = seg_grid(A.sequences, p.nseg);
            if (p.parts)
                hipLaunchKernelGGL((wkv6_bwd_part_state_kernel<IO, WT, EW>), dim3(grid), dim3(64 * PART_WAVES), 0, st, r, k, v, w, gy, q, flags, T, C, H,
                                   A.sequences, p.nseg);
            else
                hipLaunchKernelGGL((wkv6_bwd_seg_state_kernel<IO, WT, EW>), dim3(grid), dim3(256), 0, st, rr, kk, vv, ww, gy, q, flags, T, C, H,
                               (long long)A.sequences, p.nseg);
            if (!p.parts) hipLaunchKernelGGL((wkv6_seg_fold_kernel<4, true>), dim3(4, 4, (unsigned)A.sequences), dim3(256), 0, st, q, p.nseg);
        }
        if (p.nseg == 1 ? bwd_tile_takes(T, type_code<IO>) : p.parts) {
            bool loose = false;
            if constexpr (sizeof(IO) == 2) {
                loose = (((uintptr_t)r | (uintptr_t)k | (uintptr_t)v | (uintptr_t)w) & 3) != 0;               // (then uncut)
                if (loose) hipLaunchKernelGGL((wkv6_bwd_tile_kernel<IO, WT, EW, false, true>), dim3(grid), dim3(64 * PART_WAVES), 0, st, A);
            }
            if (p.nseg > 1) hipLaunchKernelGGL((wkv6_bwd_tile_kernel<IO, WT, EW, true>), dim3(grid), dim3(64 * PART_WAVES), 0, st, A);
            else if (!loose) hipLaunchKernelGGL((wkv6_bwd_tile_kernel<IO, WT, EW, false>), dim3(grid), dim3(64 * PART_WAVES), 0, st, A);
        } else {
            hipLaunchKernelGGL((wkv6_bwd_sweep_kernel<IO, WT, EW>), dim3(grid), dim3(512), 0, st, A);
        }
        part_rows = B * p.nseg;
        if (apart) round_rkv();
        if (w_apart) round_w();
    } else {
        const dim3 grid(A.sequences), block(256);
        // descending pass first (writes), ascending pass second (accumulates), as in the forward
        hipLaunchKernelGGL((wkv6_bwd_seq_s<IO, WT, 1, EW>), grid, block, 0, st, rr, kk, vv, ww, u, gy, A.pr, A.a, A.gu_part, T, C, H);
        hipLaunchKernelGGL((wkv6_bwd_seq_g<IO, WT, 1, EW>), grid, block, 0, st, rr, kk, vv, ww, u, gy, A.a, A.pk, A.pw, T, C, H);
        hipLaunchKernelGGL((wkv6_bwd_seq_v<IO, WT, 1, EW>), grid, block, 0, st, rr, kk, ww, u, gy, A.pv, T, C, H);
        hipLaunchKernelGGL((wkv6_bwd_seq_s<IO, WT, 0, EW>), grid, block, 0, st, rr, kk, vv, ww, u, gy, A.pr, A.a, A.gu_part, T, C, H);
        hipLaunchKernelGGL((wkv6_bwd_seq_g<IO, WT, 0, EW>), grid, block, 0, st, rr, kk, vv, ww, u, gy, A.a, A.pk, A.pw, T, C, H);
        hipLaunchKernelGGL((wkv6_bwd_seq_v<IO, WT, 0, EW>), grid, block, 0, st, rr, kk, ww, u, gy, A.pv, T, C, H);
        if (p.out16) round_rkv();
        if (p.w16) round_w();
    }
    // torch.sum(gu, 0), vrwkv6.py:69
    launch_batch_sum(A.gu_part, gu, nullptr, SumOut((float*)nullptr), part_rows, C, st);
    return check_launch("wkv6_bwd");
}

int backward(const void* r, const void* k, const void* v, const void* w, const float* u, const float* gy, void* gr, void* gk, void* gv,
             void* gw, float* gu, int B, int T, int C, int H, int rkv_dtype, int w_dtype, int w_is_ew, int like_inputs,
             void* workspace, size_t workspace_bytes, void* hip_stream) {
    if (B <= 0 || T <= 0 || C <= 0 || H <= 0) {
        set_error("wkv6_bwd: B, T, C, H must be positive (got %d, %d, %d, %d)", B, T, C, H);
        return VRWKV_INVALID_ARG;
    }
    if (C != H * HN) {
        set_error("wkv6_bwd: C must equal H*64 (got C=%d, H=%d)", C, H);
        return VRWKV_UNSUPPORTED_SHAPE;
    }
    for (int dt : {rkv_dtype, w_dtype})
        if (dt != VRWKV_F32 && dt != VRWKV_BF16 && dt != VRWKV_F16) {
            set_error("wkv6_bwd: unsupported dtype code %d", dt);
            return VRWKV_UNSUPPORTED_DTYPE;
        }
    if (w_dtype != VRWKV_F32 && w_dtype != rkv_dtype) {
        set_error("wkv6_bwd: w must be fp32 or have the dtype of r, k, v");
        return VRWKV_UNSUPPORTED_DTYPE;
    }
    if (!r || !k || !v || !w || !u || !gy || !gr || !gk || !gv || !gw || !gu) {
        set_error("wkv6_bwd: null pointer argument");
        return VRWKV_INVALID_ARG;
    }
    if ((long long)T * C >= (1LL << 29) || (long long)B * H > 0x7fffffffLL) {
        set_error("wkv6_bwd: tensor too large");
        return VRWKV_UNSUPPORTED_SHAPE;
    }
    const size_t es = rkv_dtype == VRWKV_F32 ? 4 : 2, ws_el = w_dtype == VRWKV_F32 ? 4 : 2;
    if ((((uintptr_t)r | (uintptr_t)k | (uintptr_t)v) & (es - 1)) || ((uintptr_t)w & (ws_el - 1)) ||
        (((uintptr_t)u | (uintptr_t)gy | (uintptr_t)gu | (uintptr_t)workspace) & 3) ||
        (((uintptr_t)gr | (uintptr_t)gk | (uintptr_t)gv) & ((like_inputs ? es : 4) - 1)) || ((uintptr_t)gw & ((like_inputs ? ws_el : 4) - 1))) {
        set_error("wkv6_bwd: pointers must be aligned to their element size, the workspace to 4 bytes");
        return VRWKV_INVALID_ARG;
    }
    // the state kernel reads pairs of elements (4-byte accesses of 16-bit rows) and keeps its states in 16-byte pieces
    const bool cut = !(((uintptr_t)r | (uintptr_t)k | (uintptr_t)v | (uintptr_t)w) & 3) && !((uintptr_t)workspace & 15);
    const Plan p = plan(B, T, C, H, rkv_dtype, w_dtype, like_inputs, cut);
    if (!workspace || workspace_bytes < p.bytes) {
        set_error("wkv6_bwd: workspace of %zu bytes required (got %zu)", p.bytes, workspace ? workspace_bytes : (size_t)0);
        return VRWKV_WORKSPACE_TOO_SMALL;
    }
    hipStream_t st = static_cast<hipStream_t>(hip_stream);
    float* ws = static_cast<float*>(workspace);
    const bool ew = w_is_ew != 0;
#define VRWKV_GO(IO, WT) (ew ? launch_all<IO, WT, true>(r, k, v, w, u, gy, gr, gk, gv, gw, gu, ws, p, B, T, C, H, st) \
                             : launch_all<IO, WT, false>(r, k, v, w, u, gy, gr, gk, gv, gw, gu, ws, p, B, T, C, H, st))
    switch (rkv_dtype) {
        case VRWKV_F32:  return VRWKV_GO(float, float);
        case VRWKV_BF16: return w_dtype == VRWKV_F32 ? VRWKV_GO(__hip_bfloat16, float) : VRWKV_GO(__hip_bfloat16, __hip_bfloat16);
        case VRWKV_F16:  return w_dtype == VRWKV_F32 ? VRWKV_GO(__half, float) : VRWKV_GO(__half, __half);
    }
#undef VRWKV_GO
    return VRWKV_UNSUPPORTED_DTYPE;
}

}  // namespace
}  // namespace vrwkv

using namespace vrwkv;

extern "C" size_t vrwkv_wkv6_bwd_workspace_bytes(int B, int T, int C, int H) {
    if (B <= 0 || T <= 0 || C <= 0 || H <= 0) return 0;
    // the same for every type: the largest of the plans
    size_t bytes = 0;
    for (int dt : {VRWKV_F32, VRWKV_BF16, VRWKV_F16}) bytes = std::max(bytes, plan(B, T, C, H, dt, VRWKV_F32, 0).bytes);
    return bytes;
}
extern "C" size_t vrwkv_wkv6_bwd_like_workspace_bytes(int B, int T, int C, int H, int rkv_dtype, int w_dtype) {
    if (B <= 0 || T <= 0 || C <= 0 || H <= 0) return 0;
    return plan(B, T, C, H, rkv_dtype, w_dtype, 1).bytes;
}

extern "C" int vrwkv_wkv6_bwd(const void* r, const void* k, const void* v, const void* w, const float* u,
                              const float* gy, float* gr, float* gk, float* gv, float* gw, float* gu,
                              int B, int T, int C, int H, int rkv_dtype, int w_dtype, int w_is_ew,
                              void* workspace, size_t workspace_bytes, void* hip_stream) {
    return backward(r, k, v, w, u, gy, gr, gk, gv, gw, gu, B, T, C, H, rkv_dtype, w_dtype, w_is_ew, 0, workspace, workspace_bytes, hip_stream);
}
extern "C" int vrwkv_wkv6_bwd_like(const void* r, const void* k, const void* v, const void* w, const float* u,
                                   const float* gy, void* gr, void* gk, void* gv, void* gw, float* gu,
                                   int B, int T, int C, int H, int rkv_dtype, int w_dtype, int w_is_ew,
                                   void* workspace, size_t workspace_bytes, void* hip_stream) {
    return backward(r, k, v, w, u, gy, gr, gk, gv, gw, gu, B, T, C, H, rkv_dtype, w_dtype, w_is_ew, 1, workspace, workspace_bytes, hip_stream);
}
