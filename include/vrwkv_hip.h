/* libvrwkv_hip.so -- C ABI of the MI355X (gfx950) WKV operators for Vision-RWKV.
 *
 * Every entry point takes plain device pointers and sizes, enqueues its kernels on the
 * HIP stream it is given (NULL = the default stream), returns without waiting for them,
 * and never allocates or frees device memory: the caller owns every buffer, including
 * the workspace whose size the *_workspace_bytes functions report.  No exception crosses
 * this boundary; a non-zero status comes with a message in vrwkv_last_error().
 *
 * Layouts are the reference's: k, v, y, r, w_raw, gy, g* are (B,T,C) with C fastest and
 * fully contiguous; per-channel parameters are (C,) -- for wkv6, u is (H,N) = (C,) -- fp32.
 */
#ifndef VRWKV_HIP_H
#define VRWKV_HIP_H

#include <stddef.h>

#ifdef __cplusplus
extern "C" {
#endif

/* Status codes.  Replaces TORCH_CHECK / assert at
 * classification/mmcls_custom/models/backbones/cuda_new/bi_wkv.cpp:6-8,
 * .../cuda_new/bi_wkv_kernel.cu:382-384 and .../cuda_v6/wkv6_cuda.cu:350-351. */
enum {
    VRWKV_OK = 0,
    VRWKV_INVALID_ARG = 1,        /* null pointer, non-positive size, misaligned pointer */
    VRWKV_UNSUPPORTED_DTYPE = 2,
    VRWKV_UNSUPPORTED_SHAPE = 3,  /* e.g. C != H*64 for wkv6 */
    VRWKV_LAUNCH_FAILED = 4,      /* hipGetLastError() after a launch */
    VRWKV_WORKSPACE_TOO_SMALL = 5
};

/* Element type of the (B,T,C) tensors. */
enum { VRWKV_F32 = 0, VRWKV_BF16 = 1, VRWKV_F16 = 2 };

int vrwkv_version(void);                 /* major*10000 + minor*100 + patch */
const char* vrwkv_last_error(void);      /* thread-local, never NULL */

/* Tuning / testing switches, process-wide (no counterpart in the reference).  Names: "biwkv_l", "biwkv_s",
 * "biwkv_grid", "biwkv_no_stage", "biwkv_no_resident", "biwkv_bwd_serial", "wkv6_fwd_scalar", "wkv6_bwd_scalar",
 * "wkv6_bwd_unfused" (no effect: the backward is one kernel), "wkv6_segments", "linear_tile", "wgrad_splits", "linear_mix"; 0 = default behaviour.  The initial
 * value of <name> is that of the environment variable VRWKV_<NAME> when the library first looks at any switch; the entry points never read the environment afterwards.
 * vrwkv_set_option rejects (VRWKV_INVALID_ARG) a value the plans would ignore: biwkv_l takes 0, 4, 8, 16, 25, 28 (tokens
 * per wave), biwkv_s 0 or 2..8 (waves per workgroup), biwkv_grid 0 or a positive workgroup count, wkv6_segments 0..64 (segments a sequence
 * is cut into), linear_tile 0, 1, 2, 4, 8 (16 to 128 results on a side), 16 (256 channels wide), wgrad_splits 0 or a positive count of token ranges,
 * linear_mix 0, 1 (norm, shift and mixes inside the projections of a block's halves, VRWKV_UNSUPPORTED_SHAPE where the default would have them in front),
 * 2 (in front), the others 0 or 1. */
int vrwkv_set_option(const char* name, int value);
int vrwkv_get_option(const char* name, int* value);

/* ---- Bi-WKV forward -------------------------------------------------------------------
 * Replaces bi_wkv_forward(w,u,k,v) -> y
 *   (classification/mmcls_custom/models/backbones/cuda_new/bi_wkv.cpp:23-33,
 *    launcher .../cuda_new/bi_wkv_kernel.cu:370-399) and the legacy
 *   forward(B,T,C,w,u,k,v,y) (.../backbones/cuda/wkv_op.cpp:6-8).
 * w, u: (C,) fp32 (already divided by T by the caller, vrwkv.py:183).
 * k, v, y: (B,T,C) of io_dtype; state and arithmetic are fp32.  No T_MAX and no
 * C >= 32 / B*C % 32 restriction; T*C must stay below 2^29 elements.
 * workspace: needed only for long sequences (see vrwkv_biwkv_fwd_workspace_bytes, which
 * returns 0 when none is); may be NULL when that size is 0. */
size_t vrwkv_biwkv_fwd_workspace_bytes(int B, int T, int C, int io_dtype);
int vrwkv_biwkv_fwd(const float* w, const float* u, const void* k, const void* v, void* y,
                    int B, int T, int C, int io_dtype,
                    void* workspace, size_t workspace_bytes, void* hip_stream);

/* Bi-WKV forward with the receptance gate applied before y is stored: y = sigmoid(r) * wkv(w, u, k, v), i.e. the
 * operator plus the step that follows it in VRWKV_SpatialMix.forward when key_norm is off
 * (classification/mmcls_custom/models/backbones/vrwkv.py:183-186: rwkv = RUN_CUDA(...); rwkv = sr * rwkv).  The
 * reference has no such entry (it runs the gate as PyTorch ops on the stored y); this one saves writing y and reading
 * it back.  r: (B,T,C) of the dtype of k, v; every other argument as vrwkv_biwkv_fwd (same workspace).  The gate runs
 * inside the emitting kernel for 16-byte aligned k, v, y with C a multiple of 16 bytes of elements, on the one-launch
 * path (T <= 224) and, for 16-bit rows, the two-launch path; other calls (unaligned rows, fp32 sequences beyond 224
 * tokens, 16-bit sequences of 225..672 tokens, which a kernel without the gate serves) run vrwkv_biwkv_fwd and then
 * gate y in place -- same result, smaller saving.  Forward only. */
int vrwkv_biwkv_fwd_gate(const float* w, const float* u, const void* k, const void* v, const void* r, void* y,
                         int B, int T, int C, int io_dtype,
                         void* workspace, size_t workspace_bytes, void* hip_stream);

/* Bi-WKV forward for callers that cannot allocate device memory (code under HIP graph capture, tight serving loops,
 * harnesses that forbid hipMalloc).  No counterpart in the reference.  Same arguments and results as vrwkv_biwkv_fwd,
 * but the long-sequence workspace is an array built into the library (4 MiB of device memory per GPU, held until the
 * process ends) and the call allocates nothing.  Shapes whose workspace (vrwkv_biwkv_fwd_workspace_bytes) exceeds
 * vrwkv_biwkv_fwd_static_max_workspace_bytes() are rejected with VRWKV_WORKSPACE_TOO_SMALL.  All calls on one GPU
 * share that array: calls that may overlap on a GPU (different streams or threads) race; use vrwkv_biwkv_fwd with
 * separate workspaces for those.  The first call on a device looks up the array's device address (hipGetSymbolAddress,
 * which may load the code object): make it outside a stream capture; every later call only launches kernels. */
size_t vrwkv_biwkv_fwd_static_max_workspace_bytes(void);
int vrwkv_biwkv_fwd_static(const float* w, const float* u, const void* k, const void* v, void* y,
                           int B, int T, int C, int io_dtype, void* hip_stream);

/* ---- Bi-WKV backward ------------------------------------------------------------------
 * Replaces bi_wkv_backward(w,u,k,v,gy) -> [gw,gu,gk,gv]
 *   (classification/mmcls_custom/models/backbones/cuda_new/bi_wkv.cpp:35-47, launcher
 *    .../cuda_new/bi_wkv_kernel.cu:401-443, kernel :119-367) and the legacy
 *   backward(B,T,C,w,u,k,v,gy,gw,gu,gk,gv) (.../backbones/cuda/wkv_op.cpp:9-11).
 * w, u, gw, gu: (C,) fp32, gw and gu already summed over batch and tokens (fully overwritten,
 * no need to zero them); k, v, gy, gk, gv: (B,T,C) of io_dtype.  The workspace (always needed)
 * replaces the three scratch tensors the reference allocates (bi_wkv_kernel.cu:415-417).  A sample's gk and gv do not depend on the
 * others in the call, but for the last bits of fp32 ones of more than 224 tokens. */
size_t vrwkv_biwkv_bwd_workspace_bytes(int B, int T, int C, int io_dtype);
int vrwkv_biwkv_bwd(const float* w, const float* u, const void* k, const void* v, const void* gy,
                    float* gw, float* gu, void* gk, void* gv, int B, int T, int C, int io_dtype,
                    void* workspace, size_t workspace_bytes, void* hip_stream);

/* ---- wkv6 forward (bidirectional RWKV-6 scan) -----------------------------------------
 * Replaces forward(B,T,C,H,r,k,v,w,u,y)
 *   (classification/mmcls_custom/models/backbones/cuda_v6/wkv6_op.cpp:7-9, launcher
 *    .../cuda_v6/wkv6_cuda.cu:348-353, kernel :6-97).
 * r, k, v: (B,T,C) of rkv_dtype; w: (B,T,C) of w_dtype (fp32, or the dtype of r, k, v);
 * u: (H,64) fp32; y: (B,T,C) fp32, caller-allocated, fully overwritten.  C must be H*64.
 * w_is_ew = 0: w is the raw decay logit and the kernel uses d = exp(-exp(w)), i.e. it folds in
 *              the `ew = -exp(w)` of WKV_6.forward (vrwkv6.py:48);
 * w_is_ew = 1: w already holds ew = -exp(w_raw), as the reference extension receives it.
 * State and accumulation are fp32.  No limit on T (T*C < 2^29).  workspace: the size function returns 0 unless the call has
 * few, long sequences, which are then cut into segments that exchange their states through it.  It may be NULL (or too small,
 * or not on 16 bytes) for every call: the sequences then run uncut, as they do when 16-bit k, v or w are not on 4 bytes.  Every
 * tensor: aligned to its elements. */
size_t vrwkv_wkv6_fwd_workspace_bytes(int B, int T, int C, int H);
int vrwkv_wkv6_fwd(const void* r, const void* k, const void* v, const void* w, const float* u,
                   float* y, int B, int T, int C, int H, int rkv_dtype, int w_dtype, int w_is_ew,
                   void* workspace, size_t workspace_bytes, void* hip_stream);
/* The same uncut and 32 tokens at a time at every length: y then has the same bits whatever the number of sequences, and the tokens
 * in front of a position are summed the same way in sequences of any length.  For 16-bit networks in training, which amplify last bits. */
int vrwkv_wkv6_fwd_whole(const void* r, const void* k, const void* v, const void* w, const float* u, float* y,
                         int B, int T, int C, int H, int rkv_dtype, int w_dtype, int w_is_ew, void* hip_stream);

/* Profiling twin of vrwkv_wkv6_fwd_whole (no counterpart in the reference; for benchmarks and tuning): the chunked kernel
 * for bf16 r, k, v and fp32 raw-logit w, with every wave storing the shader clock at the boundaries of its stages.
 * stamps: device buffer of vrwkv_wkv6_fwd_phases_bytes(B, T, H) bytes, laid out as uint64
 * [B*H][8 waves][ceil(T/32) chunk steps][8 points]: 0 element-wise stage entered, 1 its operands written (before the
 * barrier), 2 behind that barrier, 4 matrix stage entered, 5 y stored and the next decay sums formed (before the
 * barrier), 6 behind that barrier; 3 and 7 unused.  Waves 0-3 are the descending pass, 4-7 the ascending one.  y is
 * that of vrwkv_wkv6_fwd_whole bit for bit.  Sequences whose decays fall outside the chunked kernel's range leave later steps
 * unstamped. */
size_t vrwkv_wkv6_fwd_phases_bytes(int B, int T, int H);
int vrwkv_wkv6_fwd_phases(const void* r, const void* k, const void* v, const void* w, const float* u,
                          float* y, int B, int T, int C, int H, void* stamps, size_t stamp_bytes, void* hip_stream);

/* ---- wkv6 backward ---------------------------------------------------------------------
 * Replaces backward(B,T,C,H,r,k,v,w,u,gy,gr,gk,gv,gw,gu)
 *   (classification/mmcls_custom/models/backbones/cuda_v6/wkv6_op.cpp:10-12, launcher
 *    .../cuda_v6/wkv6_cuda.cu:355-362, kernels :99-346), without its T <= 256 limit.
 * r, k, v, w, u as in vrwkv_wkv6_fwd; gy, gr, gk, gv, gw: (B,T,C) fp32, fully overwritten; gw is the
 * gradient w.r.t. the raw decay logit (wkv6_cuda.cu:248,277); gu: (H,64) fp32 already summed over
 * the batch (the reference returns (B,C) and sums in Python, vrwkv6.py:69).  Every tensor aligned to its elements, the
 * workspace to 4 bytes (VRWKV_INVALID_ARG otherwise); sequences run uncut where it is not on 16 bytes, or 16-bit r, k, v or w
 * not on 4. */
size_t vrwkv_wkv6_bwd_workspace_bytes(int B, int T, int C, int H);
int vrwkv_wkv6_bwd(const void* r, const void* k, const void* v, const void* w, const float* u,
                   const float* gy, float* gr, float* gk, float* gv, float* gw, float* gu,
                   int B, int T, int C, int H, int rkv_dtype, int w_dtype, int w_is_ew,
                   void* workspace, size_t workspace_bytes, void* hip_stream);
/* The same with the gradients in their inputs' types: gr, gk, gv of rkv_dtype, gw of w_dtype (rounded once from the fp32
 * sums), as an autograd engine hands them on. */
size_t vrwkv_wkv6_bwd_like_workspace_bytes(int B, int T, int C, int H, int rkv_dtype, int w_dtype);
int vrwkv_wkv6_bwd_like(const void* r, const void* k, const void* v, const void* w, const float* u,
                        const float* gy, void* gr, void* gk, void* gv, void* gw, float* gu,
                        int B, int T, int C, int H, int rkv_dtype, int w_dtype, int w_is_ew,
                        void* workspace, size_t workspace_bytes, void* hip_stream);

/* ---- fused Q-Shift + token mix (the elementwise step in front of the r/k/v projections) -----
 * Replaces q_shift (classification/mmcls_custom/models/backbones/vrwkv.py:68-79) followed by the
 * lerps x*mix_m + q_shift(x)*(1-mix_m) of VRWKV_SpatialMix.jit_func (:160-163, n_mix = 3) and
 * VRWKV_ChannelMix.forward (:248-250, n_mix = 2); with head_dim = 64 the shift is q_shift_multihead
 * (.../vrwkv6.py:75-100).  The reference has no native code for this step (pure PyTorch ops).
 * x, out[m]: (B,T,C) of io_dtype; mix: (n_mix, C) fp32; tokens row-major over the (Hp,Wp) patch
 * grid, T == Hp*Wp or Hp*Wp + 1 (one trailing class token, passed through).
 * quarter_width = int(C*gamma) (head_dim = 0) or head_dim/4 (per-head quarters). */
int vrwkv_qshift_mix(const void* x, const float* mix, void* const* out, int n_mix,
                     int B, int T, int C, int Hp, int Wp, int shift_pixel, int quarter_width,
                     int head_dim, int io_dtype, void* hip_stream);

/* Backward of vrwkv_qshift_mix (the reference differentiates its PyTorch ops by autograd; no native code):
 * gout[m]: gradients of out[m], (B,T,C) of io_dtype; gx: (B,T,C) of io_dtype; gmix: (n_mix, C) fp32, summed over
 * batch and tokens in a fixed order.  workspace: vrwkv_qshift_mix_bwd_workspace_bytes(n_mix, B, T, C) bytes. */
size_t vrwkv_qshift_mix_bwd_workspace_bytes(int n_mix, int B, int T, int C);
int vrwkv_qshift_mix_bwd(const void* x, const float* mix, const void* const* gout, int n_mix,
                         void* gx, float* gmix, int B, int T, int C, int Hp, int Wp, int shift_pixel,
                         int quarter_width, int head_dim, int io_dtype,
                         void* workspace, size_t workspace_bytes, void* hip_stream);

/* ---- fused row-wise epilogues of the blocks (the elementwise steps behind the operator and the GEMMs) ----
 * For every row of N channels:  y = LayerNorm(pre(a)) (weight, bias; LayerNorm skipped when ln_weight is NULL),
 * out = y (post 0) | sigmoid(other) * y (post 1) | other + gamma * y (post 2, gamma NULL = 1); pre 0 = identity,
 * pre 1 = relu(a)^2.  Replaces, in one pass over memory, the PyTorch-op sequences of
 * classification/mmcls_custom/models/backbones/vrwkv.py:184-186 (key_norm, sr * rwkv), :256-261 (relu^2, key_norm,
 * sigmoid gate) and :300-313 (residual with layer scale, post- or pre-norm).  The reference has no native code here.
 * a, other, out: (rows, N) of io_dtype; ln_weight, ln_bias, gamma: (N,) of io_dtype; all 16-byte aligned;
 * N a multiple of the 4 (fp32) or 8 (16-bit) elements in 16 bytes and at most 1024 such vectors. */
int vrwkv_rowfuse(const void* a, const void* other, const void* ln_weight, const void* ln_bias,
                  const void* gamma, void* out, long long rows, int N, int pre, int post, float eps,
                  int io_dtype, void* hip_stream);

/* Backward of vrwkv_rowfuse (the reference differentiates its PyTorch ops by autograd; no native code).
 * gout: gradient of out; ga: gradient of a; gother: gradient of `other` for the sigmoid gate (for the residual it is
 * gout itself and nothing is written; may be NULL then); gparam: (3, N) fp32 = gradients of ln_weight, ln_bias and
 * gamma summed over the rows in a fixed order (required when LayerNorm or gamma take part; rows unused by the call
 * are zero).  With LayerNorm or gamma N is at most 1024.  workspace: vrwkv_rowfuse_bwd_workspace_bytes(rows, N)
 * bytes, needed only when gparam is. */
size_t vrwkv_rowfuse_bwd_workspace_bytes(long long rows, int N);
int vrwkv_rowfuse_bwd(const void* a, const void* other, const void* ln_weight, const void* ln_bias,
                      const void* gamma, const void* gout, void* ga, void* gother, float* gparam,
                      long long rows, int N, int pre, int post, float eps, int io_dtype,
                      void* workspace, size_t workspace_bytes, void* hip_stream);

/* ---- element-wise steps of the VRWKV6 spatial mix (.../backbones/vrwkv6.py:176-212), one pass each ----
 * vrwkv_maa_mix: the five data-dependent token mixes of jit_func (:190-194),
 *   out[i] = x + (sx - x) * (maa[i] + m[i]),  i = w, k, v, r, g;
 *   x, sx (the shifted x), out[i]: (rows, C) of io_dtype; m: (5, rows, C) of io_dtype (the low-rank mix of :183-186);
 *   maa: (5, C) fp32 (time_maa_w, _k, _v, _r, _g).
 * vrwkv_groupnorm_gate: jit_func_2 (:205-211), out = GroupNorm(y) * silu(gate) with groups of `group` consecutive
 *   channels per row (ln_x = GroupNorm(n_head, C) on the (B*T, C) view); y: (rows, C) fp32 (as the operator returns
 *   it) or io_dtype; gate, out: (rows, C), gn_weight, gn_bias: (C,) of io_dtype (fp32, bf16 or fp16; fp32 only beside an fp32 y).
 * All tensors 16-byte aligned, C a multiple of 8 (4 for fp32 maa_mix).  The reference has no native code here. */
int vrwkv_maa_mix(const void* x, const void* sx, const void* m, const float* maa, void* const* out,
                  long long rows, int C, int io_dtype, void* hip_stream);
int vrwkv_groupnorm_gate(const void* y, const void* gate, const void* gn_weight, const void* gn_bias, void* out,
                         long long rows, int C, int group, float eps, int y_dtype, int io_dtype, void* hip_stream);

/* Backward of the two (the reference differentiates its PyTorch ops by autograd; no native code).
 * vrwkv_maa_mix_bwd: gout[i] gradients of out[i]; gx, gsx: (rows, C), gm: (5, rows, C) of io_dtype; gmaa: (5, C) fp32
 *   summed over the rows in a fixed order; workspace vrwkv_maa_mix_bwd_workspace_bytes(rows, C) bytes.
 * vrwkv_groupnorm_gate_bwd: gout gradient of out (io_dtype); gy in y's type, ggate in io_dtype; gparam: (2, C) fp32 =
 *   gradients of gn_weight and gn_bias; C at most 1024; workspace vrwkv_groupnorm_gate_bwd_workspace_bytes(rows, C). */
size_t vrwkv_maa_mix_bwd_workspace_bytes(long long rows, int C);
int vrwkv_maa_mix_bwd(const void* x, const void* sx, const void* m, const float* maa, const void* const* gout,
                      void* gx, void* gsx, void* gm, float* gmaa, long long rows, int C, int io_dtype,
                      void* workspace, size_t workspace_bytes, void* hip_stream);
size_t vrwkv_groupnorm_gate_bwd_workspace_bytes(long long rows, int C);
int vrwkv_groupnorm_gate_bwd(const void* y, const void* gate, const void* gn_weight, const void* gn_bias,
                             const void* gout, void* gy, void* ggate, float* gparam, long long rows, int C, int group,
                             float eps, int y_dtype, int io_dtype, void* workspace, size_t workspace_bytes,
                             void* hip_stream);

/* ---- bicubic resampling of a position table (detection/mmdet_custom/models/utils/embed.py:6-47) ----
 * adjoint 0: src (Hi*Wi, C) -> dst (Ho*Wo, C), cubic convolution (A = -0.75, sample points (o + 0.5) Hi/Ho - 0.5, taps
 * clamped to the border); adjoint 1: src (Ho*Wo, C) = gradient of that result -> dst (Hi*Wi, C).  Row-major tokens, both of
 * `dtype`, fp32 arithmetic.  The reference has no native code here. */
int vrwkv_pos_resize(const void* src, void* dst, int Hi, int Wi, int Ho, int Wo, int C, int adjoint, int dtype,
                     void* hip_stream);

/* ---- inference of one VRWKV / VRWKV6 block on few tokens (.../backbones/vrwkv.py:265-319, vrwkv6.py:288-343) ----
 * x -> out, both (B, T, C) of dtype like every weight; projections (out, in) row-major; C and hidden multiples of 32, hidden <= 8192
 * (fp32: 4096); every pointer 16-byte aligned.  gamma1, gamma2 and the key_norm vectors (*_kn_*) may be NULL.
 * att_mix: (3, C) [VRWKV: k, v, r] or (2, C) [VRWKV6: zeros, 1 - time_maa_x], ffn_mix: (2, C), both fp32 as for vrwkv_qshift_mix.
 * VRWKV (heads = 0): w, u = decay and bonus divided by T, fp32; quarter = width of a shifted channel group.
 * VRWKV6 (heads = C / 64): u (heads, 64) fp32; maa (5, C) fp32; maa_w1 (160, C), maa_w2 (5, C, 32), decay_w1 (64, C) and
 * decay_w2 (C, 64) are the low-rank matrices with the contraction index innermost; att_kn_* are fp32.
 * The reference has no native code here (PyTorch modules around the operator). */
typedef struct vrwkv_block_args {
    const void *x;
    void *out, *workspace;
    size_t workspace_bytes;
    const void *ln1_w, *ln1_b, *ln2_w, *ln2_b, *gamma1, *gamma2;
    const float *att_mix, *ffn_mix, *w, *u;
    const void *key, *value, *receptance, *output, *att_kn_w, *att_kn_b;
    const void *ffn_key, *ffn_receptance, *ffn_value, *ffn_kn_w, *ffn_kn_b;
    const void *gate;
    const float *maa;
    const void *maa_w1, *maa_w2, *decay, *decay_w1, *decay_w2, *gn_w, *gn_b;
    int B, T, C, hidden, heads, Hp, Wp, shift_pixel, quarter, post_norm, dtype;
    float ln1_eps, ln2_eps, att_kn_eps, ffn_kn_eps, gn_eps;
} vrwkv_block_args;
size_t vrwkv_block_fwd_workspace_bytes(int B, int T, int C, int hidden, int heads, int dtype);
int vrwkv_block_fwd(const vrwkv_block_args* args, void* hip_stream);
/* The same for a VRWKV6 block (heads > 0) whose low-rank matrices and vectors lie as the modules hold them: maa_w1 (C, 160), maa_w2
 * (5, 32, C), decay_w1 (C, 64), decay_w2 (64, C) and att_kn_* (C) of `dtype`; maa_x, maa (w, k, v, r, g), ffn_mix_k, ffn_mix_r
 * and u of `dtype`, or fp32 where their bit of fp32_vectors is set (0: maa_x, 1..5: maa, 6: ffn_mix_k, 7: ffn_mix_r, 8: u).
 * Aligned to their elements; every call reads them anew.  The fields of `args` they stand for (att_mix, ffn_mix, u, maa, maa_w1,
 * maa_w2, decay_w1, decay_w2, att_kn_*) are not looked at.  The same workspace. */
typedef struct vrwkv_block6_params {
    const void *maa_w1, *maa_w2, *decay_w1, *decay_w2, *maa_x, *maa[5], *ffn_mix_k, *ffn_mix_r, *u, *att_kn_w, *att_kn_b;
    int fp32_vectors;
} vrwkv_block6_params;
int vrwkv_block6_fwd(const vrwkv_block_args* args, const vrwkv_block6_params* params, void* hip_stream);

/* ---- projections: several products of token matrices with weights in one launch ----
 * out (M, N) = epilogue(a w^T): a (M, K) with rows at pitch lda, w (N, K) row-major, all of `dtype`, fp32 accumulation.  epi: bit 0 relu^2,
 * bit 1 tanh, then, each optional (NULL): * sigmoid(gate) (M, N) (with bit 3: * 2 max(gate, 0), the derivative of relu^2 where gate was its
 * argument), * vec (N) (with bit 2: + vec), + res (M, N).  raw (M, N), optional: the product itself as well;
 * bit 4: the steps see the product rounded to `dtype`, as separate operators would.  1 to 5 problems of the same M; N a multiple of 16, K of 32, lda of 8, every pointer 16-byte aligned.  The reference has no native code here (nn.Linear). */
typedef struct vrwkv_linear {
    const void *a, *w;
    void* out;
    const void *gate, *vec, *res;
    void* raw;
    int N, K, lda, epi;
} vrwkv_linear;
int vrwkv_linear_group(const vrwkv_linear* problems, int n, int M, int dtype, void* hip_stream);
/* dst[i] (cols, rows) = the transpose of src[i] (rows, cols), i < n <= 5, 16-bit elements, rows and cols multiples of 8 up to 65536,
 * 16-byte aligned: the weights as the gradients of the projections' inputs take them. */
int vrwkv_transpose_group(const void* const* src, void* const* dst, const int* rows, const int* cols, int n, void* hip_stream);

/* ---- weight gradients of the projections ----
 * out[z] (O, I) = sum over m of g[z][m][o] x[z][m][i], z < n: rows of g and x at pitches ldg, ldx (elements, multiples of 8),
 * stacks at strides stride_g, stride_x; 16-bit operands and result (dtype), fp32 sums rounded once; O and I multiples of 8,
 * every pointer 16-byte aligned.  workspace: vrwkv_wgrad_workspace_bytes(n, M, O, I) bytes.  The reference has no native code
 * here (autograd of nn.Linear). */
size_t vrwkv_wgrad_workspace_bytes(int n, int M, int O, int I);
int vrwkv_wgrad(const void* g, const void* x, void* out, int n, int M, int O, int I, int ldg, int ldx, long long stride_g,
                long long stride_x, int dtype, void* workspace, size_t workspace_bytes, void* hip_stream);

/* The gradients of 1 to 5 weights over the same M tokens in one launch of 256 x 256 tiles: out[i] (O[i], I[i]) = g[i]^T x[i], rows of g[i]
 * (M, O[i]) and x[i] (M, I[i]) at pitches ldg[i], ldx[i]; as above otherwise.  M pitch < 2^30. */
size_t vrwkv_wgrad_group_workspace_bytes(const int* O, const int* I, int n, int M);
int vrwkv_wgrad_group(const void* const* g, const void* const* x, void* const* out, const int* O, const int* I, const int* ldg, const int* ldx,
                      int n, int M, int dtype, void* workspace, size_t workspace_bytes, void* hip_stream);

/* ---- the Bi-WKV operator with w and u as a model holds them: of wu_dtype (aligned to their elements), times `factor` in that type, rounded
 * to it (1: as they are; 1 / T: the block's division, vrwkv.py:183).  Backward: gw, gu of wu_dtype, rounded from the fp32 sums, then times
 * `factor` and rounded again. ---- */
int vrwkv_biwkv_fwd_as(const void* w, const void* u, int wu_dtype, float factor, const void* k, const void* v, void* y, int B, int T, int C, int io_dtype, void* workspace, size_t workspace_bytes, void* hip_stream);
int vrwkv_biwkv_bwd_as(const void* w, const void* u, int wu_dtype, float factor, const void* k, const void* v, const void* gy, void* gw, void* gu, void* gk, void* gv, int B, int T, int C, int io_dtype, void* workspace, size_t workspace_bytes, void* hip_stream);

/* ---- the same backwards with the gradients of the parameters (gparam; gmix; gparam; gw and gu) in io_dtype, rounded once from
 * the fp32 sums: what autograd asks of a 16-bit model's parameters ---- */
int vrwkv_rowfuse_bwd_like(const void* a, const void* other, const void* ln_weight, const void* ln_bias, const void* gamma, const void* gout, void* ga, void* gother, void* gparam, long long rows, int N, int pre, int post, float eps, int io_dtype, void* workspace, size_t workspace_bytes, void* hip_stream);
int vrwkv_qshift_mix_bwd_like(const void* x, const float* mix, const void* const* gout, int n_mix, void* gx, void* gmix, int B, int T, int C, int Hp, int Wp, int shift_pixel, int quarter_width, int head_dim, int io_dtype, void* workspace, size_t workspace_bytes, void* hip_stream);
/* vrwkv_maa_mix with the low-rank products of vrwkv6.py:183-186 inside: m_i = lo_i w2_i, lo (rows, 5 x 32), w2 (5, 32, C), 16-bit types, C a multiple
 * of 64.  The backward forms m again; gm (5, rows, C) are the gradients of the products.  The token matrices are 16-byte aligned. */
int vrwkv_maa_lora_mix(const void* x, const void* sx, const void* lo, const void* w2, const float* maa, void* const* out, long long rows, int C, int io_dtype, void* hip_stream);
size_t vrwkv_maa_lora_mix_bwd_workspace_bytes(long long rows, int C);
int vrwkv_maa_lora_mix_bwd(const void* x, const void* sx, const void* lo, const void* w2, const float* maa, const void* const* gout, void* gx, void* gsx, void* gm, float* gmaa, long long rows, int C, int io_dtype, void* workspace, size_t workspace_bytes, void* hip_stream);
/* out (C) = the sums over the rows of x (rows, C), both of dtype: fp32 sums in a fixed order, rounded once.  The gradient of a vector that is
 * added to every token.  workspace: vrwkv_column_sums_workspace_bytes(rows, C) bytes. */
size_t vrwkv_column_sums_workspace_bytes(long long rows, int C);
int vrwkv_column_sums(const void* x, void* out, long long rows, int C, int dtype, void* workspace, size_t workspace_bytes, void* hip_stream);
/* With the gradients that x has from elsewhere: add[i] (B, T, C) of io_dtype, i < n_add <= 2, go into gx before it is rounded; gmix of gmix_dtype,
 * fp32 or io_dtype. */
int vrwkv_qshift_mix_bwd_add(const void* x, const float* mix, const void* const* gout, int n_mix, const void* const* add, int n_add, void* gx, void* gmix, int gmix_dtype, int B, int T, int C, int Hp, int Wp, int shift_pixel, int quarter_width, int head_dim, int io_dtype, void* workspace, size_t workspace_bytes, void* hip_stream);
int vrwkv_groupnorm_gate_bwd_like(const void* y, const void* gate, const void* gn_weight, const void* gn_bias, const void* gout, void* gy, void* ggate, void* gparam, long long rows, int C, int group, float eps, int y_dtype, int io_dtype, void* workspace, size_t workspace_bytes, void* hip_stream);
int vrwkv_biwkv_bwd_like(const float* w, const float* u, const void* k, const void* v, const void* gy, void* gw, void* gu, void* gk, void* gv, int B, int T, int C, int io_dtype, void* workspace, size_t workspace_bytes, void* hip_stream);

#ifdef __cplusplus
}
#endif
#endif /* VRWKV_HIP_H */
