// A pre-norm half's first steps on few tokens: LayerNorm, Q-Shift and the token mixes in one launch, inside the block's native call
// (LN kernel and vrwkv_qshift_mix otherwise; their arithmetic, the normalised rows rounded to their type in between).
//
// With a few hundred tokens either is a launch of 3 to 6 us that waits for memory and reductions, not for bandwidth, and takes the
// host as long again.  A workgroup of four waves owns four neighbouring tokens of an image, a wave one of them: its row, the rows one
// step up and down, and, where no other wave has them, one step left and right.  All of a wave's rows are requested at once;
// a neighbour's statistics are formed anew by everyone who reads it (3.5 rows per token), which costs less than a second
// launch up to the size in ln_shift_mix_takes.  A wave per row, lane = 16 bytes of it, as in rowfuse.hip, so sums have the same order.
#include "linear.h"
#include "wave_sum.h"

namespace vrwkv {
namespace {
constexpr int TOK = 4;                                    // tokens, and waves, of a workgroup

struct LsmArgs {
    const void *x, *ln_w, *ln_b;
    const float* mix;
    void *out[3], *ln_out;                                // ln_out: optional, the normalised rows themselves
    int T, C, Hp, Wp, shift, g, head_dim, n_grid;
    float eps;
};

template <typename IO, int VPL, int NMIX>
__global__ __launch_bounds__(TOK * WAVE)
void ln_shift_mix_kernel(LsmArgs A)
{
    constexpr int V = 16 / (int)sizeof(IO), ROWS = 5;     // own, up, down, left, right
    __shared__ nt_u32x4 rows[ROWS][TOK][VPL * WAVE];
    const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int T = A.T, C = A.C, nvec = C / V, t0 = blockIdx.x * TOK, t = t0 + w;
    const size_t base = (size_t)blockIdx.y * T * C;
    const IO* x = (const IO*)A.x + base;
    // the neighbours' tokens; -1: outside the grid, or not this wave's to normalise
    int src[ROWS];
    src[0] = t < T ? t : -1;
    const int y0 = t / A.Wp, x0 = t % A.Wp;
    const bool in = t < A.n_grid;                         // (a class token stands alone)
    src[1] = in && y0 >= A.shift ? t - A.shift * A.Wp : -1;
    src[2] = in && y0 + A.shift < A.Hp ? t + A.shift * A.Wp : -1;
    src[3] = in && x0 >= A.shift ? t - A.shift : -1;
    src[4] = in && x0 + A.shift < A.Wp ? t + A.shift : -1;
    const int left = src[3], right = src[4];
    if (left >= t0) src[3] = -1;                          // another wave's own row
    if (right < t0 + TOK) src[4] = -1;
    nt_u32x4 raw[ROWS][VPL], lw[VPL], lb[VPL];
#pragma unroll
    for (int r = 0; r < ROWS; ++r)
#pragma unroll
        for (int i = 0; i < VPL; ++i) {
            const int vi = lane + WAVE * i;
            raw[r][i] = nt_u32x4{0u, 0u, 0u, 0u};
            if (src[r] >= 0 && vi < nvec) raw[r][i] = load_raw16<false>(x + (size_t)src[r] * C + vi * V);
        }
    float mu[NMIX][VPL][V];
#pragma unroll
    for (int i = 0; i < VPL; ++i) {
        const int vi = lane + WAVE * i;
        lw[i] = lb[i] = nt_u32x4{0u, 0u, 0u, 0u};
        if (vi < nvec) {
            lw[i] = load_raw16<false>((const IO*)A.ln_w + vi * V);
            lb[i] = load_raw16<false>((const IO*)A.ln_b + vi * V);
        }
#pragma unroll
        for (int m = 0; m < NMIX; ++m)
#pragma unroll
            for (int e = 0; e < V; ++e) mu[m][i][e] = vi < nvec ? A.mix[(size_t)m * C + vi * V + e] : 0.f;
    }
#pragma unroll
    for (int r = 0; r < ROWS; ++r) {
        if (src[r] < 0) continue;                         // the whole wave
        float v[VPL][V], s = 0.f, q = 0.f;
#pragma unroll
        for (int i = 0; i < VPL; ++i) {
            widen_raw16<IO, V>(raw[r][i], v[i]);
#pragma unroll
            for (int e = 0; e < V; ++e) s += v[i][e];
        }
        const float mean = wave_sum(s) / (float)C;
#pragma unroll
        for (int i = 0; i < VPL; ++i)
            if (lane + WAVE * i < nvec) {
#pragma unroll
                for (int e = 0; e < V; ++e) { const float d = v[i][e] - mean; q = fmaf(d, d, q); }
            }
        const float rstd = rsqrtf(wave_sum(q) / (float)C + A.eps);
#pragma unroll
        for (int i = 0; i < VPL; ++i) {
            float lnw[V], lnb[V];
            widen_raw16<IO, V>(lw[i], lnw);
            widen_raw16<IO, V>(lb[i], lnb);
            IO n[V];
#pragma unroll
            for (int e = 0; e < V; ++e) n[e] = from_f32<IO>(fmaf((v[i][e] - mean) * rstd, lnw[e], lnb[e]));
            __builtin_memcpy(&raw[r][i], n, 16);
            rows[r][w][lane + WAVE * i] = raw[r][i];
        }
    }
    __syncthreads();
    if (t >= T) return;
#pragma unroll
    for (int i = 0; i < VPL; ++i) {
        const int vi = lane + WAVE * i, c = vi * V;
        if (vi >= nvec) continue;
        const int cq = A.head_dim > 0 ? c % A.head_dim : c;
        const int dir = A.g > 0 && cq < 4 * A.g ? cq / A.g : 4;
        // 0: from the left, 1: from the right, 2: from above, 3: from below, 4 (and class tokens): the token itself
        nt_u32x4 n = raw[0][i];
        bool have = true;
        if (in && dir < 4) {
            const int from = dir == 0 ? left : dir == 1 ? right : dir == 2 ? src[1] : src[2];
            have = from >= 0;
            if (have) {
                if (dir < 2) n = from >= t0 && from < t0 + TOK ? rows[0][from - t0][vi] : rows[dir == 0 ? 3 : 4][w][vi];
                else n = dir == 2 ? raw[1][i] : raw[2][i];
            }
        }
        float xs[V], xx[V];
        widen_raw16<IO, V>(raw[0][i], xs);
        widen_raw16<IO, V>(n, xx);
#pragma unroll
        for (int e = 0; e < V; ++e) xx[e] = have ? xx[e] : 0.f;
        const size_t at = base + (size_t)t * C + c;
        if (A.ln_out) *reinterpret_cast<nt_u32x4*>((IO*)A.ln_out + at) = raw[0][i];
#pragma unroll
        for (int m = 0; m < NMIX; ++m) {
            float o[V];
#pragma unroll
            for (int e = 0; e < V; ++e) o[e] = xs[e] * mu[m][i][e] + xx[e] * (1.f - mu[m][i][e]);
            store_vec<IO, V>((IO*)A.out[m] + at, o);
        }
    }
}

template <typename IO>
void launch(const LsmArgs& a, int n_mix, int B, hipStream_t st) {
    constexpr int V = 16 / (int)sizeof(IO);
    const dim3 grid((a.T + TOK - 1) / TOK, B), block(TOK * WAVE);
    const bool wide = a.C / V > WAVE;
    if (n_mix == 2 && !wide) hipLaunchKernelGGL((ln_shift_mix_kernel<IO, 1, 2>), grid, block, 0, st, a);
    else if (n_mix == 2) hipLaunchKernelGGL((ln_shift_mix_kernel<IO, 2, 2>), grid, block, 0, st, a);
    else if (!wide) hipLaunchKernelGGL((ln_shift_mix_kernel<IO, 1, 3>), grid, block, 0, st, a);
    else hipLaunchKernelGGL((ln_shift_mix_kernel<IO, 2, 3>), grid, block, 0, st, a);
}
}  // namespace

// Rows of up to 128 pieces of 16 bytes, none across a group's border, and few of them.  Twelve bf16 blocks replayed as a graph, separate
// launches / this one, us: 196 x 192 475 / 397, 392 x 192 527 / 447, 784 x 384 830 / 753, 784 x 768 1256 / 1223, 3136 x 192 863 / 833; the
// neighbours' rows cost more than a launch at 6272 x 192 992 / 1049, 1568 x 768 1523 / 1573 (eager), 3136 x 768 1795 / 1980.  VRWKV6 196 x 192
// 912 / 840, 784 x 768 1850 / 1773.
bool ln_shift_mix_takes(int B, int T, int C, int g, int head_dim, int shift, int dtype) {
    const int V = dtype == VRWKV_F32 ? 4 : 8, period = head_dim > 0 ? head_dim : C;
    return C % V == 0 && g % V == 0 && period % V == 0 && C / V <= 2 * WAVE && B <= 65535 && shift >= 0 && (long long)B * T * C <= LN_SHIFT_MIX_MOST;
}

int ln_shift_mix(const void* x, const void* ln_w, const void* ln_b, float eps, const float* mix, void* const* out, int n_mix, void* ln_out,
                 int B, int T, int C, int Hp, int Wp, int shift, int g, int head_dim, int dtype, hipStream_t st) {
    if (n_mix < 2 || n_mix > 3 || (Hp * Wp != T && Hp * Wp != T - 1) || Hp <= 0 || Wp <= 0) {
        set_error("ln_shift_mix: bad sizes (T=%d Hp=%d Wp=%d n_mix=%d)", T, Hp, Wp, n_mix);
        return VRWKV_UNSUPPORTED_SHAPE;
    }
    if (g < 0 || (head_dim > 0 ? C % head_dim || 4 * g > head_dim : 4 * (long long)g > C)) {
        set_error("ln_shift_mix: groups of %d do not fit (C=%d, head_dim=%d)", g, C, head_dim);
        return VRWKV_UNSUPPORTED_SHAPE;
    }
    LsmArgs a{x, ln_w, ln_b, mix, {out[0], out[1], n_mix == 3 ? out[2] : nullptr}, ln_out, T, C, Hp, Wp, shift, g, head_dim, Hp * Wp, eps};
    if (dtype == VRWKV_F32) launch<float>(a, n_mix, B, st);
    else if (dtype == VRWKV_BF16) launch<__hip_bfloat16>(a, n_mix, B, st);
    else launch<__half>(a, n_mix, B, st);
    return check_launch("ln_shift_mix");
}

}  // namespace vrwkv
