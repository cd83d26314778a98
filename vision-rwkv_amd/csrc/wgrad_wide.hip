// Weight gradients of several large projections in one launch: out (O, I) = sum over the tokens t of g[t][o] x[t][i], 16-bit operands
// with the tokens as rows, fp32 sums.  256 x 256 tiles of the results, each over a range of the tokens; the fp32 partial sums of the ranges
// are added in a fixed order by a second kernel and rounded once.
//
// A workgroup is eight waves on a tile, a wave on 128 x 64 of it (32 products of 16 x 16 x 32 per 32 tokens), one workgroup per compute
// unit.  Slices of 32 tokens go straight from memory to LDS (512 bytes of a row per operand) into one of four stages, four slices
// ahead; the fragments are read across the rows (ds_read_b64_tr_b16) into a second set of registers during the products of the slice
// before.  The 32-byte pieces of a row lie rotated by an exclusive-or with the row, so that the eight rows that half a wave reads
// across meet no bank twice.  The products' accumulators are pinned to the accumulation registers (see linear_wide.hip).
//
// What bounds it: the partial sums' way out and in.  A chip full of workgroups leaves 64 MB whatever the results' size, so results that
// share a launch share that price.  us for 12544 tokens, here / 128 x 128 tiles one after the other (wgrad.hip) / the library's batched partial
// products in 16 bits and their sums: 768 x 768 36 / 34 / 43, three of them 64 / 110 / 127, four 72 / 148 / 173, 3072 x 768 67 / 93 / 83,
// 3072 x 768 and 768 x 3072 and 768 x 768 137 / 263 / 200, three of 384 x 384 34 / 66 / 109, three of 192 x 192 23 / 50 / 78.
#include "linear.h"
#include <algorithm>

namespace vrwkv {
namespace {
using gemm::f32x4;
using gemm::u32x2;
using gemm::u32x4;

constexpr int WTILE = 256, NT = 512, WN = 4, FM = 8, FN = 4, BK = 32, STAGES = 4;
constexpr int OPERAND = BK * WTILE * 2, STAGE = 2 * OPERAND, PER = STAGE / 1024 / (NT / 64);   // bytes; 1 KB loads of a wave and slice
constexpr int MAXP = 5;
constexpr int wait_vm_lds(int vm) { return 0x0070 | (vm & 15) | (vm >> 4 << 14); }             // vmcnt(vm) lgkmcnt(0)

struct WProblem { const void *g, *x; void* out; int O, I, ldg, ldx, tile0; long long part0, quad0; };
struct WGroup { WProblem p[MAXP]; int n, M, tiles, splits, slices_per; long long quads; };

__device__ __forceinline__ void load_lds16(__amdgpu_buffer_rsrc_t r, char* lds, unsigned voffset, unsigned soffset) {
    typedef __attribute__((address_space(3))) void* lds_ptr;
    __builtin_amdgcn_raw_ptr_buffer_load_lds(r, (lds_ptr)lds, 16, voffset, soffset, 0, 0);
}

template <typename IO>
__global__ __launch_bounds__(NT, 2)
void wgrad_wide_kernel(WGroup G, float* __restrict__ part)
{
    // separate arrays: the compiler lets a read of one pass loads in flight to another
    __shared__ __attribute__((aligned(16))) char L0[STAGE];
    __shared__ __attribute__((aligned(16))) char L1[STAGE];
    __shared__ __attribute__((aligned(16))) char L2[STAGE];
    __shared__ __attribute__((aligned(16))) char L3[STAGE];
    const int tid = threadIdx.x, lane = tid & 63, g4 = lane >> 4, c16 = lane & 15;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), wm = wave / WN, wn = wave % WN;
    // the tiles of a token range, which read the same rows, on one XCD as far as the count allows
    int id = blockIdx.x;
    const int whole = G.tiles * G.splits / 8 * 8;
    if (id < whole) id = (id & 7) * (whole / 8) + (id >> 3);
    const int split = id / G.tiles, t = id % G.tiles;
    int q = 0;
    while (q + 1 < G.n && t >= G.p[q + 1].tile0) ++q;
    const WProblem& P = G.p[q];
    const int ti = (P.I + WTILE - 1) / WTILE, l = t - P.tile0, o0 = l / ti * WTILE, i0 = l % ti * WTILE;
    // whole slices [s0, s1); the last range also takes the tokens past the last whole slice
    const int all = G.M / BK, s0 = split * G.slices_per, s1 = min(all, s0 + G.slices_per);
    const int tail = split == G.splits - 1 ? G.M - all * BK : 0;
    const int n = max(0, s1 - s0) + (tail ? 1 : 0), pad = (STAGES - n % STAGES) % STAGES + (tail ? 1 : 0);
    // The turns of the loop are whole ones: zeros fill up in front, and the tail's rows, padded with zeros, come last of those.

    const __amdgpu_buffer_rsrc_t rg = make_rsrc(P.g, ((unsigned)(G.M - 1) * P.ldg + P.O) * 2u), rx = make_rsrc(P.x, ((unsigned)(G.M - 1) * P.ldx + P.I) * 2u);
    unsigned vo[PER];                                     // columns outside an operand are requested where no descriptor reaches
#pragma unroll
    for (int i = 0; i < PER; ++i) {
        const int p = (i * 8 + wave) * 64 + lane, row = p >> 5 & (BK - 1), piece = p & 31, c = 8 * (piece ^ ((row & 7) << 1));
        if (i < PER / 2) vo[i] = o0 + c < P.O ? ((unsigned)row * P.ldg + o0 + c) * 2u : OOB_OFFSET;
        else vo[i] = i0 + c < P.I ? ((unsigned)row * P.ldx + i0 + c) * 2u : OOB_OFFSET;
    }
    unsigned sg = (unsigned)s0 * BK * P.ldg * 2u, sx = (unsigned)s0 * BK * P.ldx * 2u;
    const unsigned stepg = BK * 2u * P.ldg, stepx = BK * 2u * P.ldx;
    auto load = [&](char* L, int i) {
        load_lds16(i < PER / 2 ? rg : rx, L + (i * 8 + wave) * 1024, vo[i], i < PER / 2 ? sg : sx);
        if (i == PER - 1) { sg += stepg; sx += stepx; }
    };
    auto fill = [&](char* L, int stage) {
        if (stage >= pad) {
#pragma unroll
            for (int i = 0; i < PER; ++i) load(L, i);
            return;
        }
        const int rows = tail && stage == pad - 1 ? tail : 0;
#pragma unroll
        for (int i = 0; i < PER; ++i) {
            const int p = (i * 8 + wave) * 64 + lane, row = p >> 5 & (BK - 1), piece = p & 31, c = 8 * (piece ^ ((row & 7) << 1));
            const size_t m = (size_t)all * BK + row;
            u32x4 v = {0u, 0u, 0u, 0u};
            if (row < rows) {
                if (i < PER / 2) { if (o0 + c < P.O) v = load_raw16<false>((const IO*)P.g + m * P.ldg + o0 + c); }
                else if (i0 + c < P.I) v = load_raw16<false>((const IO*)P.x + m * P.ldx + i0 + c);
            }
            *reinterpret_cast<u32x4*>(L + p * 16) = v;
        }
    };

    // fragment of sixteen columns: lane group g4 takes the tokens 4 g4 .. and 16 + 4 g4 .., the same for both operands.  Piece q of row r
    // lies at (q ^ (r & 7)) 32 bytes into the row: an exclusive-or of the whole address.
    const int row = 4 * g4 + (c16 >> 2);
    const unsigned at = row * (2 * WTILE) + ((row & 7) << 5) + 8 * (c16 & 3);
    auto frag = [&](const char* L, unsigned a, int piece) -> u32x4 {
        typedef short s16x4 __attribute__((ext_vector_type(4)));
        typedef __attribute__((address_space(3))) s16x4 lds_s16x4;
        const char* p = L + (a ^ (unsigned)(piece << 5));
        const u32x2 lo = __builtin_bit_cast(u32x2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4*)p));
        const u32x2 hi = __builtin_bit_cast(u32x2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4*)(p + 16 * 2 * WTILE)));
        return u32x4{lo[0], lo[1], hi[0], hi[1]};
    };
    // the first two fragments of g are read over their own registers, once their products are issued; the others into a second set
    constexpr int ONE = 2;
    u32x4 fx[2][FN], f0[ONE], fg[2][FM - ONE];
    f32x4 acc[FM][FN];
    const unsigned atx = at ^ (wn * FN << 5), atg = at ^ (wm * FM << 5);
    auto read = [&](const char* L, int b, int k) {        // in the order of need
        unsigned a = k < FN ? atx : atg;
        asm volatile("" : "+v"(a));                       // addresses formed where they are used: twelve kept ones are spilled
        if (k < FN) fx[b][k] = frag(L + OPERAND, a, k);
        else if (k < FN + ONE) f0[k - FN] = frag(L, a, k - FN);
        else fg[b][k - FN - ONE] = frag(L, a, k - FN);
    };
    auto products = [&](char* L, const char* next, int b) {
#pragma unroll
        for (int i = 0; i < FM; ++i) {
#pragma unroll
            for (int j = 0; j < FN; ++j) {                // x first: a lane holds four neighbouring columns of a row
                acc[i][j] = gemm::mfma16<IO>(fx[b][j], i < ONE ? f0[i < ONE ? i : 0] : fg[b][i < ONE ? 0 : i - ONE], acc[i][j]);
                asm volatile("" : "+a"(acc[i][j]));
            }
            if (i < FM - 1) {                             // two fragments a group, those whose registers are free
                if (i < ONE) read(next, b ^ 1, FN + i);
#pragma unroll
                for (int k = i * (FM + FN - ONE) / (FM - 1); k < (i + 1) * (FM + FN - ONE) / (FM - 1); ++k) read(next, b ^ 1, k < FN ? k : k + ONE);
            }
            if (i < PER) load(L, i);
            __builtin_amdgcn_sched_barrier(0);
        }
    };
#pragma unroll
    for (int i = 0; i < FM; ++i)
#pragma unroll
        for (int j = 0; j < FN; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
    fill(L0, 0);
    fill(L1, 1);
    fill(L2, 2);
    fill(L3, 3);
    __builtin_amdgcn_s_waitcnt(wait_vm_lds(3 * PER));
    __builtin_amdgcn_s_barrier();
#pragma unroll
    for (int k = 0; k < FM + FN; ++k) read(L0, 0, k);
    // One slice: its fragments are in registers, so its stage is free behind the barrier; the next slice has landed, two are on their way
#define SLICE(L, NEXT, b)                                                                    \
        __builtin_amdgcn_s_waitcnt(wait_vm_lds(2 * PER));                                    \
        __builtin_amdgcn_s_barrier();                                                        \
        __builtin_amdgcn_sched_barrier(0);                                                   \
        products(L, NEXT, b);
    for (int turn = (n + STAGES - 1) / STAGES; turn > 0; --turn) {
        if (turn == 1) {                                  // nothing follows: the loads stay, for the counts' sake
#pragma unroll
            for (int i = 0; i < PER; ++i) vo[i] = OOB_OFFSET;
        }
        SLICE(L0, L1, 0)
        SLICE(L1, L2, 1)
        SLICE(L2, L3, 0)
        SLICE(L3, L0, 1)
    }
#undef SLICE
    float* out = part + (size_t)split * 4 * G.quads + P.part0;
#pragma unroll
    for (int i = 0; i < FM; ++i)
#pragma unroll
        for (int j = 0; j < FN; ++j) {
            const int r = o0 + 128 * wm + 16 * i + c16, c = i0 + 64 * wn + 16 * j + 4 * g4;
            if (r < P.O && c < P.I) *reinterpret_cast<f32x4*>(out + (size_t)r * P.I + c) = acc[i][j];
        }
    __builtin_amdgcn_s_waitcnt(wait_vm_lds(0));           // nothing may land in LDS once the workgroup has left it
}

// The ranges in order; one thread per four neighbouring values, eight ranges' loads in flight.
template <typename IO>
__global__ __launch_bounds__(256)
void wgrad_wide_sum_kernel(WGroup G, const float* __restrict__ part)
{
    const long long k = (long long)blockIdx.x * 256 + threadIdx.x;
    if (k >= G.quads) return;
    int q = 0;
    while (q + 1 < G.n && k >= G.p[q + 1].quad0) ++q;
    const f32x4* p = reinterpret_cast<const f32x4*>(part) + k;
    f32x4 s = {0.f, 0.f, 0.f, 0.f};
    constexpr int U = 8;
    for (int i = 0; i < G.splits; i += U) {
        f32x4 v[U];
#pragma unroll
        for (int j = 0; j < U; ++j) v[j] = i + j < G.splits ? p[(size_t)(i + j) * G.quads] : f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int j = 0; j < U; ++j) s += v[j];
    }
    const float r[4] = {s[0], s[1], s[2], s[3]};
    store_vec<IO, 4>((IO*)G.p[q].out + 4 * (k - G.p[q].quad0), r);
}

// Tiles of all problems, and token ranges of whole turns: a round of workgroups costs its slices (0.62 us each) and 5 us, a range more the partial
// sums' way out and in at 5 TB/s.
bool plan(WGroup& G, const int* O, const int* I, int n, int M) {
    if (n <= 0 || n > MAXP || M <= 0) return false;
    G.n = n;
    G.M = M;
    G.tiles = 0;
    G.quads = 0;
    for (int i = 0; i < n; ++i) {
        if (O[i] <= 0 || I[i] <= 0 || O[i] % 8 || I[i] % 8 || O[i] > 65536 || I[i] > 65536 || (long long)O[i] * I[i] > (1LL << 28)) return false;
        G.p[i].O = O[i];
        G.p[i].I = I[i];
        G.p[i].tile0 = G.tiles;
        G.p[i].quad0 = G.quads;
        G.p[i].part0 = 4 * G.quads;
        G.tiles += ((O[i] + WTILE - 1) / WTILE) * ((I[i] + WTILE - 1) / WTILE);
        G.quads += (long long)O[i] * I[i] / 4;
    }
    const int slices = std::max(1, M / BK), forced = option(OPT_WGRAD_SPLITS), cus = device_cus();
    auto cut = [&](int ranges) {
        G.slices_per = ((slices + ranges - 1) / ranges + STAGES - 1) / STAGES * STAGES;
        G.splits = (slices + G.slices_per - 1) / G.slices_per;
    };
    if (forced) { cut(forced); return true; }
    int best = 1;
    double least = 0.;
    for (int ranges = 1; ranges == 1 || (ranges <= 64 && (long long)G.tiles * ranges <= 4LL * cus); ++ranges) {
        cut(ranges);
        const long long rounds = ((long long)G.tiles * G.splits + cus - 1) / cus;
        const double cost = (double)rounds * (0.62 * G.slices_per + 5.) + (double)G.splits * G.quads * 32. / 5e6;
        if (ranges == 1 || cost < least) { best = ranges; least = cost; }
    }
    cut(best);
    return true;
}
}  // namespace
}  // namespace vrwkv

extern "C" size_t vrwkv_wgrad_group_workspace_bytes(const int* O, const int* I, int n, int M)
{
    vrwkv::WGroup G;
    return O && I && vrwkv::plan(G, O, I, n, M) ? (size_t)G.splits * G.quads * 16 : 0;
}

extern "C" int vrwkv_wgrad_group(const void* const* g, const void* const* x, void* const* out, const int* O, const int* I, const int* ldg, const int* ldx,
                                 int n, int M, int dtype, void* workspace, size_t workspace_bytes, void* hip_stream)
{
    using namespace vrwkv;
    if (!g || !x || !out || !O || !I || !ldg || !ldx || !workspace || ((size_t)workspace & 15) || n <= 0 || n > MAXP) {
        set_error("wgrad_group: null or misaligned argument, or not 1 to %d problems", MAXP);
        return VRWKV_INVALID_ARG;
    }
    WGroup G;
    if (!plan(G, O, I, n, M)) {
        set_error("wgrad_group: unsupported sizes (M=%d O=%d I=%d)", M, O[0], I[0]);
        return VRWKV_UNSUPPORTED_SHAPE;
    }
    for (int i = 0; i < n; ++i) {
        if (!g[i] || !x[i] || !out[i] || (((size_t)g[i] | (size_t)x[i] | (size_t)out[i]) & 15)) {
            set_error("wgrad_group: null or misaligned (16 bytes) pointer argument");
            return VRWKV_INVALID_ARG;
        }
        if (ldg[i] < O[i] || ldx[i] < I[i] || ldg[i] % 8 || ldx[i] % 8 || (M + 256LL) * ldg[i] >= (1LL << 30) || (M + 256LL) * ldx[i] >= (1LL << 30)) {
            set_error("wgrad_group: unsupported sizes (M=%d O=%d I=%d ldg=%d ldx=%d)", M, O[i], I[i], ldg[i], ldx[i]);
            return VRWKV_UNSUPPORTED_SHAPE;
        }
        G.p[i].g = g[i];
        G.p[i].x = x[i];
        G.p[i].out = out[i];
        G.p[i].ldg = ldg[i];
        G.p[i].ldx = ldx[i];
    }
    if (dtype != VRWKV_BF16 && dtype != VRWKV_F16) {
        set_error("wgrad_group: dtype must be bf16 or fp16");
        return VRWKV_UNSUPPORTED_DTYPE;
    }
    if (workspace_bytes < (size_t)G.splits * G.quads * 16) {
        set_error("wgrad_group: workspace of %zu bytes is too small", workspace_bytes);
        return VRWKV_WORKSPACE_TOO_SMALL;
    }
    hipStream_t st = static_cast<hipStream_t>(hip_stream);
    const dim3 grid(G.tiles * G.splits), sums((unsigned)((G.quads + 255) / 256));
    if (dtype == VRWKV_BF16) {
        hipLaunchKernelGGL((wgrad_wide_kernel<__hip_bfloat16>), grid, dim3(NT), 0, st, G, (float*)workspace);
        hipLaunchKernelGGL((wgrad_wide_sum_kernel<__hip_bfloat16>), sums, dim3(256), 0, st, G, (const float*)workspace);
    } else {
        hipLaunchKernelGGL((wgrad_wide_kernel<__half>), grid, dim3(NT), 0, st, G, (float*)workspace);
        hipLaunchKernelGGL((wgrad_wide_sum_kernel<__half>), sums, dim3(256), 0, st, G, (const float*)workspace);
    }
    return check_launch("wgrad_group");
}
