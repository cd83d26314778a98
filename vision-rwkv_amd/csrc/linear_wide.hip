// Projections of many tokens on gfx950 matrix cores: out = epilogue(A W^T) for a group of 16-bit problems in one launch of
// persistent workgroups.
//
// A workgroup is eight waves (two per SIMD) on a tile of 32 FM tokens x 256 channels, a wave on 16 FM x 64 of them (FM x 4 products
// of 16 x 16 x 32 per 32 k).  Slices of 64 k of both operands go straight from memory to LDS (whole 128-byte lines: with slices of 32 k,
// which fetch every line twice, 12544 x 3072 x 768 on tiles of 160 tokens in two stages takes 70 us instead of 64), into one of two or three stages; a row's eight
// 16-byte pieces lie rotated by an exclusive-or with the row, so that the fragment reads meet no bank twice (SQ_LDS_BANK_CONFLICT 0).
// The fragments of the next 32 k are read into a second set of registers during the products of the present ones.  A stage is
// refilled behind the barrier in the middle of its slice, when its last fragments are in registers: two half slices ahead
// of their use with two stages, four with three.  The slices of a workgroup's next tile follow those of its present one without a gap,
// so the first loads of a tile pass under the last products and the stores of the one before.  The accumulators are pinned to the
// accumulation registers (left alone the compiler moves them between products and spills addresses into the loop).
//
// What bounds it: with all 256 compute units on it the card lowers its clock (s_memtime against s_memrealtime: 1.5 GHz, 2.1 GHz with
// 147 workgroups) and the matrix pipes are busy four fifths of a tile; the fragment reads take the LDS 704 of the 896 cycles that
// the products of half a slice take it at FM = 7 (four waves of 112 x 128 read a third less, but one wave per SIMD hides less: 62 us
// instead of 54 for three of 12544 x 768 x 768); 2.5 to 3 us go by before a launch's first rows have landed.
//
// A lane ends up with 16 neighbouring channels of a token: the weights are the first operand of a product (result rows = channels),
// and LDS row 16 f + 4 q + e of a wave's 64 channels holds channel 16 q + 4 f + e.
//
// us (M x K x N), this kernel / the library, on the same operands again and again, which the caches then hold | on operands in rotation, more than they hold:
//   three of 12544 x 768 x 768, here one launch  53 / 81 | 57 / 86      three of 9216 x 1024 x 1024  60 / 92 | 66 / 94
//   one                                          22 / 30 | 22 / 29      one                          23 / 31 | 29 / 32
//   12544 x 768 x 3072                           70 / 61 | 71 / 60      9216 x 1024 x 4096           79 / 73 | 85 / 74
//   12544 x 3072 x 768                           51 / 59 | 55 / 63      9216 x 4096 x 1024           66 / 66 | 87 / 70
// In a training step of 64 images of 224 x 224 at 768 channels, between other kernels and with epilogues, three of 12544 x 768 x 768 take 65 to 75, the
// key's product with its two results 106 to 110.  The figures further down are of the first kind.
#include "linear.h"
#include <algorithm>

namespace vrwkv {
namespace {
using gemm::f32x4;
using gemm::u32x4;

constexpr int WM = 2, WN = 4, FN = 4, NT = 64 * WM * WN, TN = WN * FN * 16;
// s_waitcnt for at most `vm` vector memory operations in flight; LDS operations too
constexpr int wait_vm(int vm) { return 0x0F70 | (vm & 15) | (vm >> 4 << 14); }
constexpr int wait_vm_lds(int vm) { return wait_vm(vm) & ~0x0F00; }

__device__ __forceinline__ void load_lds16(__amdgpu_buffer_rsrc_t r, char* lds, unsigned voffset, unsigned soffset) {
    typedef __attribute__((address_space(3))) void* lds_ptr;
    __builtin_amdgcn_raw_ptr_buffer_load_lds(r, (lds_ptr)lds, 16, voffset, soffset, 0, 0);
}

template <typename IO, int FM, int STAGES>
__global__ __launch_bounds__(NT, 2)
void linear_wide_kernel(LinGroup G, int tiles)
{
    constexpr int TM = WM * FM * 16, ROWS = TN + TM, PW = TN * 8 / NT, PER = PW + (TM * 8 + NT - 1) / NT;
    // separate arrays: the compiler lets a read of one pass loads in flight to another
    __shared__ __attribute__((aligned(16))) char L0[ROWS * 128];
    __shared__ __attribute__((aligned(16))) char L1[ROWS * 128];
    __shared__ __attribute__((aligned(16))) char L2[STAGES == 3 ? ROWS * 128 : 16];
    const int tid = threadIdx.x, lane = tid & 63, g4 = lane >> 4, c16 = lane & 15;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), wm = wave / WN, wn = wave % WN;
    const int grid = gridDim.x;
    // the workgroup's tile of a round; an XCD (workgroups are dealt round-robin to the eight) takes a contiguous eighth of it
    auto tile_of = [&](int round) {
        const int base = round * grid, count = min(grid, tiles - base), whole = count / 8 * 8, l = blockIdx.x;
        return l >= count ? tiles : base + (l < whole ? (l & 7) * (whole / 8) + (l >> 3) : l);
    };
    auto locate = [&](int t, int& q, int& m0, int& n0) {
        q = 0;
        while (q + 1 < G.n && t >= G.p[q + 1].tile0) ++q;
        const int nt = (G.p[q].N + TN - 1) / TN, l = t - G.p[q].tile0;
        m0 = l / nt * TM;
        n0 = l % nt * TN;
    };

    // ---- rows on their way: the slices of the workgroup's tiles one after the other
    int lround = 0;
    unsigned ls = 0;                                      // bytes into the rows
    __amdgpu_buffer_rsrc_t rw, ra;
    unsigned vo[PER];                                     // this thread's pieces; rows outside an operand lie outside its descriptor
    // a wave's load i: eight rows.  Where the rows run out the wave repeats its load before, so that every wave counts the same.
    auto instr = [&](int i) { return (i * (NT / 64) + wave < ROWS / 8 ? i : i - 1) * (NT / 64) + wave; };
    auto open = [&]() {
        const int t = tile_of(lround++);
        ls = 0;
        if (t >= tiles) {                                 // nothing follows: the loads stay, at an offset no descriptor reaches
#pragma unroll
            for (int i = 0; i < PER; ++i) vo[i] = OOB_OFFSET;
            return;
        }
        int q, m0, n0;
        locate(t, q, m0, n0);
        const LinProblem& P = G.p[q];
        rw = make_rsrc(P.w, (unsigned)P.N * P.K * 2u);
        ra = make_rsrc(P.a, ((unsigned)(G.M - 1) * P.lda + P.K) * 2u);
        int th = tid;
        asm volatile("" : "+v"(th));                      // formed here, not kept from the kernel's start
#pragma unroll
        for (int i = 0; i < PER; ++i) {
            const int p = instr(i) * 64 + (th & 63), row = p >> 3, piece = (p & 7) ^ (row & 7);
            if (i < PW) {
                const int r = row & 63, channel = (row & ~63) + ((r & 15) >> 2) * 16 + (r >> 4) * 4 + (r & 3);
                vo[i] = (unsigned)(n0 + channel) * P.K * 2u + 16u * piece;
            } else {
                vo[i] = (unsigned)(m0 + row - TN) * P.lda * 2u + 16u * piece;
            }
        }
    };
    auto load = [&](char* L, int i) {
        load_lds16(i < PW ? rw : ra, L + instr(i) * 1024, vo[i], ls);
        if (i == PER - 1) ls += 128;
    };

    // ---- fragments and products
    const unsigned fo[2] = {c16 * 128u + ((g4 ^ (c16 & 7)) << 4), c16 * 128u + (((4 + g4) ^ (c16 & 7)) << 4)};
    const unsigned ow = wn * FN * 2048, oa = TN * 128 + wm * FM * 2048;
    u32x4 fw[2][FN], fa[2][FM];
    f32x4 acc[FM][FN];
    // fragment q of a half slice in the order of need: the channels', then the tokens'
    auto read = [&](const char* L, int half, int q) {
        if (q < FN) fw[half][q] = *reinterpret_cast<const u32x4*>(L + fo[half] + ow + q * 2048);
        else fa[half][q - FN] = *reinterpret_cast<const u32x4*>(L + fo[half] + oa + (q - FN) * 2048);
    };
    // the products of half a slice; the fragments of the next half from `next`, and with `fill` a new slice into `L`
    auto products = [&](auto fill, char* L, const char* next, int half) {
#pragma unroll
        for (int g = 0; g < FM; ++g) {
            if (g < FM - 1) {
#pragma unroll
                for (int q = g * (FM + FN) / (FM - 1); q < (g + 1) * (FM + FN) / (FM - 1); ++q) read(next, half ^ 1, q);
            }
#pragma unroll
            for (int j = 0; j < FN; ++j) {
                acc[g][j] = gemm::mfma16<IO>(fw[half][j], fa[half][g], acc[g][j]);
                asm volatile("" : "+a"(acc[g][j]));
            }
#pragma unroll
            for (int i = 2 * g; i < 2 * g + 2 && i < PER; ++i)
                if (decltype(fill)::value) load(L, i);
            __builtin_amdgcn_sched_barrier(0);
        }
    };

    open();
#pragma unroll
    for (int i = 0; i < PER; ++i) load(L0, i);
#pragma unroll
    for (int i = 0; i < PER; ++i) load(L1, i);
    if constexpr (STAGES == 3) {
#pragma unroll
        for (int i = 0; i < PER; ++i) load(L2, i);
    }
    __builtin_amdgcn_s_waitcnt(wait_vm((STAGES - 1) * PER));
    __builtin_amdgcn_s_barrier();
#pragma unroll
    for (int q = 0; q < FM + FN; ++q) read(L0, 0, q);
    for (int round = 0;; ++round) {
        const int t = tile_of(round);
        if (t >= tiles) break;
        int q, m0, n0;
        locate(t, q, m0, n0);
        const LinProblem& P = G.p[q];
#pragma unroll
        for (int i = 0; i < FM; ++i)
#pragma unroll
            for (int j = 0; j < FN; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
        // One slice: behind the barrier everyone has read all of L, and the next stage has landed.  (After a tile that waits for its
        // stores as well; counting them out measured the same, and nothing then hangs on the order in which loads and stores retire.)
#define SLICE(L, NEXT)                                                                       \
        products(std::false_type{}, L, L, 0);                                                \
        __builtin_amdgcn_s_waitcnt(wait_vm_lds((STAGES - 2) * PER));                         \
        __builtin_amdgcn_s_barrier();                                                        \
        __builtin_amdgcn_sched_barrier(0);                                                   \
        products(std::true_type{}, L, NEXT, 1);
        for (int s = P.K / (64 * STAGES); s > 0; --s) {   // a slice per stage a turn; the last turn's loads are the next tile's
            if (s == 1) open();
            SLICE(L0, L1)
            if constexpr (STAGES == 3) {
                SLICE(L1, L2)
                SLICE(L2, L0)
            } else {
                SLICE(L1, L0)
            }
        }
#undef SLICE
        // the epilogue, a token's sixteen channels as two pieces of eight; outside the result reads give 0 and stores are
        // dropped.  The rows that an epilogue reads are requested a token ahead.
        typedef BufRaw<16>::type piece_t;
        const unsigned bytes = (unsigned)G.M * P.N * 2u;
        const __amdgpu_buffer_rsrc_t ro = make_rsrc(P.out, bytes), rg = make_rsrc(P.gate, bytes), rr = make_rsrc(P.res, bytes), rp = make_rsrc(P.raw, bytes);
        const int n = n0 + 64 * wn + 16 * g4;
        auto at = [&](int i) {
            const int m = m0 + (wm * FM + i) * 16 + c16;
            return m < G.M && n < P.N ? ((unsigned)m * P.N + n) * 2u : OOB_OFFSET;
        };
        auto pack = [](piece_t& p, const float (&v)[8]) {
            IO b[8];
#pragma unroll
            for (int e = 0; e < 8; ++e) b[e] = from_f32<IO>(v[e]);
            __builtin_memcpy(&p, b, 16);
        };
        piece_t gate[2], res[2], vec[2] = {};
        auto fetch = [&](unsigned o) {
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                if (P.gate) gate[h] = BufRaw<16>::ld(rg, o, 16 * h);
                if (P.res) res[h] = BufRaw<16>::ld(rr, o, 16 * h);
            }
        };
        if (P.vec && n < P.N) {
            vec[0] = load_raw16<false>((const IO*)P.vec + n);
            vec[1] = load_raw16<false>((const IO*)P.vec + n + 8);
        }
        fetch(at(0));
#pragma unroll
        for (int i = 0; i < FM; ++i) {
            const unsigned o = at(i);
            piece_t out[2];
#pragma unroll
            for (int j = 0; j < FN; ++j) asm volatile("" : "+a"(acc[i][j]));         // not copied out before its turn
            if (P.raw) {
#pragma unroll
                for (int h = 0; h < 2; ++h) {
                    float v[8];
#pragma unroll
                    for (int e = 0; e < 8; ++e) v[e] = acc[i][2 * h + (e >> 2)][e & 3];
                    pack(out[h], v);
                    BufRaw<16>::st(out[h], rp, o, 16 * h);
                }
            }
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                float v[8], x[8];
#pragma unroll
                for (int e = 0; e < 8; ++e) v[e] = acc[i][2 * h + (e >> 2)][e & 3];
                if (P.epi & EPI_ROUND) {
#pragma unroll
                    for (int e = 0; e < 8; ++e) v[e] = to_f32(from_f32<IO>(v[e]));
                }
                if (P.epi & EPI_RELU_SQ) {
#pragma unroll
                    for (int e = 0; e < 8; ++e) { const float r = fmaxf(v[e], 0.f); v[e] = r * r; }
                }
                if (P.gate) {
                    widen_raw16<IO, 8>(gate[h], x);
#pragma unroll
                    for (int e = 0; e < 8; ++e)
                        v[e] *= P.epi & EPI_RELU_SQ_BWD ? 2.f * fmaxf(x[e], 0.f) : fast_rcp(1.f + fast_exp2(-LOG2E * x[e]));
                }
                if (P.vec) {
                    widen_raw16<IO, 8>(vec[h], x);
#pragma unroll
                    for (int e = 0; e < 8; ++e) v[e] = P.epi & EPI_ADD_VEC ? v[e] + x[e] : v[e] * x[e];
                }
                if (P.res) {
                    widen_raw16<IO, 8>(res[h], x);
#pragma unroll
                    for (int e = 0; e < 8; ++e) v[e] += x[e];
                }
                pack(out[h], v);
            }
            if (i + 1 < FM) fetch(at(i + 1));
#pragma unroll
            for (int h = 0; h < 2; ++h) BufRaw<16>::st(out[h], ro, o, 16 * h);
            __builtin_amdgcn_sched_barrier(0);
        }
    }
    __builtin_amdgcn_s_waitcnt(wait_vm(0));               // nothing may land in LDS once the workgroup has left it
}

// The tile: the taller the less is read per product, but the last round of workgroups should be full; and up to 160 tokens three
// stages fit the LDS, where the contraction is a multiple of three slices, which hide the loads' way better.  A round takes about FM + 0.5
// units with three stages, FM + 1.3 with two.  Measured, us:
//                              FM 4, 5, 6, 7 with two stages   4, 5 with three    rounds
//   12544 x 768 x 768          28   20   22   24               25   21            2 1 1 1
//   three of them              66   59   67   54               60   54            4 3 3 2
//   12544 x 768 x 3072         71   66   71   65               65   66            5 4 4 3
//   12544 x 3072 x 768         106  64   67   73               85   56            2 1 1 1
//   9216 x 1024 x 4096         89   81   74   81                                  5 4 3 3
struct Tile { int fm, stages; };
Tile tile_for(const LinGroup& G, int cus) {
    bool three = true;
    for (int i = 0; i < G.n; ++i) three = three && G.p[i].K % 192 == 0;
    Tile best = {0, 0};
    float least = 0.f;
    for (int fm = 4; fm <= 7; ++fm) {
        const int stages = three && fm <= 5 ? 3 : 2;
        bool fits = true;
        long long tiles = 0;
        for (int i = 0; i < G.n; ++i) {
            fits = fits && G.p[i].K % (64 * stages) == 0;
            tiles += (long long)((G.M + 32 * fm - 1) / (32 * fm)) * ((G.p[i].N + TN - 1) / TN);
        }
        const float cost = (float)((tiles + cus - 1) / cus) * (fm + (stages == 3 ? 0.5f : 1.3f));
        if (fits && (!best.fm || cost < least)) { best = {fm, stages}; least = cost; }
    }
    return best;
}

template <typename IO, int FM, int STAGES>
void launch(LinGroup& G, int cus, hipStream_t st) {
    int tiles = 0;
    for (int i = 0; i < G.n; ++i) {
        G.p[i].tile0 = tiles;
        tiles += ((G.M + 32 * FM - 1) / (32 * FM)) * ((G.p[i].N + TN - 1) / TN);
    }
    hipLaunchKernelGGL((linear_wide_kernel<IO, FM, STAGES>), dim3(std::min(tiles, cus)), dim3(NT), 0, st, G, tiles);
}
template <typename IO>
void launch_tile(LinGroup& G, hipStream_t st) {
    const int cus = device_cus();
    const Tile t = tile_for(G, cus);
    if (t.stages == 3) return t.fm == 4 ? launch<IO, 4, 3>(G, cus, st) : launch<IO, 5, 3>(G, cus, st);
    switch (t.fm) {
    case 4: return launch<IO, 4, 2>(G, cus, st);
    case 5: return launch<IO, 5, 2>(G, cus, st);
    case 6: return launch<IO, 6, 2>(G, cus, st);
    default: return launch<IO, 7, 2>(G, cus, st);
    }
}
// ---- weights with the contraction index innermost, for the gradients of the inputs (g W = g (W^T)^T) ----
// 64 x 64 tiles turned through LDS, 16-byte accesses on either side; one launch for the matrices of a backward (3 x 768 x 768: 4 us).
struct Turn { const void* src[LIN_MAX]; void* dst[LIN_MAX]; int rows[LIN_MAX], cols[LIN_MAX], tile0[LIN_MAX], n; };
__global__ __launch_bounds__(256)
void transpose_kernel(Turn T)
{
    __shared__ unsigned short tile[64][66];               // 33 banks a row: neither direction meets a bank twice
    int q = 0;
    while (q + 1 < T.n && (int)blockIdx.x >= T.tile0[q + 1]) ++q;
    const int rows = T.rows[q], cols = T.cols[q], nc = (cols + 63) / 64, l = blockIdx.x - T.tile0[q], r0 = l / nc * 64, c0 = l % nc * 64;
    const unsigned short* src = (const unsigned short*)T.src[q];
    unsigned short* dst = (unsigned short*)T.dst[q];
    const int x = 8 * (threadIdx.x & 7), y = threadIdx.x >> 3;
#pragma unroll
    for (int i = 0; i < 64; i += 32)
        if (r0 + y + i < rows && c0 + x < cols) {
            const nt_u32x4 v = load_raw16<false>(src + (size_t)(r0 + y + i) * cols + c0 + x);
#pragma unroll
            for (int e = 0; e < 4; ++e) { tile[y + i][x + 2 * e] = (unsigned short)v[e]; tile[y + i][x + 2 * e + 1] = (unsigned short)(v[e] >> 16); }
        }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < 64; i += 32)
        if (c0 + y + i < cols && r0 + x < rows) {
            nt_u32x4 v;
#pragma unroll
            for (int e = 0; e < 4; ++e) v[e] = tile[x + 2 * e][y + i] | (unsigned)tile[x + 2 * e + 1][y + i] << 16;
            *reinterpret_cast<nt_u32x4*>(dst + (size_t)(c0 + y + i) * rows + r0 + x) = v;
        }
}

}  // namespace

// 16-bit problems whose contraction is a whole number of turns of the loop (and whose epilogue is not the low-rank maps' tanh); byte
// offsets are 32 bits wide and leave room for the rows of a tile past the end.
bool wide_takes(const LinGroup& G, int dtype) {
    if (dtype == VRWKV_F32 || G.M <= 0) return false;
    bool two = true, three = true;
    for (int i = 0; i < G.n; ++i) {
        const LinProblem& p = G.p[i];
        if (p.epi & EPI_TANH || p.K <= 0 || p.N <= 0 || p.N % 16 || p.lda < p.K || p.lda % 8 || (G.M + 256LL) * std::max(p.lda, p.N) >= (1LL << 30) ||
            (p.N + 256LL) * p.K >= (1LL << 30))
            return false;
        two = two && p.K % 128 == 0;
        three = three && p.K % 192 == 0;
    }
    return two || three;
}

int wide_group(LinGroup& G, int dtype, hipStream_t st) {
    if (dtype == VRWKV_BF16) launch_tile<__hip_bfloat16>(G, st);
    else launch_tile<__half>(G, st);
    return check_launch("linear_wide");
}

}  // namespace vrwkv

extern "C" int vrwkv_transpose_group(const void* const* src, void* const* dst, const int* rows, const int* cols, int n, void* hip_stream)
{
    using namespace vrwkv;
    if (!src || !dst || !rows || !cols || n <= 0 || n > LIN_MAX) {
        set_error("transpose_group: null argument, or not 1 to %d matrices", LIN_MAX);
        return VRWKV_INVALID_ARG;
    }
    Turn T;
    T.n = n;
    int tiles = 0;
    for (int i = 0; i < n; ++i) {
        if (!src[i] || !dst[i] || (((size_t)src[i] | (size_t)dst[i]) & 15)) {
            set_error("transpose_group: null or misaligned (16 bytes) pointer argument");
            return VRWKV_INVALID_ARG;
        }
        if (rows[i] <= 0 || cols[i] <= 0 || rows[i] % 8 || cols[i] % 8 || rows[i] > 65536 || cols[i] > 65536) {
            set_error("transpose_group: unsupported sizes (%d x %d)", rows[i], cols[i]);
            return VRWKV_UNSUPPORTED_SHAPE;
        }
        T.src[i] = src[i]; T.dst[i] = dst[i]; T.rows[i] = rows[i]; T.cols[i] = cols[i]; T.tile0[i] = tiles;
        tiles += ((rows[i] + 63) / 64) * ((cols[i] + 63) / 64);
    }
    hipLaunchKernelGGL(transpose_kernel, dim3(tiles), dim3(256), 0, static_cast<hipStream_t>(hip_stream), T);
    return check_launch("transpose_group");
}
