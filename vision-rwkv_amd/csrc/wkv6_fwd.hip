// wkv6 forward entry points.
#include "wkv6_fwd_scalar.h"
#include "wkv6_fwd_chunk.h"
#include "wkv6_fwd_tile.h"
#include <algorithm>
#include <cstdlib>
#include <cstring>

using namespace vrwkv;
using namespace vrwkv::wkv6_detail;

namespace {

int validate(int B, int T, int C, int H, int rkv_dtype, int w_dtype) {
    if (B <= 0 || T <= 0 || C <= 0 || H <= 0) {
        set_error("wkv6_fwd: B, T, C, H must be positive (got %d, %d, %d, %d)", B, T, C, H);
        return VRWKV_INVALID_ARG;
    }
    if (C != H * N) {                                   // assert(H*_N_ == C), wkv6_cuda.cu:350
        set_error("wkv6_fwd: C must equal H*64 (got C=%d, H=%d)", C, H);
        return VRWKV_UNSUPPORTED_SHAPE;
    }
    for (int dt : {rkv_dtype, w_dtype})
        if (dt != VRWKV_F32 && dt != VRWKV_BF16 && dt != VRWKV_F16) {
            set_error("wkv6_fwd: unsupported dtype code %d", dt);
            return VRWKV_UNSUPPORTED_DTYPE;
        }
    if (w_dtype != VRWKV_F32 && w_dtype != rkv_dtype) {
        set_error("wkv6_fwd: w must be fp32 or have the dtype of r, k, v");
        return VRWKV_UNSUPPORTED_DTYPE;
    }
    if ((long long)B * T * C >= (1LL << 40) || (long long)B * H > 0x7fffffffLL || (long long)T * C >= (1LL << 29)) {
        set_error("wkv6_fwd: tensor too large");
        return VRWKV_UNSUPPORTED_SHAPE;
    }
    return VRWKV_OK;
}

// Segments per sequence of a call (1: not split); OPT_WKV6_SEGMENTS forces a number (testing).  parts: the tile kernels run them.
int segments(int B, int T, int H, int rkv_dtype, bool& parts) {
    const int nchunk = (T + LC - 1) / LC, forced = option(OPT_WKV6_SEGMENTS);
    if (forced > 0 && (long long)B * H <= SEG_SEQUENCES) {
        const int n = forced < nchunk ? forced : nchunk, cps = (nchunk + n - 1) / n;
        parts = rkv_dtype == VRWKV_BF16 ? cps * LC <= TILE_TOKENS : cps * LC <= PART && (nchunk + cps - 1) / cps <= FOLD_SEGMENTS;
        return (nchunk + cps - 1) / cps;
    }
    parts = false;
    return forced > 0 ? 1 : wkv6_fwd_segments((long long)B * H, nchunk, device_cus(), rkv_dtype, parts);
}
// Segments of one part fold the states themselves where there are few, without a launch that does it first (bf16, 48 sequences of 577 tokens: 29.9 and 26.9
// us), and want room for the result.
bool folds(int T, int nseg, bool parts) { return parts && nseg <= FOLD_SEGMENTS && ((T + LC - 1) / LC + nseg - 1) / nseg * LC <= PART; }
size_t states_bytes(long long sequences, int T, int nseg, bool parts) { return seg_bytes(sequences, nseg, SEG_FLOATS * (folds(T, nseg, parts) ? 2 : 1)); }

template <typename IO, typename WT>
int launch_scalar(const void* r, const void* k, const void* v, const void* w, const float* u, float* y,
                  int B, int T, int C, int H, bool w_is_ew, hipStream_t st) {
    const dim3 grid(B * H), block(256);
    const IO* rr = static_cast<const IO*>(r);
    const IO* kk = static_cast<const IO*>(k);
    const IO* vv = static_cast<const IO*>(v);
    const WT* ww = static_cast<const WT*>(w);
    if (w_is_ew) {
        hipLaunchKernelGGL((wkv6_fwd_scalar_kernel<IO, WT, 1, true>), grid, block, 0, st, rr, kk, vv, ww, u, y, T, C, H);
        hipLaunchKernelGGL((wkv6_fwd_scalar_kernel<IO, WT, 0, true>), grid, block, 0, st, rr, kk, vv, ww, u, y, T, C, H);
    } else {
        hipLaunchKernelGGL((wkv6_fwd_scalar_kernel<IO, WT, 1, false>), grid, block, 0, st, rr, kk, vv, ww, u, y, T, C, H);
        hipLaunchKernelGGL((wkv6_fwd_scalar_kernel<IO, WT, 0, false>), grid, block, 0, st, rr, kk, vv, ww, u, y, T, C, H);
    }
    return check_launch("wkv6_fwd");
}

// Both passes of a (b,h) sequence side by side in one workgroup, out-of-range sequences redone in place by the sequential
// recurrence; few long sequences are cut into segments first (wkv6_segment.h) when the caller's workspace allows it.
template <typename IO, typename WT, bool EW>
int launch_chunked(const void* r, const void* k, const void* v, const void* w, const float* u, float* y, void* ws, size_t ws_bytes,
                   int B, int T, int C, int H, bool whole, hipStream_t st) {
    const dim3 block(64 * FW_WAVES);
    const IO* rr = static_cast<const IO*>(r);
    const IO* kk = static_cast<const IO*>(k);
    const IO* vv = static_cast<const IO*>(v);
    const WT* ww = static_cast<const WT*>(w);
    const long long sequences = (long long)B * H;
    bool parts = false;
    int nseg = whole ? 1 : segments(B, T, H, type_code<IO>, parts);
    // (the state kernels read several elements at a time: 16-bit rows on 4 bytes; wider accesses need no more either)
    const bool cut = !(((uintptr_t)k | (uintptr_t)v | (uintptr_t)w) & 3), loose = !cut || ((uintptr_t)r & 3);
    if (!ws || ws_bytes < states_bytes(sequences, T, nseg, parts) || ((uintptr_t)ws & 15) || !cut) nseg = 1;
    float *states = nullptr, *own = nullptr;
    int* flags = nullptr;
    unsigned grid = (unsigned)sequences;
    if (nseg > 1) {
        states = static_cast<float*>(ws);
        const size_t all = (size_t)sequences * nseg * SEG_FLOATS;
        if (folds(T, nseg, parts)) own = states + all;
        flags = reinterpret_cast<int*>((own ? own : states) + all);
        grid = seg_grid(sequences, nseg);
        if (parts)
            hipLaunchKernelGGL((wkv6_part_state_kernel<IO, WT, EW>), dim3(grid), dim3(64 * PART_WAVES), 0, st, kk, vv, ww, states, flags, T, C, H,
                               sequences, nseg);
        else
            hipLaunchKernelGGL((wkv6_seg_state_kernel<IO, WT, EW>), dim3(grid), dim3(256), 0, st, kk, vv, ww, states, flags, T, C, H, sequences, nseg);
        if (!own) hipLaunchKernelGGL((wkv6_seg_fold_kernel<2, false>), dim3(4, 2, (unsigned)sequences), dim3(256), 0, st, states, nseg);
    }
    // Up to 256 tokens in one or two parts (the tile kernel is ahead of the chunked one at every size measured, 3 to 768 sequences of 33 to 256 tokens in
    // all types: 1.03 to 1.8 times, least where a second part is nearly empty); more tokens uncut, and calls that ask for it (vrwkv_wkv6_fwd_whole),
    // are the chunked kernel's, cut sequences the tile kernel's where their segments are parts.
    const FwdTileArgs tile{r, k, v, w, u, y, T, C, H, (int)sequences, nseg, states, flags, own};
    if (nseg == 1 && T <= TILE_TOKENS && !whole) {
        if constexpr (sizeof(IO) == 2) {
            if (loose) {
                hipLaunchKernelGGL((wkv6_fwd_tile_kernel<IO, WT, EW, 0, true>), dim3(grid), dim3(64 * PART_WAVES), 0, st, tile);
                return check_launch("wkv6_fwd (tile, rows off 4 bytes)");
            }
        }
        hipLaunchKernelGGL((wkv6_fwd_tile_kernel<IO, WT, EW, 0>), dim3(grid), dim3(64 * PART_WAVES), 0, st, tile);
        return check_launch("wkv6_fwd (tile)");
    }
    if (nseg > 1 && parts) {
        auto go = [&](auto segments, auto off) {
            hipLaunchKernelGGL((wkv6_fwd_tile_kernel<IO, WT, EW, decltype(segments)::value, decltype(off)::value>), dim3(grid), dim3(64 * PART_WAVES), 0, st, tile);
        };
        constexpr std::integral_constant<int, 1> folded{};
        constexpr std::integral_constant<int, 2> fold{};
        if constexpr (type_code<IO> == VRWKV_BF16) {                     // (the other types have no segments that do not fold)
            if (!own) {
                if (loose) go(folded, std::true_type{});
                else go(folded, std::false_type{});
                return check_launch("wkv6_fwd (tile, segments)");
            }
        }
        if constexpr (sizeof(IO) == 2) {
            if (loose) {
                go(fold, std::true_type{});
                return check_launch("wkv6_fwd (tile, segments, r off 4 bytes)");
            }
        }
        go(fold, std::false_type{});
        return check_launch("wkv6_fwd (tile, segments)");
    }
    hipLaunchKernelGGL((wkv6_fwd_chunk_kernel<IO, WT, EW>), dim3(grid), block, 0, st, rr, kk, vv, ww, u, y, T, C, H, (int)sequences,
                       nseg, states, flags, nullptr);
    return check_launch("wkv6_fwd (chunked)");
}

bool force_scalar() { return option(OPT_WKV6_FWD_SCALAR) != 0; }   // testing override

template <typename IO, typename WT>
int launch_any(const void* r, const void* k, const void* v, const void* w, const float* u, float* y,
               void* ws, size_t ws_bytes, int B, int T, int C, int H, bool w_is_ew, bool whole, hipStream_t st) {
    if (force_scalar()) return launch_scalar<IO, WT>(r, k, v, w, u, y, B, T, C, H, w_is_ew, st);
    return w_is_ew ? launch_chunked<IO, WT, true>(r, k, v, w, u, y, ws, ws_bytes, B, T, C, H, whole, st)
                   : launch_chunked<IO, WT, false>(r, k, v, w, u, y, ws, ws_bytes, B, T, C, H, whole, st);
}

}  // namespace

extern "C" size_t vrwkv_wkv6_fwd_phases_bytes(int B, int T, int H) {
    if (B <= 0 || T <= 0 || H <= 0) return 0;
    return (size_t)B * H * FW_WAVES * ((T + LC - 1) / LC) * FW_STAMP_POINTS * sizeof(unsigned long long);
}

extern "C" int vrwkv_wkv6_fwd_phases(const void* r, const void* k, const void* v, const void* w, const float* u,
                                     float* y, int B, int T, int C, int H, void* stamps, size_t stamp_bytes,
                                     void* hip_stream) {
    int rc = validate(B, T, C, H, VRWKV_BF16, VRWKV_F32);
    if (rc != VRWKV_OK) return rc;
    if (!r || !k || !v || !w || !u || !y || !stamps) {
        set_error("wkv6_fwd_phases: null pointer argument");
        return VRWKV_INVALID_ARG;
    }
    if ((((uintptr_t)r | (uintptr_t)k | (uintptr_t)v) & 1) || (((uintptr_t)w | (uintptr_t)u | (uintptr_t)y) & 3) ||
        ((uintptr_t)stamps & 7)) {
        set_error("wkv6_fwd_phases: pointers must be aligned to their element size");
        return VRWKV_INVALID_ARG;
    }
    const size_t need = vrwkv_wkv6_fwd_phases_bytes(B, T, H);
    if (stamp_bytes < need) {
        set_error("wkv6_fwd_phases: stamp buffer of %zu bytes required (got %zu)", need, stamp_bytes);
        return VRWKV_WORKSPACE_TOO_SMALL;
    }
    hipLaunchKernelGGL((wkv6_fwd_chunk_kernel<__hip_bfloat16, float, false, true>), dim3(B * H), dim3(64 * FW_WAVES), 0,
                       static_cast<hipStream_t>(hip_stream), static_cast<const __hip_bfloat16*>(r),
                       static_cast<const __hip_bfloat16*>(k), static_cast<const __hip_bfloat16*>(v),
                       static_cast<const float*>(w), u, y, T, C, H, B * H, 1, (const float*)nullptr, (const int*)nullptr,
                       static_cast<unsigned long long*>(stamps));
    return check_launch("wkv6_fwd_phases");
}

extern "C" size_t vrwkv_wkv6_fwd_workspace_bytes(int B, int T, int C, int H) {
    (void)C;
    if (B <= 0 || T <= 0 || H <= 0) return 0;
    // the same for every type: the largest of the plans
    size_t bytes = 0;
    for (int dt : {VRWKV_F32, VRWKV_BF16, VRWKV_F16}) {
        bool parts;
        const int nseg = segments(B, T, H, dt, parts);
        bytes = std::max(bytes, states_bytes((long long)B * H, T, nseg, parts));
    }
    return bytes;
}

namespace vrwkv {
namespace {
int forward(const void* r, const void* k, const void* v, const void* w, const float* u, float* y, int B, int T, int C, int H, int rkv_dtype,
            int w_dtype, int w_is_ew, bool whole, void* workspace, size_t workspace_bytes, void* hip_stream) {
    int rc = validate(B, T, C, H, rkv_dtype, w_dtype);
    if (rc != VRWKV_OK) return rc;
    if (!r || !k || !v || !w || !u || !y) {
        set_error("wkv6_fwd: null pointer argument");
        return VRWKV_INVALID_ARG;
    }
    const size_t esz = rkv_dtype == VRWKV_F32 ? 4 : 2, wsz = w_dtype == VRWKV_F32 ? 4 : 2;
    if ((((uintptr_t)r | (uintptr_t)k | (uintptr_t)v) & (esz - 1)) || ((uintptr_t)w & (wsz - 1)) ||
        (((uintptr_t)u | (uintptr_t)y) & 3)) {
        set_error("wkv6_fwd: pointers must be aligned to their element size");
        return VRWKV_INVALID_ARG;
    }
    hipStream_t st = static_cast<hipStream_t>(hip_stream);
    const bool ew = w_is_ew != 0;
    switch (rkv_dtype) {
        case VRWKV_F32:
            return launch_any<float, float>(r, k, v, w, u, y, workspace, workspace_bytes, B, T, C, H, ew, whole, st);
        case VRWKV_BF16:
            return w_dtype == VRWKV_F32
                       ? launch_any<__hip_bfloat16, float>(r, k, v, w, u, y, workspace, workspace_bytes, B, T, C, H, ew, whole, st)
                       : launch_any<__hip_bfloat16, __hip_bfloat16>(r, k, v, w, u, y, workspace, workspace_bytes, B, T, C, H, ew, whole, st);
        case VRWKV_F16:
            return w_dtype == VRWKV_F32
                       ? launch_any<__half, float>(r, k, v, w, u, y, workspace, workspace_bytes, B, T, C, H, ew, whole, st)
                       : launch_any<__half, __half>(r, k, v, w, u, y, workspace, workspace_bytes, B, T, C, H, ew, whole, st);
    }
    return VRWKV_UNSUPPORTED_DTYPE;
}
}  // namespace
}  // namespace vrwkv

extern "C" int vrwkv_wkv6_fwd(const void* r, const void* k, const void* v, const void* w, const float* u,
                              float* y, int B, int T, int C, int H, int rkv_dtype, int w_dtype, int w_is_ew,
                              void* workspace, size_t workspace_bytes, void* hip_stream) {
    return forward(r, k, v, w, u, y, B, T, C, H, rkv_dtype, w_dtype, w_is_ew, false, workspace, workspace_bytes, hip_stream);
}
extern "C" int vrwkv_wkv6_fwd_whole(const void* r, const void* k, const void* v, const void* w, const float* u, float* y,
                                    int B, int T, int C, int H, int rkv_dtype, int w_dtype, int w_is_ew, void* hip_stream) {
    return forward(r, k, v, w, u, y, B, T, C, H, rkv_dtype, w_dtype, w_is_ew, true, nullptr, 0, hip_stream);
}
