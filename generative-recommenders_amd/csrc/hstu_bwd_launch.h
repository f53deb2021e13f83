// Launching the two kernels of the attention's backward (hstu_bwd_kernel.h, hstu_bwd_pp_kernel.h) for an element type; shared by the
// translation units that instantiate them: hstu_bwd_api.hip (bf16 and fp16 gradients), hstu_bwd_f32.hip (fp32 gradients).
#pragma once
#include "hstu_hip.h"

#include <hip/hip_runtime.h>

#include <atomic>

#include "hstu_bwd_kernel.h"
#include "hstu_bwd_pp_kernel.h"

// defined with the forward entry points (hstu_api.hip); internal to the library
extern "C" __attribute__((visibility("hidden"))) int hstu_hip_device_is_gfx950(void);
extern "C" __attribute__((visibility("hidden"))) void hstu_hip_set_last_error(const char* what, int hip_error);

// hstu_bwd_api.hip: checks a call with 16-bit operands, ranks its sequences where that is asked for, and fills `bp`.  `grad_mask`: the bits that the
// strides of dq, dk, dv may not have set (16 bytes in their elements).  `nothing`: there are no rows.
int hstu_bwd_params(const HstuFwdArgs* a, const HstuBwdGrads* g, int64_t grad_mask, hstu::BwdParams& bp, bool& nothing, void* stream);

namespace {

constexpr int kBwdWaves = 4, kBwdTile = 64, kBwdRows = kBwdWaves * 32;
constexpr int kStoredWaves = 8, kStoredRows = kStoredWaves * 32;  // the dQ kernel that reads stored dS

template <class TT, int DQK, int DV, bool STORE>
auto key_stationary_kernel(std::true_type) {
    return hstu::hstu_bwd_dkdv_pp_kernel<TT, DQK, DV, STORE>;
}
template <class TT, int DQK, int DV, bool STORE>
auto key_stationary_kernel(std::false_type) {
    return hstu::hstu_bwd_dkdv_kernel<TT, DQK, DV, kBwdWaves, kBwdTile, STORE>;
}

template <class TT, int DQK, int DV>
auto both_kernel(std::true_type) {
    return hstu::hstu_bwd_dkdv_pp_kernel<TT, DQK, DV, false, true>;
}
template <class TT, int DQK, int DV>
auto both_kernel(std::false_type) {
    return hstu::hstu_bwd_dkdv_kernel<TT, DQK, DV, kBwdWaves, kBwdTile, false>;  // (not launched)
}

// One launch for both kernels' items while few of them leave the chip idle: two latencies become one.  An item of the one launch holds what the larger of the two
// kernels needs: with 128 columns a CU alone, up to 64 columns two or three fit.  `items` is counted from the sizes the host knows (rows / 128 and one more per
// sequence, no more than the grid), as if every XCD had as many as the busiest, since fewer than 8 pairs of sequence and head lie on as many XCDs; `len` is at most twice the
// mean length.  us, two launches / one (a count in front: items):
//   128 columns, len to 128    128 19.5 / 12.4, 332 21.4 / 21.9 (128 of 24 .. 60 rows, 4 heads, 31 / 35)
//                to 256        196 32.3 / 24.6 (256 of 20 .. 250, 1 head, 54 / 64)
//                to 2048       296 94.6 / 84.9, 410 139 / 137; contextual rows, which make dQ's first block of a sequence the longest chain, only while each has a CU, past
//                              1024 rows half of one: 116 111 / 107, 160 139 / 155 (8 of 1000 .. 1200, 2 heads, 168 / 183), 161 (33 of 230 .. 769) 58.1 / 53.4
//                beyond        256 220 / 146, 312 264 / 227, 396 365 / 361, 504 442 / 497, 616 647 / 776; contextual: 4 of 1600 .. 6400, 1 head, 403 / 464, also with a window: 2 of 1557 .. 2595, 648, 146 / 184
//                windows that make the chains as long as one another, of short, of long and of equal sequences: 144 62.9 / 44.0, 176 31.5 / 33.5, 192 62.8 / 67.4, 196 (7 of 749)
//                              31.9 / 34.9, 268 162 / 168; others 269 (58 of 350 .. 584) 50.5 / 43.5
//   64 columns, len to 256     384 36.3 / 28.2, 432 28.4 / 30.8 (128 of 20 .. 250, 4 heads, 52 / 57)
//                beyond        576 409 / 320, 752 205 / 190, 824 689 / 651, 936 1218 / 1363
// Workgroups that find no rows (max_seq_len far above the lengths) cost more than those of the two kernels do.  128 columns: a grid of 960 32.9 / 30.4, 1304 61 / 86, 1760 66 / 92,
// 2160 73 / 93, with such a window 560 63.9 / 68.4, 904 54 / 63; 64 columns: 3744 81 / 58, 5600 31 / 40, 60144 137 / 211.
inline bool one_launch(int dqk, int dv, int64_t batch, int64_t heads, int64_t rows, int64_t max_seq_len, int64_t window, bool contextual, int64_t grid) {
    if (batch <= 0 || heads <= 0) return false;
    const int64_t pairs = batch * heads, upper = heads * (rows / 128 + batch);
    int64_t items = upper < grid ? upper : grid;
    if (pairs < 8) items = items * 8 / pairs;
    const int64_t len = max_seq_len < 2 * rows / batch ? max_seq_len : 2 * rows / batch;
    if (dqk <= 64 && dv <= 64) return grid <= 4096 && items <= (len <= 256 ? 384 : 768);
    if (grid > 1024 || (contextual && max_seq_len > 2048)) return false;
    if (window > 0 && window < len / 2 && (len <= 256 || len > 1400 || 8 * batch * max_seq_len <= 9 * rows)) return items <= 144 && grid <= 512;
    if (contextual && max_seq_len > 768) return items <= (len > 1024 ? 128 : 256);
    if (len <= 256) return items <= (len <= 128 ? 128 : 256);
    return items <= (len <= 2048 ? 512 : 384);
}

template <class TT, int DQK, int DV>
int launch_bwd(const hstu::BwdParams& bp, hipStream_t stream) {
    // three tile slots for the key-stationary kernel, two for the other; + 64: transposing reads of a 16-wide tile's unused half
    constexpr int smem1 = 3 * kBwdTile * (DQK + DV) * 2 + 64;
    constexpr int smem = 2 * kBwdTile * (DQK + DV) * 2 + 64;
    constexpr int smem3 = 3 * kBwdTile * DQK * 2 + kStoredWaves * 3 * 4096;
    // The key-stationary kernel: with two waves per SIMD where a tile copy gives every copying wave something to do and
    // the byte offsets inside a tile of 64 rows fit its 32-bit arithmetic; the one-wave kernel otherwise.
    constexpr bool kPairedDims = DQK >= 32 && DV >= 32;
    auto k1p = key_stationary_kernel<TT, DQK, DV, false>(std::integral_constant<bool, kPairedDims>{});
    auto k1ps = key_stationary_kernel<TT, DQK, DV, true>(std::integral_constant<bool, kPairedDims>{});
    constexpr int smem1p = kPairedDims ? hstu::bwd_pp_lds_bytes<(DQK < 32 ? 32 : DQK), (DV < 32 ? 32 : DV)>() : 0;
    const bool paired = kPairedDims && bp.f.q_rs < (1 << 22) && bp.do_rs < (1 << 22);
    auto k12 = both_kernel<TT, DQK, DV>(std::integral_constant<bool, kPairedDims>{});
    auto k1 = hstu::hstu_bwd_dkdv_kernel<TT, DQK, DV, kBwdWaves, kBwdTile, false>;
    auto k1s = hstu::hstu_bwd_dkdv_kernel<TT, DQK, DV, kBwdWaves, kBwdTile, true>;
    // dQ with 64 columns of q: one workgroup per CU more where that counts.  128 of v: always (512 sequences of 5 .. 120 rows, 8 heads 204 -> 189 us, 16 of 1024 ..
    // 8192, 4 heads 1325 -> 1314).  32 and 64 of v: up to 256 rows, where it is latency (512 of 5 .. 64 rows, 2 heads 29.0 -> 27.8; 8 heads 87 -> 84); longer ones are
    // faster without (64 of 200 .. 2048 rows, 2 heads 212, with it 232).
    auto k2 = hstu::hstu_bwd_dq_kernel<TT, DQK, DV, kBwdWaves, kBwdTile, DQK == 64 && DV == 128>;
    auto k2short = hstu::hstu_bwd_dq_kernel<TT, DQK, DV, kBwdWaves, kBwdTile, DQK == 64 && DV >= 32>;
    auto k3 = hstu::hstu_bwd_dq_stored_kernel<TT, DQK, kStoredWaves, kBwdTile>;
    // (a function attribute belongs to the device it was set on: one flag per device)
    static std::atomic<bool> attr_done[64];
    int dev = -1;
    if (hipGetDevice(&dev) != hipSuccess || dev >= 64) dev = -1;
    if (dev < 0 || !attr_done[dev]) {
        hipError_t e = hipFuncSetAttribute((const void*)k1, hipFuncAttributeMaxDynamicSharedMemorySize, smem1);
        if (e == hipSuccess) e = hipFuncSetAttribute((const void*)k1s, hipFuncAttributeMaxDynamicSharedMemorySize, smem1);
        if (kPairedDims) {
            if (e == hipSuccess) e = hipFuncSetAttribute((const void*)k1p, hipFuncAttributeMaxDynamicSharedMemorySize, smem1p);
            if (e == hipSuccess) e = hipFuncSetAttribute((const void*)k12, hipFuncAttributeMaxDynamicSharedMemorySize, smem1p);
            if (e == hipSuccess) e = hipFuncSetAttribute((const void*)k1ps, hipFuncAttributeMaxDynamicSharedMemorySize, smem1p);
        }
        if (e == hipSuccess) e = hipFuncSetAttribute((const void*)k2, hipFuncAttributeMaxDynamicSharedMemorySize, smem);
        if (e == hipSuccess) e = hipFuncSetAttribute((const void*)k2short, hipFuncAttributeMaxDynamicSharedMemorySize, smem);
        if (e == hipSuccess) e = hipFuncSetAttribute((const void*)k3, hipFuncAttributeMaxDynamicSharedMemorySize, smem3);
        if (e != hipSuccess) {
            hstu_hip_set_last_error("hipFuncSetAttribute", (int)e);
            return HSTU_ERR_LAUNCH;
        }
        if (dev >= 0) attr_done[dev] = true;
    }
    const unsigned grid = (unsigned)bp.f.slots_per_xcd * 8;
    if constexpr (kPairedDims) {
        const bool one = one_launch(DQK, DV, bp.f.B, bp.f.H, bp.total_q, bp.f.max_seq_len, bp.f.w, bp.f.c > 0, grid);
        if (!bp.ds && paired && one) {
            hipLaunchKernelGGL(k12, dim3(grid * 2), dim3(hstu::kBwdPpWaves * 64), smem1p, stream, bp);
            const hipError_t e = hipGetLastError();
            if (e == hipSuccess) return HSTU_OK;
            hstu_hip_set_last_error("backward kernel launch", (int)e);
            return HSTU_ERR_LAUNCH;
        }
    }
    if (bp.ds) {
        if (paired) hipLaunchKernelGGL(k1ps, dim3(grid), dim3(hstu::kBwdPpWaves * 64), smem1p, stream, bp);
        else hipLaunchKernelGGL(k1s, dim3(grid), dim3(kBwdWaves * 64), smem1, stream, bp);
        hstu::BwdParams b3 = bp;  // the same items in blocks of 256 query rows
        b3.f.num_mb = (bp.f.max_seq_len + kStoredRows - 1) / kStoredRows;
        b3.f.slots_per_xcd = bp.f.pairs_per_xcd * b3.f.num_mb;
        hipLaunchKernelGGL(k3, dim3((unsigned)b3.f.slots_per_xcd * 8), dim3(kStoredWaves * 64), smem3, stream, b3);
    } else {
        if (paired) hipLaunchKernelGGL(k1p, dim3(grid), dim3(hstu::kBwdPpWaves * 64), smem1p, stream, bp);
        else hipLaunchKernelGGL(k1, dim3(grid), dim3(kBwdWaves * 64), smem1, stream, bp);
        hipLaunchKernelGGL(bp.f.max_seq_len <= 256 ? k2short : k2, dim3(grid), dim3(kBwdWaves * 64), smem, stream, bp);
    }
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) {
        hstu_hip_set_last_error("backward kernel launch", (int)e);
        return HSTU_ERR_LAUNCH;
    }
    return HSTU_OK;
}

template <class TT, int DQK>
int launch_bwd_dv(const hstu::BwdParams& bp, int dv, hipStream_t stream) {
    switch (dv) {
        case 16: return launch_bwd<TT, DQK, 16>(bp, stream);
        case 32: return launch_bwd<TT, DQK, 32>(bp, stream);
        case 64: return launch_bwd<TT, DQK, 64>(bp, stream);
        case 128: return launch_bwd<TT, DQK, 128>(bp, stream);
        default: return HSTU_ERR_BAD_HEAD_DIM;
    }
}

template <class TT>
int launch_bwd_dim(const hstu::BwdParams& bp, int dqk, int dv, hipStream_t stream) {
    switch (dqk) {
        case 16: return launch_bwd_dv<TT, 16>(bp, dv, stream);
        case 32: return launch_bwd_dv<TT, 32>(bp, dv, stream);
        case 64: return launch_bwd_dv<TT, 64>(bp, dv, stream);
        case 128: return launch_bwd_dv<TT, 128>(bp, dv, stream);
        default: return HSTU_ERR_BAD_HEAD_DIM;
    }
}

}  // namespace
