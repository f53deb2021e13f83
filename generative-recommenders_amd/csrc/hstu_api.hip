// C ABI of libhstu_hip.so: argument validation, kernel selection and launch.
// Declarations and the reference interfaces they replace are in include/hstu_hip.h.
#include "hstu_hip.h"

#include <hip/hip_runtime.h>

#include <atomic>
#include <cstdio>
#include <cstring>
#include <initializer_list>
#include <mutex>

#include "hstu_fwd_kernel.h"
#include "hstu_fwd_pp_kernel.h"
#include "hstu_fwd_stream_kernel.h"
#include "hstu_jagged_kernels.h"

// Scratch area of hstu_hip_mha_fwd_noalloc: what the caller's `workspace` is to hstu_hip_mha_fwd (work-item counters,
// sequence ranking, work lists, partial sums of a kv-split), held by every device the library is loaded on until the
// process ends.  In host code this name is only a handle for hipGetSymbolAddress: the device address it yields (one
// per device) is what kernels and copies are given.  Its size, HSTU_NOALLOC_SCRATCH_BYTES, is part of the interface.
static __device__ __align__(256) unsigned char scratch[HSTU_NOALLOC_SCRATCH_BYTES];

namespace hstu {

// Work done ahead of the forward kernel, in the caller's workspace (either part may be absent):
// * order[rank] = sequence index, longest sequence first (ties by index).  One wave per sequence: its lanes share
//   out the other sequences and count, by ballot, those that precede it.
// * queue[16 * xcd] = first work item the persistent workgroups of that XCD have not taken statically.
__global__ __launch_bounds__(256) void hstu_prep_kernel(const void* offsets, int offsets_i64, int B, int* order, int* queue,
                                                        int queue_start) {
    if (queue && blockIdx.x == 0 && threadIdx.x < 8) queue[threadIdx.x * 16] = queue_start;
    if (!order) return;
    auto len = [&](int j) -> long long {
        return offsets_i64 ? ((const long long*)offsets)[j + 1] - ((const long long*)offsets)[j]
                           : (long long)(((const int*)offsets)[j + 1] - ((const int*)offsets)[j]);
    };
    const int i = (blockIdx.x * 256 + threadIdx.x) >> 6;  // wave-uniform
    const int lane = threadIdx.x & 63;
    if (i >= B) return;
    const long long ni = len(i);
    int rank = 0;
    for (int j0 = 0; j0 < B; j0 += 64) {
        const int j = j0 + lane;
        bool before = false;
        if (j < B) {
            const long long nj = len(j);
            before = (nj > ni) || (nj == ni && j < i);
        }
        rank += __popcll(__ballot(before));
    }
    if (lane == 0) order[rank] = i;
}

// The caller contract checked on the device: report[0] = number of sequences that break it, report[1] = the first
// such sequence, report[2] = what it breaks (bit 0: offsets decrease, 1: longer than max_seq_len, 2: num_targets outside
// [0, length], 3: fewer non-target positions than contextual_seq_len, 4: shorter than delta_size), report[3] = 1 if
// seq_offsets[0] != 0 or seq_offsets[batch] != total_kv.  One thread per sequence.
__global__ __launch_bounds__(256) void hstu_check_contract_kernel(const void* offsets, int offsets_i64, const void* targets, int targets_i64,
                                                                   int B, long long total_kv, int max_seq_len, int c, int delta,
                                                                   int* report) {
    auto off = [&](int j) -> long long { return offsets_i64 ? ((const long long*)offsets)[j] : (long long)((const int*)offsets)[j]; };
    const int b = blockIdx.x * 256 + threadIdx.x;
    if (b == 0 && (off(0) != 0 || off(B) != total_kv)) report[3] = 1;
    if (b >= B) return;
    const long long n = off(b + 1) - off(b);
    long long t = 0;
    if (targets) t = targets_i64 ? ((const long long*)targets)[b] : (long long)((const int*)targets)[b];
    int what = 0;
    if (n < 0) what |= 1;
    if (n > max_seq_len) what |= 2;
    if (t < 0 || t > n) what |= 4;
    if (n > 0 && n - t < c) what |= 8;
    if (delta > 0 && n < delta) what |= 16;
    if (what) {
        atomicAdd(report, 1);
        atomicMin(report + 1, b);
        atomicOr(report + 2, what);
    }
}

}  // namespace hstu

// The pipelined kernels' variant for fitted runs: a translation unit of its own (hstu_fwd_fitted.hip).
extern "C" __attribute__((visibility("hidden"))) void hstu_hip_launch_fitted(const hstu::FwdParams* p, int dtype, int dim, int cfg, int grid_per_xcd,
                                                                           hipStream_t stream);

namespace {

constexpr int kMaxSortBatch = 8192;  // beyond this the quadratic ranking is not worth its time

thread_local char g_last_error[256] = "";

void set_last_error(const char* what, hipError_t e) {
    snprintf(g_last_error, sizeof(g_last_error), "%s: %s", what, hipGetErrorString(e));
}

struct TileConfig {
    const char* name;
    int qt, nw, bn;  // query tiles (of 32 rows) per wave, waves per workgroup, kv rows per tile
};
// id 1..: see hstu_hip_tile_configs()
const TileConfig kConfigs[] = {
    {"m128n64w4", 1, 4, 64},
    {"m256n64w8pp", 1, 8, 64},
    {"m128n64w4pl", 1, 4, 64},
};
constexpr int kNumConfigs = sizeof(kConfigs) / sizeof(kConfigs[0]);

// `p` arrives complete (num_mb, pairs_per_xcd, slots_per_xcd, queue ...); these only pick the instantiation.
template <class TT, int DQK, int DV, int QT, int NW, int BN, int OCC>
int launch(const hstu::FwdParams& p, hipStream_t stream) {
    // + 64: with dv = 16 the transposing reads of the unused upper half of the tile reach past the last V row
    constexpr int smem = 2 * BN * (DQK + DV) * TT::ES + 64;
    auto kern = hstu::hstu_fwd_kernel<TT, DQK, DV, QT, NW, BN, OCC>;
    // once per device (the attribute belongs to the device's copy of the kernel); raising the dynamic LDS limit is
    // idempotent, so racing threads only set the same value twice
    static std::atomic<bool> attr_done[64];
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) dev = -1;
    if (dev < 0 || !attr_done[dev]) {
        hipError_t e = hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, smem);
        if (e != hipSuccess) {
            set_last_error("hipFuncSetAttribute", e);
            return HSTU_ERR_LAUNCH;
        }
        if (dev >= 0) attr_done[dev] = true;
    }
    const long long grid = (long long)p.slots_per_xcd * 8;  // one workgroup per work item
    hipLaunchKernelGGL(kern, dim3((unsigned)grid), dim3(NW * 64), smem, stream, p);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) {
        set_last_error("kernel launch", e);
        return HSTU_ERR_LAUNCH;
    }
    return HSTU_OK;
}

// Constants for fast_div (device side): x / d == (x * magic) >> (32 + shift) for 0 <= x < 2^31; magic 0 means d == 1.
void fast_div_constants(unsigned d, unsigned* magic, unsigned* shift) {
    if (d <= 1) {
        *magic = 0;
        *shift = 0;
        return;
    }
    unsigned l = 0;
    while ((1ull << l) < d) ++l;  // ceil(log2 d) >= 1
    *magic = (unsigned)((1ull << (31 + l)) / d + 1);
    *shift = l - 1;
}

template <class TT, int DQK, int DV, int BN, int NG>
int launch_pp(const hstu::FwdParams& p, int grid_per_xcd, int64_t total_q, hipStream_t stream) {
    if (p.fit_runs > 0) {
        hstu_hip_launch_fitted(&p, TT::CODE, DQK, NG == 0 ? 2 : 3, grid_per_xcd, stream);
    } else if constexpr (NG == 0) {  // the streaming form of the 8-wave kernel
        hipLaunchKernelGGL((hstu::hstu_fwd_stream_kernel<TT, DQK, DV, BN, false>), dim3((unsigned)grid_per_xcd * 8), dim3(512), 0, stream, p);
    } else {
        hipLaunchKernelGGL((hstu::hstu_fwd_pp_kernel<TT, DQK, DV, BN, NG, false>), dim3((unsigned)grid_per_xcd * 8), dim3(NG * 256), 0, stream,
                           p);  // LDS is a static array
    }
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) {
        set_last_error("kernel launch", e);
        return HSTU_ERR_LAUNCH;
    }
    if (p.kv_splits > 1 || p.fit_runs > 0) {
        constexpr int LG = DV == 32 ? 3 : DV == 64 ? 4 : 5;
        static_assert(DV == 4 << LG, "the reduce kernel's threads per row and head");
        const long long rows = (long long)total_q * p.H, blocks = (rows + (256 >> LG) - 1) / (256 >> LG);
        if (rows > 0x7fffffffLL) return HSTU_ERR_BAD_SHAPE;
        hstu::ReduceParams rp;
        rp.offsets = p.offsets, rp.offsets_i64 = p.offsets_i64, rp.partial = p.partial, rp.counts = p.split_counts;
        rp.o = p.o, rp.o_rs = p.o_rs, rp.o_hs = p.o_hs;
        rp.attn_scale = p.attn_scale, rp.attn_scale_per_row = p.attn_scale_per_row, rp.oscale = p.oscale, rp.oscale_unit = p.oscale_unit;
        rp.B = p.B, rp.H = p.H, rp.num_mb = p.num_mb, rp.max_seq_len = p.max_seq_len, rp.delta = p.delta, rp.rows = (unsigned)rows;
        rp.fit_slots = p.fit_runs > 0 ? p.fit_slots : 0, rp.pitch = p.fit_runs > 0 ? (int64_t)p.fit_rows * DV : p.partial_stride;
        rp.h_magic = p.h_magic, rp.h_shift = p.h_shift;
        fast_div_constants((unsigned)(p.delta > 0 ? p.delta : 1), &rp.delta_magic, &rp.delta_shift);
        hipLaunchKernelGGL((hstu::hstu_reduce_splits_kernel<typename TT::out_elem, LG, NG == 1 ? 128 : 256>), dim3((unsigned)blocks), dim3(256), 0, stream, rp);
        e = hipGetLastError();
        if (e != hipSuccess) {
            set_last_error("reduce kernel launch", e);
            return HSTU_ERR_LAUNCH;
        }
    }
    return HSTU_OK;
}

template <class TT, int D>
int launch_cfg(const hstu::FwdParams& p, int cfg, int grid_per_xcd, int64_t total_q, hipStream_t stream) {
    if (cfg == 2) return launch_pp<TT, D, D, 64, 0>(p, grid_per_xcd, total_q, stream);  // 8 waves, two groups: the streaming kernel
    if (cfg == 3) return launch_pp<TT, D, D, 64, 1>(p, grid_per_xcd, total_q, stream);  // 4 waves, one group
    return launch<TT, D, D, 1, 4, 64, 2>(p, stream);
}

// Unequal or 16-wide head dims: only the barrier-per-tile kernel is generic in (dqk, dv).
template <class TT, int DQK>
int launch_mixed_dv(const hstu::FwdParams& p, int dv, hipStream_t stream) {
    switch (dv) {
        case 16:
            if constexpr (TT::ES == 2) return launch<TT, DQK, 16, 1, 4, 64, 2>(p, stream);
            return HSTU_ERR_BAD_HEAD_DIM;
        case 32: return launch<TT, DQK, 32, 1, 4, 64, 2>(p, stream);
        case 64: return launch<TT, DQK, 64, 1, 4, 64, 2>(p, stream);
        case 128: return launch<TT, DQK, 128, 1, 4, 64, 2>(p, stream);
        default: return HSTU_ERR_BAD_HEAD_DIM;
    }
}

template <class TT>
int launch_mixed(const hstu::FwdParams& p, int dqk, int dv, hipStream_t stream) {
    switch (dqk) {
        case 16:
            if constexpr (TT::ES == 2) return launch_mixed_dv<TT, 16>(p, dv, stream);
            return HSTU_ERR_BAD_HEAD_DIM;
        case 32: return launch_mixed_dv<TT, 32>(p, dv, stream);
        case 64: return launch_mixed_dv<TT, 64>(p, dv, stream);
        case 128: return launch_mixed_dv<TT, 128>(p, dv, stream);
        default: return HSTU_ERR_BAD_HEAD_DIM;
    }
}

template <class TT>
int launch_dim(const hstu::FwdParams& p, int d, int dv, int cfg, int grid_per_xcd, int64_t total_q, hipStream_t stream) {
    if (cfg == 1 && (d != dv || d == 16)) return launch_mixed<TT>(p, d, dv, stream);
    switch (d) {
        case 32: return launch_cfg<TT, 32>(p, cfg, grid_per_xcd, total_q, stream);
        case 64: return launch_cfg<TT, 64>(p, cfg, grid_per_xcd, total_q, stream);
        case 128: return launch_cfg<TT, 128>(p, cfg, grid_per_xcd, total_q, stream);
        default: return HSTU_ERR_BAD_HEAD_DIM;
    }
}

// What a call will do, from sizes the host knows without reading the offsets.
struct Plan {
    int cfg;               // tile configuration, 1-based
    int splits;            // workgroups per row block along kv (1 = no split)
    bool one_each;         // a workgroup for every item there could be: no counters, no lists
    int chunk;             // kv tiles per run when split
    int fit_runs;          // runs fitted to the lengths (decode_fitted): workgroups per (head, row block), 0 = off; `splits` is then
                           // their average number per row block
    int line_weight;       // > 0: those workgroups share the plane's tiles as one line instead (decode_line)
    // the workspace, in this order:
    size_t queue_bytes;    // work-item counters and list lengths of the persistent kernels
    size_t order_bytes;    // sequence ranking
    size_t counts_bytes;   // runs per row block of a kv-split
    size_t partial_bytes;  // fp32 partial outputs of the runs (256-byte aligned: 256 bytes of slack are added)
    size_t items_bytes;    // work lists: 8 lists of 32-byte records (see FwdParams::items)
    size_t cast_bytes;     // fp16 copies of fp32 q, k, v, each 256-byte aligned
    size_t total() const {
        return queue_bytes + order_bytes + counts_bytes + (partial_bytes ? partial_bytes + 256 : 0) + items_bytes + cast_bytes;
    }
};

constexpr int kMaxSplits = 8;
constexpr int kTileRows = 64;  // kv rows per tile of every configuration

// The pipelined kernels address the rows of a sequence through buffer descriptors with 32-bit byte offsets: the longest
// sequence times the largest row stride has to stay below 2^32 bytes.
bool rows_fit_buffer_offsets(const HstuFwdArgs* a) {
    const int64_t es = a->dtype == HSTU_FP8_E4M3 ? 1 : 2;
    int64_t rs = a->q_row_stride > a->k_row_stride ? a->q_row_stride : a->k_row_stride;
    if (a->v_row_stride > rs) rs = a->v_row_stride;
    return (int64_t)a->max_seq_len * rs * es < (1LL << 32);
}

// `scratch`: bytes of workspace at hand; an automatic kv-split is one that fits.  `line`: whether a plane's tiles may be cut as one line.
Plan make_plan(const HstuFwdArgs* a, size_t scratch = SIZE_MAX, bool line = true) {
    Plan pl{};
    pl.splits = 1;
    // The streaming two-group kernel (256-row blocks, one workgroup per CU) wins when the average sequence is long;
    // the one-group pipeline (128-row blocks, two workgroups per CU) wastes less on short or very uneven sequences
    // and in delta mode.
    pl.cfg = a->tile_config;
    const long long avg_tiles = a->batch > 0 ? a->total_kv / a->batch / kTileRows : 0;
    if (a->dqk != a->dv || a->dqk == 16) pl.cfg = 1;  // the only kernel generic in (dqk, dv)
    if (pl.cfg == 0 && !rows_fit_buffer_offsets(a)) pl.cfg = 1;  // the only kernel with 64-bit row addresses
    if (a->dtype == HSTU_FP32) {
        pl.cfg = 1;  // and the only one with an fp32 store
        pl.cast_bytes = 2 * ((size_t)a->total_q * a->heads * a->dqk + (size_t)a->total_kv * a->heads * (a->dqk + a->dv)) + 4 * 256;
    }
    if (pl.cfg == 0) {
        if (a->delta_size == 0) {
            // (measured, H = 4, d = 128, by average length: 544 rows -- the streaming kernel is 6 % behind; 900 to 1000
            // -- 1 to 3 % ahead; 1280 -- level; 1800 -- 3 % ahead; 2048 to 2560 -- 6 to 8 % ahead)
            pl.cfg = avg_tiles >= 960 / kTileRows ? 2 : 3;
        } else {
            // Few long histories: 256-row blocks, whose kv range is then split below so that every CU gets one -- where their
            // second half exists (5 histories of 8000 .. 16000 x 100 candidates, 4 heads: 44 us against 38 with 128-row blocks)
            // and a CU's share is at least 8 tiles, below which what an item costs besides its steps counts for more
            // (256 candidates: 2 and 8 histories of 1000 .. 4000: 25 and 35 us against 22 and 32; 5 of 8000 .. 16000: 51
            // against 56; 32 of 1024 .. 4096: 73 against 78).
            const long long mb256 = (a->delta_size + 255) / 256, blocks256 = (long long)a->batch * a->heads * mb256;
            const bool half_empty = (a->delta_size - 1) % 256 < 128;
            const bool long_runs = a->total_kv / kTileRows * a->heads * mb256 >= 8 * 256;
            pl.cfg = (blocks256 * 2 <= 256 && avg_tiles >= 32 && !half_empty && long_runs) ? 2 : 3;
        }
    }
    if (a->sort_by_length && a->batch >= 2 && a->batch <= kMaxSortBatch) pl.order_bytes = (size_t)a->batch * sizeof(int);
    if (pl.cfg < 2 || a->batch <= 0) return pl;
    pl.queue_bytes = 8 * 64 + 64;  // one counter per XCD, 64 bytes apart, then the 8 list lengths
    const int bm = pl.cfg == 2 ? 256 : 128;
    const int rows_per_pair = a->delta_size > 0 ? a->delta_size : a->max_seq_len;
    const long long blocks = (long long)a->batch * a->heads * ((rows_per_pair + bm - 1) / bm);
    const int max_tiles = (a->max_seq_len + kTileRows - 1) / kTileRows;
    const size_t split_counts_bytes = (size_t)blocks * sizeof(int), split_bytes = (size_t)a->total_q * a->heads * a->dv * sizeof(float);
    int s = 1;
    if (a->kv_splits > 0) {
        s = a->kv_splits;
    } else if (a->delta_size > 0) {
        // Delta mode has few query rows per sequence: with a small batch the row blocks alone do not fill the
        // 256 CUs.  Cut the kv range so that the chip is just filled (more runs than that only add partial-sum
        // traffic: with every CU busy the clock drops and the time per tile rises), in runs of at least 16 tiles.
        const long long resident = pl.cfg == 2 ? 256 : 512;  // workgroups the chip holds at once
        // Runs fitted to the lengths where the whole history is in reach of every row (no window, no contextual prefix), for at
        // most 64 sequences (decode_fitted has a lane for each).  128-row blocks: one workgroup per CU (a second one halves
        // the runs but not what an item costs, and both wait for the same HBM: 16 x 1000 .. 4000 x 128 candidates 31 us
        // with 256 workgroups, 40 with 512; 5 x 8000 .. 16000 x 100: 37 and 45) unless the row blocks alone are more than 64
        // (30 x 7300 .. 14600 x 91: 173 and 150).  Short runs still pay: 50 candidates x 400 rows, 16.7 us unsplit, 12.4 us in
        // runs of one tile.  Below 6 tiles saved the extra kernel and the partial sums cost more than the shorter runs save;
        // with fewer than four workgroups per sequence there is little to fit (32 x 1024 .. 4096 x 256: 76 us, equal counts 73).
        const bool fits = a->max_attn_len == 0 && a->contextual_seq_len == 0 && a->batch <= 64 && max_tiles <= (1 << 20);
        const long long chip = pl.cfg == 2 ? 256 : blocks * 4 <= 256 ? 256 : 512;
        const long long num_mb = (rows_per_pair + bm - 1) / bm, planes = a->heads * num_mb;
        const long long tiles = a->total_kv / kTileRows + a->batch;  // of a plane, at most
        const size_t run_bytes = (size_t)planes * (rows_per_pair < bm ? rows_per_pair : bm) * a->dv * sizeof(float);
        long long runs = chip / 8 / num_mb * 8 / a->heads;
        if (runs > tiles) runs = tiles;
        if (fits && runs >= 4 * a->batch && max_tiles - (tiles + runs - 1) / runs >= 6) {
            pl.fit_runs = (int)runs;
            pl.splits = (int)(runs / a->batch);
            pl.counts_bytes = split_counts_bytes;
            pl.partial_bytes = runs * run_bytes;
            if (pl.total() <= scratch) return pl;
            pl.fit_runs = 0, pl.splits = 1;  // their partial sums take more than those of equal counts can
            pl.counts_bytes = pl.partial_bytes = 0;
        }
        long long want = resident / blocks;
        if (want > max_tiles / 16) want = max_tiles / 16;
        if (want > kMaxSplits) want = kMaxSplits;
        while (want >= 2 && pl.total() + split_counts_bytes + want * split_bytes + 256 > scratch) --want;
        if (want >= 2) s = (int)want;
        // Fewer workgroups than that per sequence: the plane's tiles as one line (decode_line), where the longest run is at least 8 tiles longer than a workgroup's part of
        // it (14 without equal runs and with several row blocks, whose rows all go through partial sums).  us without / with (bf16, lengths of the histories x candidates): 34 of 2400 .. 2550 x 19, 8
        // heads of 32 67 / 45; 18 of 250 .. 4200 x 3, 8 of 128 57 / 35; 46 of 400 .. 1600 x 3, 4 of 128 40 / 28; 39 of 650 .. 10800 x 212, 4 of 128 243 / 157; 16 of 500 .. 8000 x 512 105 / 89; 32 of
        // 1024 .. 4096 x 256 74 / 74.  Not for shorter ones (36 of 550 x 278 38 / 52; 40 of 100 .. 400 x 30 16 / 21) nor for many row blocks (46 of 4500 .. 9000 x 389, 8 heads 798 / 877; 64 of
        // 500 .. 4000 x 500 214 / 221).  Where max_seq_len is more than 2.5 times the mean length it says little about the longest: then the mean has to be that much longer (51 of 38 .. 64 x 132,
        // max_seq_len 5666, 4 of 128 15.3 / 28.2; 49 of 2112 x 72, 45342, 8 of 128 95 / 118; 37 of 668 .. 13378 x 23, 33629, 8 of 32 213 / 102), or, beside equal runs, which such a
        // max_seq_len makes too long, at least 8 tiles (17 of 258 .. 431 x 103, 12971, 8 of 64 17.3 / 19.9; 32 of 212 .. 4247 x 5, 9300, 8 of 32 88 / 36).
        // What an item costs besides its steps, in tiles (2, 5, 9: the first 45 / 47 / 50, the last but one of the gains 91 / 89 / 87):
        const int weight = pl.cfg == 2 ? 8 : 4;
        const bool near_mean = 2ll * a->max_seq_len * a->batch <= 5ll * a->total_kv;
        const long long part = runs > 0 ? (tiles + a->batch * weight + runs - 1) / runs : 0;
        const bool pays = s > 1 ? avg_tiles >= 8 && (max_tiles + s - 1) / s - part >= 8
                                : (near_mean ? max_tiles : avg_tiles) - part >= (num_mb > 1 ? 14 : 8);
        if (line && fits && runs > 0 && pays && (tiles + a->batch * weight) * runs < (1ll << 31)) {
            pl.fit_runs = (int)runs, pl.line_weight = weight, pl.splits = 2;
            pl.counts_bytes = split_counts_bytes;
            pl.partial_bytes = (runs + a->batch) * run_bytes;
            if (pl.total() <= scratch) return pl;
            pl.fit_runs = pl.line_weight = 0, pl.splits = 1;
            pl.counts_bytes = pl.partial_bytes = 0;
        }
    }
    // Work lists for ragged batches (equal lengths are dealt arithmetically, a kv-split enumerates its runs
    // arithmetically too): 32 bytes per possible item; beyond 64 MB the arithmetic enumeration stays.
    const bool uniform = a->delta_size == 0 && a->total_kv == (int64_t)a->batch * a->max_seq_len;
    // For few of the one-group kernel's items the list (for which the workspace still has room) costs more than it gives: the kernel that builds it takes 5 to 6 us
    // (ranking the sequences another 10 at 256 of them), a workgroup that finds no rows leaves at once.  us, lists / a workgroup for every item there could be (4 heads of
    // 64, ragged, ranked): 96 sequences of 20 .. 276 rows, 144 items per XCD, 23.3 / 16.4; 256 of 20 .. 128 33.9 / 14.9; 48 of 200 .. 700 27.5 / 24.2; 8 heads, 28 of 64 .. 1000,
    // 224 items, 31.5 / 29.5, 64 of 100 .. 512, 256 items, 35.7 / 34.0; 8 heads of 128, 20 of 300 .. 1300, 220 items 67.1 / 63.0.  More of them want the heaviest first (with a list
    // that took 2 us longer): 64 of 200 .. 960, 4 heads of 128, 256 items 65.0 / 67.4; 100 of 300 .. 900, 400 items 81 / 86; 1024 items 190 / 203.  One row block per sequence:
    // 500 of 20 .. 128, 8 heads, 500 items, 56.7 / 44.3; 32 columns, where more than two workgroups fit a CU: 100 of 300 .. 900 47.0 / 44.7.
    const long long num_mb = (rows_per_pair + bm - 1) / bm, slots = (a->batch * (long long)a->heads + 7) / 8 * num_mb;
    pl.one_each = s == 1 && !uniform && pl.cfg == 3 && a->delta_size == 0 && slots <= (num_mb == 1 || a->dqk == 32 ? 512 : num_mb <= 4 ? 256 : 224);
    if (s == 1 && !uniform) {
        const unsigned long long bytes = (unsigned long long)slots * 256ull;
        if (bytes <= (64ull << 20)) pl.items_bytes = (size_t)bytes + 32;  // 32: room to align the records
    }
    if (s > 1) {
        pl.splits = s;
        pl.chunk = (max_tiles + s - 1) / s;
        pl.counts_bytes = split_counts_bytes;
        pl.partial_bytes = (size_t)s * split_bytes;
    }
    return pl;
}

size_t scratch_bytes(const HstuFwdArgs* a) { return a->workspace ? (size_t)a->workspace_bytes : 0; }

// The launch of a plan on a device of `cus` CUs: work items per XCD, and for the persistent kernels the workgroups that stay resident
// (the same number on every XCD).
struct Grid {
    int num_mb;
    long long pairs_per_xcd;
    long long fit_wgs;  // per XCD: workgroups of fitted runs, 0 without
    long long slots;    // per XCD: items
    int per_xcd;        // per XCD: workgroups
};

Grid make_grid(const HstuFwdArgs* a, const Plan& plan, int cus) {
    const int rows_per_pair = a->delta_size > 0 ? a->delta_size : a->max_seq_len;
    const int bm = plan.cfg == 2 ? 256 : 128;
    Grid g;
    g.num_mb = (rows_per_pair + bm - 1) / bm;
    g.pairs_per_xcd = ((long long)a->batch * a->heads + 7) / 8;
    g.fit_wgs = (((long long)plan.fit_runs * a->heads + 7) / 8) * g.num_mb;
    g.slots = plan.fit_runs > 0 ? g.fit_wgs * (plan.line_weight > 0 ? a->batch : 1) : g.pairs_per_xcd * g.num_mb * plan.splits;
    // workgroups of a CU: of the one-group kernel two, with 32 columns (161 registers in bf16, 129 in fp16) the three that fit (us, two / three: 256 sequences of 64 .. 1024, 4 heads 112 / 104; 256 of
    // 256 31 / 26; 200 of 512 56 / 52; 100 of 300 .. 900 50 / 50).  Of 64 columns in bf16 (190 registers) two fit, and a grid for three queues the third behind them (256 of 64 .. 1024 138 / 149; 200
    // of 512 73 / 86); in fp16 (162) three fit and are 8 % faster to 3 % slower (118 of 531, 8 heads 135 / 126; 147 of 1113, 4 heads 213 / 217): not taken.
    const int per_cu = plan.cfg == 2 ? 1 : a->dqk == 32 && a->dtype != HSTU_FP8_E4M3 ? 3 : 2;
    long long resident = (long long)cus * per_cu / 8;
    if (resident < 1) resident = 1;
    if (plan.one_each) resident = g.slots;
    // Fitted runs: a workgroup each, also where the device has fewer CUs than make_plan sized them for (a partition of it): the kernel's
    // workgroups end at the first item that decodes to nothing, as those behind the last run of a head do.
    if (plan.fit_runs > 0) resident = g.fit_wgs;
    g.per_xcd = (int)(g.slots < resident ? g.slots : resident);
    return g;
}

void fill_decode_params(hstu::FwdParams& p) {
    hstu::DecodeParams& d = p.dec;
    memset(&d, 0, sizeof(d));
    d.items = p.items;
    d.nitems = p.nitems;
    d.order = p.order;
    d.offsets = p.offsets;
    d.targets = p.targets;
    d.items_cap = p.items_cap;
    d.kv_splits = p.kv_splits;
    d.kv_chunk = p.kv_chunk;
    d.c = p.c;
    d.pairs_per_xcd = p.pairs_per_xcd;
    d.num_mb = p.num_mb;
    d.B = p.B;
    d.H = p.H;
    d.uniform = p.uniform;
    d.max_seq_len = p.max_seq_len;
    d.offsets_i64 = p.offsets_i64;
    d.targets_i64 = p.targets_i64;
    d.delta = p.delta;
    d.w = p.w;
    d.f = p.f;
    d.fit_runs = p.fit_runs;
    d.line_weight = p.line_weight;
    d.line_wgs = p.line_wgs;
    d.mb_magic = p.mb_magic;
    d.mb_shift = p.mb_shift;
    d.h_magic = p.h_magic;
    d.h_shift = p.h_shift;
}

bool aligned16(const void* ptr) { return (reinterpret_cast<uintptr_t>(ptr) & 15) == 0; }

// 1 if the current device is gfx950, 0 if not, cached per device ordinal (the kernels use gfx950-only
// instructions; the reference's native op makes the same kind of check, flash_common.cpp:420-422).
int current_device_is_gfx950() {
    static std::atomic<int> cache[64];  // 0 unknown, 1 yes, 2 no; racing threads store the same value
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess) return 0;
    if (dev < 0 || dev >= 64) return 0;
    if (cache[dev] == 0) {
        hipDeviceProp_t prop;
        if (hipGetDeviceProperties(&prop, dev) != hipSuccess) return 0;
        cache[dev] = strncmp(prop.gcnArchName, "gfx950", 6) == 0 ? 1 : 2;
    }
    return cache[dev] == 1;
}

// Compute units of the current device (256 on MI355X), cached per device ordinal.
int current_device_cus() {
    static std::atomic<int> cache[64];
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) return 256;
    if (cache[dev] == 0) {
        int n = 0;
        if (hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || n <= 0) n = 256;
        cache[dev] = n;
    }
    return cache[dev];
}

}  // namespace

// for the library's other translation units; not exported
extern "C" __attribute__((visibility("hidden"))) int hstu_hip_device_is_gfx950(void) { return current_device_is_gfx950(); }
extern "C" __attribute__((visibility("hidden"))) void hstu_hip_set_last_error(const char* what, int hip_error) {
    set_last_error(what, (hipError_t)hip_error);
}

// order[rank] = sequence index, longest first, for the backward entry point's schedule; 0 or HSTU_ERR_LAUNCH
extern "C" __attribute__((visibility("hidden"))) int hstu_hip_launch_rank(const void* offsets, int offsets_i64, int batch, int* order,
                                                                          void* stream) {
    const unsigned blocks = (unsigned)(((long long)batch * 64 + 255) / 256);
    hipLaunchKernelGGL(hstu::hstu_prep_kernel, dim3(blocks), dim3(256), 0, (hipStream_t)stream, offsets, offsets_i64, batch, order,
                       (int*)nullptr, 0);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) {
        set_last_error("rank kernel launch", e);
        return HSTU_ERR_LAUNCH;
    }
    return HSTU_OK;
}

extern "C" {

int hstu_hip_version(void) { return 101; }

const char* hstu_hip_status_string(int status) {
    switch (status) {
        case HSTU_OK: return "ok";
        case HSTU_ERR_NULL_POINTER: return "a required pointer is NULL";
        case HSTU_ERR_BAD_DTYPE: return "only bf16, fp16, fp8_e4m3 and fp32 data types are supported";
        case HSTU_ERR_BAD_HEAD_DIM: return "unsupported head dimension (built: dqk, dv in {16, 32, 64, 128}; 8-bit types from 32)";
        case HSTU_ERR_MISALIGNED:
            return "q/k/v/out must be 16-byte aligned with row and head strides that are multiples of 16 bytes";
        case HSTU_ERR_BAD_SHAPE: return "inconsistent sizes";
        case HSTU_ERR_UNSUPPORTED: return "argument combination not built";
        case HSTU_ERR_LAUNCH: return "HIP launch failed";
        case HSTU_ERR_BAD_DEVICE: return "current device is not gfx950";
        case HSTU_ERR_SCRATCH_LIMIT: return "the call needs more scratch memory than the library's fixed area holds";
        case HSTU_ERR_BUSY: return "the library's fixed scratch area is still in use by a call on another stream";
        default: return "unknown status";
    }
}

const char* hstu_hip_last_error(void) { return g_last_error; }

size_t hstu_hip_workspace_bytes(const HstuFwdArgs* a) {
    if (!a || a->batch <= 0 || a->heads <= 0 || a->total_q <= 0) return 0;
    return make_plan(a).total();
}

int hstu_hip_plan(const HstuFwdArgs* a, int32_t* tile_config, int32_t* kv_splits) {
    int rc = hstu_hip_check_args(a);
    if (rc != HSTU_OK) return rc;
    const Plan pl = make_plan(a, scratch_bytes(a));
    if (tile_config) *tile_config = pl.cfg;
    if (kv_splits) *kv_splits = pl.splits;
    return HSTU_OK;
}

int hstu_hip_plan_grid(const HstuFwdArgs* a, int32_t cus, int32_t* form, int32_t* items, int32_t* workgroups) {
    const int rc = hstu_hip_check_args(a);
    if (rc != HSTU_OK) return rc;
    if (cus <= 0) return HSTU_ERR_BAD_SHAPE;
    const Plan pl = make_plan(a, scratch_bytes(a));
    const Grid g = make_grid(a, pl, cus);
    if (g.slots * 8 > 0x7fffffffLL) return HSTU_ERR_BAD_SHAPE;
    if (form) *form = pl.line_weight > 0 ? HSTU_PLAN_LINE : pl.fit_runs > 0 ? HSTU_PLAN_FITTED : pl.splits > 1 ? HSTU_PLAN_EQUAL_RUNS : HSTU_PLAN_WHOLE;
    if (items) *items = (int32_t)g.slots;
    if (workgroups) *workgroups = pl.cfg < 2 ? (int32_t)g.slots : g.per_xcd;
    return HSTU_OK;
}

int hstu_hip_tile_configs(void) { return kNumConfigs; }

const char* hstu_hip_tile_config_name(int id) {
    if (id < 1 || id > kNumConfigs) return "";
    return kConfigs[id - 1].name;
}

int hstu_hip_check_args(const HstuFwdArgs* a) {
    if (!a) return HSTU_ERR_NULL_POINTER;
    if (a->dtype != HSTU_BF16 && a->dtype != HSTU_FP16 && a->dtype != HSTU_FP8_E4M3 && a->dtype != HSTU_FP32) return HSTU_ERR_BAD_DTYPE;
    if (a->batch < 0 || a->heads <= 0 || a->total_q < 0 || a->total_kv < 0 || a->max_seq_len <= 0 ||
        a->delta_size < 0 || a->max_attn_len < 0 || a->contextual_seq_len < 0 || a->min_full_attn_seq_len < 0)
        return HSTU_ERR_BAD_SHAPE;
    if (a->delta_size > 0 && a->total_q != (int64_t)a->batch * a->delta_size) return HSTU_ERR_BAD_SHAPE;
    if (a->delta_size == 0 && a->total_q != a->total_kv) return HSTU_ERR_BAD_SHAPE;
    if (a->total_kv > 0x7fffffffLL) return HSTU_ERR_BAD_SHAPE;
    if (a->tile_config < 0 || a->tile_config > kNumConfigs) return HSTU_ERR_BAD_SHAPE;
    if (a->kv_splits < 0 || a->kv_splits > kMaxSplits || (a->kv_splits > 1 && a->tile_config == 1)) return HSTU_ERR_BAD_SHAPE;
    if (a->workspace && (a->workspace_bytes < 0 || (reinterpret_cast<uintptr_t>(a->workspace) & 3) != 0)) return HSTU_ERR_MISALIGNED;
    if (a->attn_scale && (reinterpret_cast<uintptr_t>(a->attn_scale) & 3) != 0) return HSTU_ERR_MISALIGNED;
    if (a->attn_scale && a->delta_size > 0) return HSTU_ERR_UNSUPPORTED;  // the reference's cached form has no attn_scale
    // head dims 16 / 32 / 64 / 128, independently for q/k and v (the grid of the reference's tests,
    // hstu_attention_test.py:266-267; its native op wants them equal, flash_common.cpp:543-545); 8-bit rows are at
    // least 32 wide
    for (int d : {a->dqk, a->dv})
        if (d != 32 && d != 64 && d != 128 && !(d == 16 && a->dtype != HSTU_FP8_E4M3)) return HSTU_ERR_BAD_HEAD_DIM;
    // unequal or 16-wide dims and fp32 run on tile config 1 only
    if ((a->dqk != a->dv || a->dqk == 16 || a->dtype == HSTU_FP32) && a->tile_config > 1) return HSTU_ERR_UNSUPPORTED;
    // ... and so do sequences whose rows span 4 GB or more
    if (a->tile_config > 1 && !rows_fit_buffer_offsets(a)) return HSTU_ERR_UNSUPPORTED;
    if (a->total_q == 0 || a->batch == 0) return HSTU_OK;  // nothing to do; pointers may be anything
    if (!a->q || !a->k || !a->v || !a->out || !a->seq_offsets) return HSTU_ERR_NULL_POINTER;
    if (!aligned16(a->q) || !aligned16(a->k) || !aligned16(a->v) || !aligned16(a->out)) return HSTU_ERR_MISALIGNED;
    const int64_t strides[8] = {a->q_row_stride, a->q_head_stride, a->k_row_stride, a->k_head_stride,
                                a->v_row_stride, a->v_head_stride, a->o_row_stride, a->o_head_stride};
    // rows of q/k/v start on 16-byte boundaries: 8 elements of 16 bits, 16 of 8 bits, 4 of 32 bits; the output is 16
    // bit, or 32 bit for fp32 inputs
    const int64_t in_mask = a->dtype == HSTU_FP8_E4M3 ? 15 : a->dtype == HSTU_FP32 ? 3 : 7;
    const int64_t out_mask = a->dtype == HSTU_FP32 ? 3 : 7;
    for (int i = 0; i < 8; ++i)
        if (strides[i] < 0 || (strides[i] & (i < 6 ? in_mask : out_mask)) != 0) return HSTU_ERR_MISALIGNED;
    return HSTU_OK;
}

int hstu_hip_check_contract(const HstuFwdArgs* a, int32_t* report, void* stream_) {
    g_last_error[0] = 0;
    int rc = hstu_hip_check_args(a);
    if (rc != HSTU_OK) return rc;
    if (!report) return HSTU_ERR_NULL_POINTER;
    hipStream_t stream = (hipStream_t)stream_;
    // a small fill kernel would do as well; this copy is outside anything a caller captures (the check reads back).
    // The source outlives the call: an asynchronous copy from pageable memory may read it after this function returns.
    static const int32_t init[4] = {0, 0x7fffffff, 0, 0};
    hipError_t e = hipMemcpyAsync(report, init, sizeof(init), hipMemcpyHostToDevice, stream);
    if (e != hipSuccess) {
        set_last_error("hipMemcpyAsync", e);
        return HSTU_ERR_LAUNCH;
    }
    if (a->batch == 0 || !a->seq_offsets) return HSTU_OK;
    hipLaunchKernelGGL(hstu::hstu_check_contract_kernel, dim3((a->batch + 255) / 256), dim3(256), 0, stream, a->seq_offsets,
                       a->seq_offsets_i64, a->num_targets, a->num_targets_i64, a->batch, (long long)a->total_kv, a->max_seq_len,
                       a->contextual_seq_len, a->delta_size, report);
    e = hipGetLastError();
    if (e != hipSuccess) {
        set_last_error("contract kernel launch", e);
        return HSTU_ERR_LAUNCH;
    }
    return HSTU_OK;
}

int hstu_hip_mha_fwd(const HstuFwdArgs* a, void* stream_) {
    g_last_error[0] = 0;
    int rc = hstu_hip_check_args(a);
    if (rc != HSTU_OK) return rc;
    if (a->total_q == 0 || a->batch == 0) return HSTU_OK;
    if (!current_device_is_gfx950()) return HSTU_ERR_BAD_DEVICE;
    hipStream_t stream = (hipStream_t)stream_;

    hstu::FwdParams p;
    memset(&p, 0, sizeof(p));
    p.q = (const char*)a->q;
    p.k = (const char*)a->k;
    p.v = (const char*)a->v;
    p.o = (char*)a->out;
    p.q_rs = a->q_row_stride;
    p.q_hs = a->q_head_stride;
    p.k_rs = a->k_row_stride;
    p.k_hs = a->k_head_stride;
    p.v_rs = a->v_row_stride;
    p.v_hs = a->v_head_stride;
    p.o_rs = a->o_row_stride;
    p.o_hs = a->o_head_stride;
    p.offsets = a->seq_offsets;
    p.targets = a->num_targets;
    p.offsets_i64 = a->seq_offsets_i64;
    p.targets_i64 = a->num_targets_i64;
    p.B = a->batch;
    p.H = a->heads;
    p.max_seq_len = a->max_seq_len;
    p.delta = a->delta_size;
    p.w = a->max_attn_len;
    p.c = a->contextual_seq_len;
    p.f = a->min_full_attn_seq_len;
    p.c1 = -a->alpha * 1.4426950408889634f;
    p.oscale = a->alpha == 0.0f ? 0.0f : -1.0f / ((float)a->max_seq_len * 1.4426950408889634f);
    p.oscale_unit = a->alpha == 0.0f ? 0.0f : -1.0f / 1.4426950408889634f;
    p.attn_scale = (const float*)a->attn_scale;
    p.attn_scale_per_row = a->attn_scale_per_row;
    if (a->dtype == HSTU_FP8_E4M3) {
        // real value = stored value * scale: the score scales go into c1 (applied to the accumulator), the
        // value scale and the factor P is stored with go into the output scale
        p.c1 *= a->q_scale * a->k_scale;
        p.oscale *= a->v_scale / hstu::Fp8::PSCALE;
        p.oscale_unit *= a->v_scale / hstu::Fp8::PSCALE;
    }

    // Every use of the caller's scratch memory is an optimisation that never changes the result: without enough of
    // it an automatic choice falls back to the plain schedule, an explicit kv_splits > 1 is an error.
    Plan plan = make_plan(a, scratch_bytes(a));
    const bool ws_ok = a->workspace && (size_t)a->workspace_bytes >= plan.total();
    if (a->dtype == HSTU_FP32) {
        // the one use of the workspace that is not optional: rounded copies of the inputs
        if (!ws_ok) return a->workspace ? HSTU_ERR_BAD_SHAPE : HSTU_ERR_NULL_POINTER;
        char* cur = (char*)a->workspace + plan.total() - plan.cast_bytes;
        const void* src[3] = {a->q, a->k, a->v};
        const int64_t rs[3] = {a->q_row_stride, a->k_row_stride, a->v_row_stride};
        const int64_t hs[3] = {a->q_head_stride, a->k_head_stride, a->v_head_stride};
        const int64_t rows[3] = {a->total_q, a->total_kv, a->total_kv};
        const int d[3] = {a->dqk, a->dqk, a->dv};
        const char** dst[3] = {&p.q, &p.k, &p.v};
        int64_t* prs[3] = {&p.q_rs, &p.k_rs, &p.v_rs};
        int64_t* phs[3] = {&p.q_hs, &p.k_hs, &p.v_hs};
        hstu::CastParams cast{};
        cast.H = a->heads;
        long long blocks = 0;
        for (int i = 0; i < 3; ++i) {
            cur = (char*)((reinterpret_cast<uintptr_t>(cur) + 255) & ~(uintptr_t)255);
            const long long threads = (long long)rows[i] * a->heads * (d[i] / 8);
            cast.src[i] = (const float*)src[i], cast.dst[i] = (_Float16*)cur;
            cast.rs[i] = rs[i], cast.hs[i] = hs[i], cast.rows[i] = rows[i], cast.d[i] = d[i];
            cast.first[i] = (unsigned)blocks;
            blocks += (threads + 255) / 256;
            if (blocks > 0x7fffffffLL) return HSTU_ERR_BAD_SHAPE;
            *dst[i] = cur;
            *prs[i] = (int64_t)a->heads * d[i];
            *phs[i] = d[i];
            cur += (size_t)rows[i] * a->heads * d[i] * 2;
        }
        if (blocks > 0) {
            hipLaunchKernelGGL(hstu::hstu_cast_f32_f16_kernel, dim3((unsigned)blocks), dim3(256), 0, stream, cast);
            hipError_t e = hipGetLastError();
            if (e != hipSuccess) {
                set_last_error("cast kernel launch", e);
                return HSTU_ERR_LAUNCH;
            }
        }
    }
    if (plan.splits > 1 && !ws_ok) return a->workspace ? HSTU_ERR_BAD_SHAPE : HSTU_ERR_NULL_POINTER;  // (asked for: make_plan's own fit)
    char* ws = (char*)a->workspace;
    const size_t ws_bytes = a->workspace ? (size_t)a->workspace_bytes : 0;
    int* queue = plan.queue_bytes > 0 && ws_bytes >= plan.queue_bytes ? (int*)ws : nullptr;
    int* order = plan.order_bytes > 0 && ws_bytes >= plan.queue_bytes + plan.order_bytes ? (int*)(ws + plan.queue_bytes) : nullptr;
    if (plan.splits > 1) {
        char* base = ws + plan.queue_bytes + plan.order_bytes;
        p.split_counts = (int*)base;
        p.partial = reinterpret_cast<float*>((reinterpret_cast<uintptr_t>(base + plan.counts_bytes) + 255) & ~(uintptr_t)255);
        p.partial_stride = (int64_t)a->total_q * a->heads * a->dv;
        p.kv_chunk = plan.chunk;
        if (plan.fit_runs > 0) {
            p.fit_runs = plan.fit_runs, plan.splits = 1;  // (an item is one run: decode_fitted, decode_line)
            p.line_weight = plan.line_weight, p.fit_slots = plan.fit_runs + (plan.line_weight > 0 ? a->batch : 0);
        }
    }
    p.kv_splits = plan.splits;

    const int cfg = plan.cfg;
    const int rows_per_pair = a->delta_size > 0 ? a->delta_size : a->max_seq_len;
    const int bm = cfg == 2 ? 256 : 128;
    const Grid grid = make_grid(a, plan, current_device_cus());
    p.num_mb = grid.num_mb;
    p.line_wgs = (int)grid.fit_wgs;
    p.fit_rows = rows_per_pair < bm ? rows_per_pair : bm;
    const long long slots = grid.slots;
    if (slots <= 0) return HSTU_OK;
    if (slots * 8 > 0x7fffffffLL) return HSTU_ERR_BAD_SHAPE;
    p.pairs_per_xcd = (int)grid.pairs_per_xcd;
    p.slots_per_xcd = (int)slots;
    fast_div_constants((unsigned)p.num_mb, &p.mb_magic, &p.mb_shift);
    fast_div_constants((unsigned)p.H, &p.h_magic, &p.h_shift);
    // a workgroup each, few row blocks: long sequences first only where there can be long ones, which repays the launch that ranks them (4 heads of 128,
    // one in four of 32 sequences 1500 rows, the others 100: 65 us unranked, 45 ranked; 60 sequences of 100 .. 512, 8 heads 48 and 56)
    if (plan.one_each && p.num_mb <= 4) order = nullptr;
    const int grid_per_xcd = grid.per_xcd;
    if (cfg < 2 || slots <= grid_per_xcd || p.line_weight > 0) queue = nullptr;  // every workgroup has exactly one item (or its part of a line)
    int* items = nullptr;
    if (queue && plan.items_bytes > 0 && ws_bytes >= plan.total()) items = (int*)(ws + plan.total() - plan.cast_bytes - plan.items_bytes);
    // Equal-length sequences (every one as long as max_seq_len allows): dealing the items with a fixed stride is
    // perfectly balanced and keeps all workgroups of an XCD on the same (sequence, head) pair at the same time,
    // which measures 4-5 % faster than the counter; any other batch needs the counter for balance.
    if (a->delta_size == 0 && a->total_kv == (int64_t)a->batch * a->max_seq_len) {
        queue = nullptr;
        // ... and (the caller's contract: no sequence is longer than max_seq_len) sequence b is rows b * max_seq_len
        // onwards: the kernels need neither the offsets nor a ranking by length
        p.uniform = 1;
        order = nullptr;
    }

    // ahead of the forward kernel: sequence ranking and / or the start value of the work-item counters; where work lists are built, the
    // kernel that builds them does both (up to a number of sequences)
    const bool plan_ranks = items && queue && (!order || a->batch <= hstu::kPlanRank);
    if (!plan_ranks && (order || queue)) {
        const int blocks = order ? (a->batch + 3) / 4 : 1;
        hipLaunchKernelGGL(hstu::hstu_prep_kernel, dim3(blocks), dim3(256), 0, stream, a->seq_offsets, a->seq_offsets_i64,
                           a->batch, order, queue, grid_per_xcd);
        hipError_t e = hipGetLastError();
        if (e != hipSuccess) {
            set_last_error("prep kernel launch", e);
            return HSTU_ERR_LAUNCH;
        }
    }
    p.order = plan_ranks ? nullptr : order;  // (the lists name the sequences)
    p.queue = queue;
    if (items && queue) {
        // the lists are 32-byte records behind everything else in the workspace; align them
        items = (int*)((reinterpret_cast<uintptr_t>(items) + 31) & ~(uintptr_t)31);
        p.items_cap = (int)slots;
        hipLaunchKernelGGL(hstu::hstu_plan_kernel, dim3(8), dim3(HSTU_PLAN_THREADS), 0, stream, p, bm, 64, queue + 8 * 16, items,
                           plan_ranks && order ? 1 : 0, queue, grid_per_xcd);
        hipError_t e = hipGetLastError();
        if (e != hipSuccess) {
            set_last_error("plan kernel launch", e);
            return HSTU_ERR_LAUNCH;
        }
        p.items = items;
        p.nitems = queue + 8 * 16;
    }

    // (after everything above: the block decode_work reads is made of copies)
    fill_decode_params(p);
    if (a->dtype == HSTU_FP32) return launch_mixed<hstu::Fp16F32>(p, a->dqk, a->dv, stream);
    if (a->dtype == HSTU_BF16) return launch_dim<hstu::Bf16>(p, a->dqk, a->dv, cfg, grid_per_xcd, a->total_q, stream);
    if (a->dtype == HSTU_FP16) return launch_dim<hstu::Fp16>(p, a->dqk, a->dv, cfg, grid_per_xcd, a->total_q, stream);
    return launch_dim<hstu::Fp8>(p, a->dqk, a->dv, cfg, grid_per_xcd, a->total_q, stream);
}

namespace {

// Per device, set up on the first call with that device current: the device address of `scratch` (each device holds
// its own copy of the array at its own address) and an event that marks the end of the last call that used the area.
struct NoallocState {
    void* scratch = nullptr;
    hipEvent_t done = nullptr;
    hipStream_t last_stream = nullptr;
    bool in_use = false;  // `done` has been recorded
};
std::mutex g_noalloc_mutex;

NoallocState* noalloc_state_of_current_device() {
    static NoallocState state[64];
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) return nullptr;
    NoallocState& st = state[dev];
    if (!st.scratch) {
        void* ptr = nullptr;
        hipError_t e = hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch));
        if (e != hipSuccess || !ptr) {
            set_last_error("hipGetSymbolAddress(scratch)", e);
            return nullptr;
        }
        e = hipEventCreateWithFlags(&st.done, hipEventDisableTiming);
        if (e != hipSuccess) {
            set_last_error("hipEventCreateWithFlags", e);
            return nullptr;
        }
        st.scratch = ptr;
    }
    return &st;
}

}  // namespace

int hstu_hip_mha_fwd_noalloc(const HstuFwdArgs* a, void* stream_) {
    g_last_error[0] = 0;
    int rc = hstu_hip_check_args(a);
    if (rc != HSTU_OK) return rc;
    if (a->total_q == 0 || a->batch == 0) return HSTU_OK;
    if (!current_device_is_gfx950()) return HSTU_ERR_BAD_DEVICE;
    const size_t need = make_plan(a, SIZE_MAX, false).total();  // (a line's partial sums may take more: it is cut where they fit)
    if (need > (size_t)HSTU_NOALLOC_SCRATCH_BYTES) {
        snprintf(g_last_error, sizeof(g_last_error), "this call would use %zu bytes of scratch memory; the fixed area holds %zu", need,
                 (size_t)HSTU_NOALLOC_SCRATCH_BYTES);
        return HSTU_ERR_SCRATCH_LIMIT;
    }
    hipStream_t stream = (hipStream_t)stream_;
    std::lock_guard<std::mutex> lock(g_noalloc_mutex);  // check, launch and record belong together
    NoallocState* st = noalloc_state_of_current_device();
    if (!st) return HSTU_ERR_LAUNCH;
    // A call on another stream while the last one has not finished would race on the area.  (Not under capture: an
    // event recorded into a graph cannot be queried, and a captured launch runs whenever the graph is replayed.)
    hipStreamCaptureStatus capture = hipStreamCaptureStatusNone;
    const bool capturing = hipStreamIsCapturing(stream, &capture) == hipSuccess && capture != hipStreamCaptureStatusNone;
    if (!capturing && st->in_use && st->last_stream != stream && hipEventQuery(st->done) == hipErrorNotReady) {
        snprintf(g_last_error, sizeof(g_last_error), "the scratch area of this device is in use by a call on another stream");
        return HSTU_ERR_BUSY;
    }
    HstuFwdArgs b = *a;
    b.workspace = st->scratch;  // the device address, never the array's name
    b.workspace_bytes = (int64_t)HSTU_NOALLOC_SCRATCH_BYTES;
    // Everything the kernels read from the area is written earlier in the same call (counters and ranking by the prep
    // kernel, work lists by the plan kernel, run counts and partial sums by the forward kernel), so what an earlier
    // call left behind is never looked at and nothing has to be cleared.
    rc = hstu_hip_mha_fwd(&b, stream_);
    if (rc == HSTU_OK && !capturing && hipEventRecord(st->done, stream) == hipSuccess) {
        st->last_stream = stream;
        st->in_use = true;
    }
    return rc;
}

}  // extern "C"

namespace {

// Largest power of two <= 16 that divides every value given (addresses, strides, row size).
int common_vector_bytes(std::initializer_list<uint64_t> values) {
    uint64_t all = 16;
    for (uint64_t v : values) all |= v;
    int vec = 1;
    while (vec < 16 && (all & vec) == 0) vec <<= 1;
    return vec;
}

constexpr int kJaggedRows = 32;  // rows per workgroup of the copy kernel
constexpr int64_t kShortRow = 1 << 26;           // accesses of a row up to which a block's are counted in 32 bits

int check_jagged_args(const HstuJaggedCopyArgs* a) {
    if (!a) return HSTU_ERR_NULL_POINTER;
    if (a->batch < 0 || a->row_bytes < 0 || a->max_len_left < 0 || a->max_len_right < 0 || a->total_left < 0 || a->total_right < 0)
        return HSTU_ERR_BAD_SHAPE;
    if (a->left_row_stride < a->row_bytes || a->right_row_stride < a->row_bytes || a->joined_row_stride < a->row_bytes)
        return HSTU_ERR_BAD_SHAPE;
    if (!a->offsets_left && a->total_left != (int64_t)a->batch * a->max_len_left) return HSTU_ERR_BAD_SHAPE;
    if (!a->offsets_right && a->total_right != (int64_t)a->batch * a->max_len_right) return HSTU_ERR_BAD_SHAPE;
    if (a->batch == 0 || a->row_bytes == 0 || a->total_left + a->total_right == 0) return HSTU_OK;
    if (!a->joined || (a->total_left > 0 && !a->left) || (a->total_right > 0 && !a->right)) return HSTU_ERR_NULL_POINTER;
    return HSTU_OK;
}

template <bool SPLIT>
int launch_jagged_copy(const HstuJaggedCopyArgs* a, hipStream_t stream) {
    g_last_error[0] = 0;
    int rc = check_jagged_args(a);
    if (rc != HSTU_OK) return rc;
    if (a->batch == 0 || a->row_bytes == 0 || a->total_left + a->total_right == 0) return HSTU_OK;
    hstu::JaggedCopyParams p;
    p.left = (char*)a->left;
    p.right = (char*)a->right;
    p.joined = (char*)a->joined;
    p.left_rs = a->left_row_stride;
    p.right_rs = a->right_row_stride;
    p.joined_rs = a->joined_row_stride;
    p.row_bytes = a->row_bytes;
    p.offsets_left = a->offsets_left;
    p.offsets_right = a->offsets_right;
    p.offsets_left_i64 = a->offsets_left_i64;
    p.offsets_right_i64 = a->offsets_right_i64;
    p.batch = a->batch;
    p.max_len_left = a->max_len_left;
    p.max_len_right = a->max_len_right;
    const long long rows = (long long)a->max_len_left + a->max_len_right;
    const long long gx = (rows + kJaggedRows - 1) / kJaggedRows;
    if (gx <= 0) return HSTU_OK;
    if (gx > 0x7fffffffLL || a->batch > 65535) return HSTU_ERR_BAD_SHAPE;  // grid.y limit
    const dim3 grid((unsigned)gx, (unsigned)a->batch);
    const int vec = common_vector_bytes({(uint64_t)(uintptr_t)a->left, (uint64_t)(uintptr_t)a->right, (uint64_t)(uintptr_t)a->joined,
                                         (uint64_t)a->left_row_stride, (uint64_t)a->right_row_stride,
                                         (uint64_t)a->joined_row_stride, (uint64_t)a->row_bytes});
    // (rows of more bytes than that, counted in 64 bits and copied byte by byte, took 17 times as long: 8 rows of 64 MB + 32 bytes 611 ms, so 35)
#define HSTU_COPY_LAUNCH(V)                                                                                                      \
    do {                                                                                                                         \
        if (a->row_bytes / V > kShortRow)                                                                                        \
            hipLaunchKernelGGL((hstu::hstu_jagged_copy_kernel<SPLIT, V, kJaggedRows, uint64_t>), grid, dim3(256), 0, stream, p); \
        else                                                                                                                     \
            hipLaunchKernelGGL((hstu::hstu_jagged_copy_kernel<SPLIT, V, kJaggedRows, unsigned>), grid, dim3(256), 0, stream, p); \
    } while (0)
    switch (vec) {
        case 16: HSTU_COPY_LAUNCH(16); break;
        case 8: HSTU_COPY_LAUNCH(8); break;
        case 4: HSTU_COPY_LAUNCH(4); break;
        case 2: HSTU_COPY_LAUNCH(2); break;
        default: HSTU_COPY_LAUNCH(1); break;
    }
#undef HSTU_COPY_LAUNCH
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) {
        set_last_error("jagged copy kernel launch", e);
        return HSTU_ERR_LAUNCH;
    }
    return HSTU_OK;
}

}  // namespace

extern "C" {

int hstu_hip_concat_2d_jagged(const HstuJaggedCopyArgs* a, void* stream) { return launch_jagged_copy<false>(a, (hipStream_t)stream); }

int hstu_hip_split_2d_jagged(const HstuJaggedCopyArgs* a, void* stream) { return launch_jagged_copy<true>(a, (hipStream_t)stream); }

int hstu_hip_jagged_write_tail(void* joined, int64_t joined_row_stride, const void* offsets, int32_t offsets_i64, const void* tail,
                               int64_t tail_row_stride, int64_t row_bytes, int32_t batch, int32_t tail_len, void* stream_) {
    g_last_error[0] = 0;
    if (batch < 0 || tail_len < 0 || row_bytes < 0 || joined_row_stride < row_bytes || tail_row_stride < row_bytes) return HSTU_ERR_BAD_SHAPE;
    if (batch == 0 || tail_len == 0 || row_bytes == 0) return HSTU_OK;
    if (!joined || !offsets || !tail) return HSTU_ERR_NULL_POINTER;
    if (batch > 65535) return HSTU_ERR_BAD_SHAPE;
    hipStream_t stream = (hipStream_t)stream_;
    const int vec = common_vector_bytes({(uint64_t)(uintptr_t)joined, (uint64_t)(uintptr_t)tail, (uint64_t)joined_row_stride,
                                         (uint64_t)tail_row_stride, (uint64_t)row_bytes});
    // Rows per workgroup: 16 where they are two accesses or more of every thread (rows of 512 bytes), 32 of shorter rows, and the tail divided evenly:
    // 20 rows as 16 and 4 took longer than one workgroup with all of them (1000 sequences of 20 rows of 1 KB 8.7 us, undivided 6.6, as 10 and 10
    // 6.1; 256 sequences of 20 rows of 32 bytes, 16 per workgroup 2.06, 32 1.96).
    const int most = row_bytes / vec >= 32 ? 16 : 32;
    const int64_t blocks = ((int64_t)tail_len + most - 1) / most;
    const int rows = (int)((tail_len + blocks - 1) / blocks);
    const dim3 grid((unsigned)blocks, (unsigned)batch);
#define HSTU_TAIL_KERNEL(V, INDEX)                                                                                            \
    hipLaunchKernelGGL((hstu::hstu_jagged_write_tail_kernel<V, INDEX>), grid, dim3(256), 0, stream, (char*)joined,   \
                       joined_row_stride, offsets, offsets_i64, rows, (const char*)tail, tail_row_stride, row_bytes, tail_len)
#define HSTU_TAIL_LAUNCH(V)                                           \
    do {                                                              \
        if (row_bytes / V > kShortRow) HSTU_TAIL_KERNEL(V, uint64_t); \
        else HSTU_TAIL_KERNEL(V, unsigned);                           \
    } while (0)
    switch (vec) {
        case 16: HSTU_TAIL_LAUNCH(16); break;
        case 8: HSTU_TAIL_LAUNCH(8); break;
        case 4: HSTU_TAIL_LAUNCH(4); break;
        case 2: HSTU_TAIL_LAUNCH(2); break;
        default: HSTU_TAIL_LAUNCH(1); break;
    }
#undef HSTU_TAIL_KERNEL
#undef HSTU_TAIL_LAUNCH
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) {
        set_last_error("jagged write-tail kernel launch", e);
        return HSTU_ERR_LAUNCH;
    }
    return HSTU_OK;
}

}  // extern "C"
