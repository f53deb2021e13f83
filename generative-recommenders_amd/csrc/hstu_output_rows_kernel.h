// The output step for a few hundred rows, in one kernel (gfx950):
//
//     out[r, n] = x[r, n] + sum_k joined[r, k] * W[k, n],   joined = [u' | attn | y],  y = act(u) * norm(attn)
// (hstu_compute_output of the reference, ops/hstu_compute.py:107-170).
//
// For many rows the step is the norm-multiply kernel and a GEMM of its own.  For a serving micro-batch that is two launches, a matrix
// written and read, and a library call whose host time is more than the kernels'.  Here a workgroup owns 32 rows x 32 columns (few enough that 50 rows are 32 workgroups, each reading 96 KB
// of W).  Its four waves make the 32 rows of `joined` together (a row across the lanes, 8 rows per wave) and leave them in LDS,
// rounded as the matrix would be; then each multiplies a quarter of the depth, with W's tiles in a ring of its own, so that the serial chain
// is short and there is no barrier until the four partial sums are added, in a fixed order, with the residual.
// 3 x 512 into 512 columns, us on the GPU and of the host's call, the two kernels -> this one: 50 rows 10.4 and 13.5 -> 7.7 and 3.4, 256 rows 11.9 and
// 13.7 -> 7.9 and 3.2.  What is left is latency: the launch, its instructions (ACT: u goes through an activation; without those of that 7.7 -> 7.5, one row 7.6 -> 7.25, 384 columns of u 7.4 -> 7.0), the
// rows from memory, their statistics.  (All of W that the LDS holds asked for at once, and the residual at the start, gained nothing: 7.9.)
#pragma once
#include "hstu_common.h"
#include "hstu_rows.h"

namespace hstu {

struct OutputRowsParams {
    NormMulParams nm;  // `joined` unused; no dropout
    const char* x;     // [rows, n]
    int64_t x_rs;
    const char* w;     // [k, n] row-major
    char* out;         // [rows, n] dense
    int n, k;          // k = blocks * d, a multiple of 128
};

constexpr int kOutRowsTile = 32 * 32 * 2;   // a W tile: 32 k x 32 columns
constexpr int kOutRowsRing = 6;             // tiles in a wave's ring
constexpr int kOutRowsMostK = 1536;         // the rows of `joined` and the rings share the LDS
constexpr int kOutRowsSumRow = 32 * 4 + 16; // a row of partial sums
constexpr int out_rows_lds(int k) { return 4 * kOutRowsRing * kOutRowsTile + 32 * k * 2; }
static_assert(4 * 32 * kOutRowsSumRow <= 4 * kOutRowsRing * kOutRowsTile, "the partial sums take the place of the rings");

template <class TT, bool GROUP, bool ACT>
__global__ __launch_bounds__(256, 1) void hstu_output_rows_kernel(const OutputRowsParams p) {
    typedef typename TT::vec8 vec8;
    typedef typename TT::elem elem;
    typedef __attribute__((ext_vector_type(4))) elem elem4;
    constexpr int RING = kOutRowsRing;
    extern __shared__ __attribute__((aligned(1024))) char smem[];
    const NormMulParams& nm = p.nm;

    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int g = lane >> 5, l32 = lane & 31;
    const int64_t row0 = (int64_t)blockIdx.y * 32;
    const int col0 = (int)blockIdx.x * 32;
    const int ntiles = p.k >> 7, first_tile = wave * ntiles;  // this wave's quarter of the depth

    // ---- the rows' operands (rows past the end repeat the last one)
    const int chunks = nm.d >> 3;  // at most 64
    const bool holds = lane < chunks;
    vec8 av[8], uv[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) {
        int64_t r = row0 + wave * 8 + i;
        r = r < nm.rows ? r : nm.rows - 1;
        av[i] = vec8{}, uv[i] = vec8{};
        if (holds) {
            av[i] = *(const vec8*)(nm.attn + (r * nm.attn_rs + lane * 8) * 2);
            uv[i] = *(const vec8*)(nm.u + (r * nm.u_rs + lane * 8) * 2);
        }
    }
    float w[8], b[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) w[j] = b[j] = 0.f;
    if (holds) {
        if constexpr (GROUP) {
            const int head = lane / nm.group_lanes;
#pragma unroll
            for (int j = 0; j < 8; ++j) w[j] = (float)((const elem*)nm.weight)[head], b[j] = (float)((const elem*)nm.bias)[head];
        } else {
            const vec8 wv = *(const vec8*)(nm.weight + lane * 16), bv = *(const vec8*)(nm.bias + lane * 16);
#pragma unroll
            for (int j = 0; j < 8; ++j) w[j] = (float)wv[j], b[j] = (float)bv[j];
        }
    }

    // ---- copies of W's tiles: 16 k rows of 64 bytes per instruction
    unsigned coff[2];
#pragma unroll
    for (int i = 0; i < 2; ++i) coff[i] = (unsigned)(i * 16 + lane / 4) * (unsigned)(p.n * 2) + (lane & 3) * 16;
    auto slot_at = [&](int slot) __attribute__((always_inline)) { return smem + (slot * 4 + wave) * kOutRowsTile; };
    auto issue = [&](int t, int slot) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < 2; ++i) global_load_lds16_soff(p.w + ((int64_t)(first_tile + t) * 32 * p.n + col0) * 2, coff[i], slot_at(slot) + i * 1024);
    };
#pragma unroll
    for (int t = 0; t < RING - 1; ++t)
        if (t < ntiles) issue(t, t);

    // ---- the rows of `joined`
    char* const panel = smem + 4 * RING * kOutRowsTile;
    const int pitch = p.k * 2;
    const float inv_n = GROUP ? 1.0f / (float)(nm.group_lanes * 8) : 1.0f / (float)nm.d;
    // sums over the lanes of a row (of a head), the eight rows side by side: one after the other, through LDS, they took 4 of the kernel's 10 us
    auto row_sums = [&](float (&s)[8]) __attribute__((always_inline)) {
        const int lanes = GROUP ? nm.group_lanes : 64;
#define HSTU_LEVEL(distance, add)                                  \
    if (lanes > distance) {                                        \
        _Pragma("unroll") for (int i = 0; i < 8; ++i) s[i] = add(s[i]); \
    }
        HSTU_LEVEL(1, add_dpp<0xB1>)   // quad_perm [1, 0, 3, 2]
        HSTU_LEVEL(2, add_dpp<0x4E>)   // quad_perm [2, 3, 0, 1]
        HSTU_LEVEL(4, add_dpp<0x141>)  // row_half_mirror: the other quad of 8, whose lanes agree
        HSTU_LEVEL(8, add_dpp<0x140>)  // row_mirror: the other 8 of 16
        HSTU_LEVEL(16, add_xor16)
        HSTU_LEVEL(32, add_xor32)
#undef HSTU_LEVEL
    };
    auto put = [&](int row, int column, const vec8& v) __attribute__((always_inline)) {  // a chunk of 8, swizzled as 16 rows' reads of it want
        *HSTU_LDS(vec8, panel + row * pitch + (((column >> 3) ^ (row & 15)) * 16)) = v;
    };
    float mean[8], sq[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) {
        mean[i] = 0.f;
#pragma unroll
        for (int j = 0; j < 8; ++j) mean[i] += (float)av[i][j];
    }
    row_sums(mean);
#pragma unroll
    for (int i = 0; i < 8; ++i) {
        mean[i] *= inv_n;
        sq[i] = 0.f;
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            const float dv = (float)av[i][j] - mean[i];
            sq[i] += dv * dv;
        }
        if (!holds) sq[i] = 0.f;
    }
    row_sums(sq);
#pragma unroll
    for (int i = 0; i < 8; ++i) {
        const float rstd = __builtin_amdgcn_rsqf(sq[i] * inv_n + nm.eps);
        vec8 y, ucopy = uv[i];
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            const float uf = (float)uv[i][j];
            float mul = uf;
            if constexpr (ACT) {
                const float sg = sigmoid_f(uf), us = uf * sg;
                if constexpr (GROUP) {
                    if (nm.silu_u) mul = us;
                } else {
                    if (nm.mul_act == HSTU_MUL_U_SIGMOID) mul = sg;
                    if (nm.mul_act == HSTU_MUL_U_SILU) mul = us;
                }
                if (nm.silu_u) ucopy[j] = (elem)us;
            }
            y[j] = (elem)(mul * (((float)av[i][j] - mean[i]) * rstd * w[j] + b[j]));
        }
        const int row = wave * 8 + i;
        if (holds) {
            if (nm.off_u >= 0) put(row, nm.off_u + lane * 8, ucopy);
            if (nm.off_x >= 0) put(row, nm.off_x + lane * 8, av[i]);
            put(row, nm.off_y + lane * 8, y);
        }
    }
    __syncthreads();

    // ---- the products: A = W^T (transposing reads), B = the rows of `joined`
    int waddr[2];
    {
        const int i16 = lane & 15, half = (lane >> 4) & 1, jrow = i16 >> 2, q4 = i16 & 3;
#pragma unroll
        for (int sec = 0; sec < 2; ++sec) waddr[sec] = (8 * g + 4 * sec + jrow) * 64 + (2 * half + (q4 >> 1)) * 16 + (q4 & 1) * 8;
    }
    vec8 wf[2], jf[2];
    auto load_ops = [&](int t, int slot, int kk) __attribute__((always_inline)) {
        const char* tile = slot_at(slot) + kk * 16 * 64;
        wf[kk] = read_vt_operand<TT>(tile + waddr[0], tile + waddr[1]);
        // (past the last tile: the last one's rows again, which nothing uses)
        const int c = ((first_tile + (t < ntiles ? t : ntiles - 1)) * 4 + 2 * kk + g) ^ (l32 & 15);
        jf[kk] = *HSTU_LDS(const vec8, panel + l32 * pitch + c * 16);
    };
    f32x16_t acc[2];
#pragma unroll
    for (int r = 0; r < 16; ++r) acc[0][r] = acc[1][r] = 0.f;
    if (ntiles >= RING - 1) asm volatile("s_waitcnt vmcnt(%0)" : : "n"(2 * (RING - 2)) : "memory");
    else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    load_ops(0, 0, 0);
    load_ops(0, 0, 1);
    int slot = 0;
    for (int t = 0; t < ntiles; ++t) {
        const int next = slot + 1 == RING ? 0 : slot + 1, before = slot == 0 ? RING - 1 : slot - 1;
        // the next tile has landed: at most the copies of the RING - 3 behind it are outstanding
        if (t + RING - 2 < ntiles) asm volatile("s_waitcnt vmcnt(%0)" : : "n"(2 * (RING - 3)) : "memory");
        else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
#pragma unroll
        for (int kk = 0; kk < 2; ++kk) {
            __builtin_amdgcn_sched_barrier(0);
            acc[kk] = TT::mfma(wf[kk], jf[kk], acc[kk]);
            load_ops(t + 1, next, kk);
        }
        __builtin_amdgcn_sched_barrier(0);
        if (t + RING - 1 < ntiles) issue(t + RING - 1, before);  // (the tile before this one: its operands have been multiplied)
        slot = next;
    }
    // ---- the four partial sums, the residual
    __syncthreads();  // nobody reads or fills a ring any more
    char* const sums = smem + wave * 32 * kOutRowsSumRow;
#pragma unroll
    for (int r4 = 0; r4 < 4; ++r4) {
        f32x4_t s;
#pragma unroll
        for (int j = 0; j < 4; ++j) s[j] = acc[0][r4 * 4 + j] + acc[1][r4 * 4 + j];
        *HSTU_LDS(f32x4_t, sums + l32 * kOutRowsSumRow + (r4 * 8 + g * 4) * 4) = s;
    }
    __syncthreads();
    const int row = threadIdx.x >> 3, c4 = (threadIdx.x & 7) * 4;
    const int64_t r = row0 + row;
    if (r >= nm.rows) return;
    const elem4 xv = *(const elem4*)(p.x + (r * p.x_rs + col0 + c4) * 2);
    f32x4_t s = *HSTU_LDS(const f32x4_t, smem + row * kOutRowsSumRow + c4 * 4);
#pragma unroll
    for (int k = 1; k < 4; ++k) s += *HSTU_LDS(const f32x4_t, smem + (k * 32 + row) * kOutRowsSumRow + c4 * 4);
    elem4 o;
#pragma unroll
    for (int j = 0; j < 4; ++j) o[j] = (elem)(s[j] + (float)xv[j]);
    *(elem4*)(p.out + (r * p.n + col0 + c4) * 2) = o;
}

}  // namespace hstu
