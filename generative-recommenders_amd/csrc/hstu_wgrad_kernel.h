// Gradient of a weight for gfx950:  out[m, n] = sum_r a[r, m] * b[r, n]  over the rows r of a batch, and on request the column
// sums of b (the gradient of the bias).
//
// The product is as deep as the batch is long (10^4 .. 10^6 rows) and its result is small (512 x 2048): tiles of the result alone
// leave most of the chip idle -- the library's choice for 57819 rows ran 32 workgroups and took 317 us, 0.38 PFLOP/s.  So the rows
// are cut into splits, one workgroup per (tile of 256 x 256, split); each writes its fp32 sums and a second kernel adds
// the splits in order (no atomics: the same bits from run to run) and rounds once.
//
// Both operands have the summed index along their rows, so both are read from LDS with transposing reads
// (ds_read_b64_tr_b16).  A workgroup of 8 waves, two per SIMD, walks its rows in tiles of 32: 256 columns of a and of b as two slabs
// of 128 columns each, 32 KB, in a ring of four, copied three tiles ahead with LDS-DMA through buffer descriptors (rows past the
// split's end arrive as zeros).  Wave (wm, wn) accumulates 64 x 128 of the tile in 2 x 4 MFMA blocks: six operands feed
// eight MFMAs, 0.75 KB of LDS reads per MFMA.  One barrier per tile, between its two 16-deep steps, with the operands of the step
// behind it already in registers.  What bounds it: the operand reads and copies next to the MFMAs, as in the output projection's kernel.
// Measured (kernel + reduce): 57819 rows, 512 x 2048: 138 us = 0.88 PFLOP/s where torch.mm takes 307; 300000 rows 577 us = 1.09
// PFLOP/s (1317); 706 rows, 256 x 768: 13 us (20).  The column sums cost 14 us at 57819 x 2048 (a pass of its own: 53 us).
#pragma once
#include <type_traits>

#include "hstu_common.h"
#include "hstu_uqvk_kernel.h"

namespace hstu {

struct WgradParams {
    const char* a;  // [rows, m]
    const char* b;  // [rows, n]
    unsigned a_rsb, b_rsb;  // row strides in bytes
    int m, n;
    int64_t rows;
    int rows_per_split;     // a multiple of 32; the host keeps rows_per_split * stride below 2^31
    int tiles_m, tiles_n, splits;
    float* partial;         // [splits][tile][256 * 256] in the order of the waves' accumulators
    float* colsum;          // NULL, or [splits][n]
};

constexpr int kWgTile = 256, kWgDepth = 32, kWgWaves = 8, kWgRing = 4;
constexpr int kWgSlab = kWgDepth * 128 * 2;      // 128 columns of one operand: 8 KB
constexpr int kWgSlot = 4 * kWgSlab;             // two slabs of a, two of b
constexpr int kWgLds = kWgRing * kWgSlot;
constexpr int kWgTileFloats = kWgTile * kWgTile;

// Row m and first of four columns n (inside the tile) of the four floats at position 4 * i of a tile's partial sums: wave, block of 32
// rows, block of 32 columns, group of 8 columns, lane -- the order in which the waves store their accumulators.
__host__ __device__ inline void wgrad_position(int i, int& m, int& n) {
    const int lane = i & 63, r4 = (i >> 6) & 3, nb = (i >> 8) & 3, mb = (i >> 10) & 1, wave = i >> 11;
    m = (wave >> 1) * 64 + mb * 32 + (lane & 31);
    n = (wave & 1) * 128 + nb * 32 + r4 * 8 + (lane >> 5) * 4;
}

// acc + the sum of eight elements: four dot products with (1, 1), accumulated in fp32.
template <class TT>
__device__ __forceinline__ float sum_of_8(typename TT::vec8 v, float acc) {
    typedef typename TT::elem elem;
    typedef __attribute__((ext_vector_type(2))) elem elem2;
    const elem2 one = {(elem)1.0f, (elem)1.0f};
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        const elem2 x = {v[2 * j], v[2 * j + 1]};
        if constexpr (std::is_same<TT, Bf16>::value) acc = __builtin_amdgcn_fdot2_f32_bf16(x, one, acc, false);
        else acc = __builtin_amdgcn_fdot2(x, one, acc, false);
    }
    return acc;
}

template <class TT>
__global__ __launch_bounds__(kWgWaves * 64, 2) void hstu_wgrad_kernel(const WgradParams p) {
    typedef typename TT::vec8 vec8;
    extern __shared__ __attribute__((aligned(1024))) char smem[];
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int g = lane >> 5;
    const int wm = wave >> 1, wn = wave & 1;
    // Workgroup ids go round-robin over the 8 XCDs: each XCD gets a contiguous run of (split, tile), so that the tiles of a split,
    // which read the same rows at the same time, find them in one L2.
    const int tiles = p.tiles_m * p.tiles_n;
    const int work = (int)(blockIdx.x & 7) * (int)(gridDim.x >> 3) + (int)(blockIdx.x >> 3);
    if (work >= tiles * p.splits) return;
    const int split = work / tiles, tile = work - split * tiles;
    const int tm = tile / p.tiles_n, tn = tile - tm * p.tiles_n;
    const int64_t r0 = (int64_t)split * p.rows_per_split;
    const int rows = (int)(p.rows - r0 < p.rows_per_split ? p.rows - r0 : p.rows_per_split);
    const int ntiles = (rows + kWgDepth - 1) / kWgDepth;

    // Copies: instruction i (0, 1) of this wave per operand brings rows 4 j .. 4 j + 3 of a slab, j = (wave + 8 i) % 8, slab = i.
    // A descriptor ends with the last row of the split that exists: what lies behind it arrives as zeros.  (Columns past m or n
    // of the last tile read whatever follows in the row or the next one, inside the descriptor: those sums are never stored.)
    const i32x4_t ra = make_buffer_rsrc(p.a + r0 * p.a_rsb + (int64_t)tm * kWgTile * 2,
                                        (unsigned)((int64_t)(rows - 1) * p.a_rsb + (p.m - tm * kWgTile) * 2));
    const i32x4_t rb = make_buffer_rsrc(p.b + r0 * p.b_rsb + (int64_t)tn * kWgTile * 2,
                                        (unsigned)((int64_t)(rows - 1) * p.b_rsb + (p.n - tn * kWgTile) * 2));
    const int crow = wave * 4 + (lane >> 4);
    const unsigned ccol = ((lane & 15) ^ swz_w(crow)) * 16;
    const unsigned aoff = (unsigned)crow * p.a_rsb + ccol, boff = (unsigned)crow * p.b_rsb + ccol;
    auto issue = [&](int i, int t, int slot) __attribute__((always_inline)) {  // i = 0 .. 3: slabs a0, a1, b0, b1
        char* dst = smem + slot * kWgSlot + i * kWgSlab + wave * 1024;
        if (i < 2) buffer_load_lds16(ra, aoff, (unsigned)t * (kWgDepth * p.a_rsb) + i * 256, dst);
        else buffer_load_lds16(rb, boff, (unsigned)t * (kWgDepth * p.b_rsb) + (i - 2) * 256, dst);
    };

    // transposing reads of a slab, as for the producer's weight tiles: 32 columns dt * 32 .. of rows 8 g + 4 sec + j (+ 16 ks)
    int addr[2][4];
    {
        const int i16 = lane & 15, half = (lane >> 4) & 1, jrow = i16 >> 2, q4 = i16 & 3;
#pragma unroll
        for (int sec = 0; sec < 2; ++sec) {
            const int row = 8 * g + 4 * sec + jrow;
#pragma unroll
            for (int dt = 0; dt < 4; ++dt) {
                const int chunk = dt * 4 + 2 * half + (q4 >> 1);
                addr[sec][dt] = row * 256 + ((chunk ^ swz_w(row)) * 16) + (q4 & 1) * 8;
            }
        }
    }
    int aaddr[2][2], baddr[2][4];  // this wave's: 64 columns of a (half of slab wm / 2), 128 of b (slab wn)
#pragma unroll
    for (int sec = 0; sec < 2; ++sec) {
#pragma unroll
        for (int mb = 0; mb < 2; ++mb) aaddr[sec][mb] = (wm >> 1) * kWgSlab + ((wm & 1) ? addr[sec][2 + mb] : addr[sec][mb]);
#pragma unroll
        for (int nb = 0; nb < 4; ++nb) baddr[sec][nb] = (2 + wn) * kWgSlab + addr[sec][nb];
    }

    f32x16_t acc[2][4];
#pragma unroll
    for (int mb = 0; mb < 2; ++mb)
#pragma unroll
        for (int nb = 0; nb < 4; ++nb)
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[mb][nb][r] = 0.f;
    // column sums: the four waves of a column half take one block of 32 columns each, in the first row of tiles only
    const bool sums = p.colsum != nullptr && tm == 0;
    float csum = 0.f;

    vec8 fa[2][2], fb[2][4];
    auto read_op = [&](int j, int slot, int ks, vec8(&a)[2], vec8(&b)[4]) __attribute__((always_inline)) {  // j = 0 .. 5
        const char* base = smem + slot * kWgSlot + ks * 16 * 256;
        if (j < 4) b[j] = read_vt_operand<TT>(base + baddr[0][j], base + baddr[1][j]);
        else a[j - 4] = read_vt_operand<TT>(base + aaddr[0][j - 4], base + aaddr[1][j - 4]);
    };
    auto column_sum = [&](const vec8(&b)[4]) __attribute__((always_inline)) {
        if (sums) csum = sum_of_8<TT>(wm == 0 ? b[0] : wm == 1 ? b[1] : wm == 2 ? b[2] : b[3], csum);
    };

#pragma unroll
    for (int t = 0; t < 3; ++t)
#pragma unroll
        for (int i = 0; i < 4; ++i) issue(i, t, t);
    asm volatile("s_waitcnt vmcnt(8)\n\ts_barrier" ::: "memory");
#pragma unroll
    for (int j = 0; j < 6; ++j) read_op(j, 0, 0, fa[0], fb[0]);

    // Tile t.  Step A multiplies its first 16 rows, reads the operands of step B and issues the copies of tile t + 3 into the slot of
    // tile t - 1 (nobody reads that any more since the barrier in tile t - 1); the barrier publishes tile t + 1 (behind its copies came
    // eight); step B multiplies the other 16 rows and reads the operands of tile t + 1.
    for (int t = 0; t < ntiles; ++t) {
        const int slot = t & (kWgRing - 1), slot1 = (t + 1) & (kWgRing - 1), slot3 = (t + 3) & (kWgRing - 1);
#pragma unroll
        for (int k = 0; k < 8; ++k) {
            const int mb = k >> 2, nb = k & 3;
            acc[mb][nb] = TT::mfma(fb[0][nb], fa[0][mb], acc[mb][nb]);
            __builtin_amdgcn_sched_barrier(0);
            if (k < 6) read_op(k, slot, 1, fa[1], fb[1]);
            if (k >= 4) issue(k - 4, t + 3, slot3);
            __builtin_amdgcn_sched_barrier(0);
        }
        column_sum(fb[0]);
        asm volatile("s_waitcnt vmcnt(8) lgkmcnt(0)\n\ts_barrier" ::: "memory");
#pragma unroll
        for (int k = 0; k < 8; ++k) {
            const int mb = k >> 2, nb = k & 3;
            acc[mb][nb] = TT::mfma(fb[1][nb], fa[1][mb], acc[mb][nb]);
            __builtin_amdgcn_sched_barrier(0);
            if (k < 6) read_op(k, slot1, 0, fa[0], fb[0]);
            __builtin_amdgcn_sched_barrier(0);
        }
        column_sum(fb[1]);
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // copies past the end (zeros) must land before the LDS is released

    float* out = p.partial + ((int64_t)split * tiles + tile) * kWgTileFloats + ((int64_t)wave * 2048 + lane) * 4;
#pragma unroll
    for (int mb = 0; mb < 2; ++mb)
#pragma unroll
        for (int nb = 0; nb < 4; ++nb)
#pragma unroll
            for (int r4 = 0; r4 < 4; ++r4) {
                f32x4_t v;
#pragma unroll
                for (int i = 0; i < 4; ++i) v[i] = acc[mb][nb][r4 * 4 + i];
                *(f32x4_t*)(out + (((mb * 4 + nb) * 4 + r4) * 64) * 4) = v;
            }
    if (sums) {
        csum += __shfl_xor(csum, 32, 64);
        const int col = tn * kWgTile + wn * 128 + wm * 32 + (lane & 31);
        if (g == 0 && col < p.n) p.colsum[(int64_t)split * p.n + col] = csum;
    }
}

// out = the splits' sums added in order, rounded once; four columns per thread.  The last workgroups add the column sums.
template <class E>
__global__ __launch_bounds__(256) void hstu_wgrad_reduce_kernel(const WgradParams p, E* out, E* colsum_out, int tile_blocks) {
    typedef __attribute__((ext_vector_type(4))) E elem4;
    const int tiles = p.tiles_m * p.tiles_n;
    if ((int)blockIdx.x >= tile_blocks) {
        const int c = ((int)blockIdx.x - tile_blocks) * 256 + threadIdx.x;
        if (c >= p.n) return;
        float s = 0.f;
        for (int k = 0; k < p.splits; ++k) s += p.colsum[(int64_t)k * p.n + c];
        colsum_out[c] = (E)s;
        return;
    }
    const int idx = blockIdx.x * 256 + threadIdx.x;
    const int tile = idx / (kWgTileFloats / 4), i = idx - tile * (kWgTileFloats / 4);
    int m, n;
    wgrad_position(i, m, n);
    m += (tile / p.tiles_n) * kWgTile, n += (tile % p.tiles_n) * kWgTile;
    if (m >= p.m || n >= p.n) return;
    const float* src = p.partial + (int64_t)tile * kWgTileFloats + (int64_t)i * 4;
    const int64_t pitch = (int64_t)tiles * kWgTileFloats;
    f32x4_t s = *(const f32x4_t*)src;
    int k = 1;
    for (; k + 4 <= p.splits; k += 4) {  // four loads in flight, added in order
        f32x4_t v[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) v[j] = *(const f32x4_t*)(src + (k + j) * pitch);
#pragma unroll
        for (int j = 0; j < 4; ++j) s += v[j];
    }
    for (; k < p.splits; ++k) s += *(const f32x4_t*)(src + k * pitch);
    elem4 o;
#pragma unroll
    for (int j = 0; j < 4; ++j) o[j] = (E)s[j];
    *(elem4*)(out + (int64_t)m * p.n + n) = o;
}

}  // namespace hstu
