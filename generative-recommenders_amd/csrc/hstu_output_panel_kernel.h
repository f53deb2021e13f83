// The output step in one kernel, for more rows than hstu_output_rows_kernel.h takes (gfx950):
//
//     out[r, n] = x[r, n] + sum_k joined[r, k] * W[k, n],   joined = [u | attn | y],  y = u * norm(attn)
// (hstu_compute_output of the reference, ops/hstu_compute.py:107-170).
//
// A workgroup of NW waves owns RB blocks of 32 rows and 32 NW columns.  Its waves read the rows of u and attn once (a row across D / 8 lanes) and
// keep them in registers, y beside them; block after block of `joined` goes from there into LDS (the panel), rounded as the matrix would be, and every
// wave multiplies it with its own 32 columns of W, whose tiles come through a private ring: barriers stand only where the panel changes.  The order of
// all sums is that of the norm-multiply kernel and of the GEMM behind it (hstu_output_kernel.h): in bf16 the results are theirs bit for bit (in fp16 the
// compiler rounds y's last product once here and twice there, or the other way round).
//
// Against the norm-multiply kernel and a GEMM (the library's), us on the GPU: 3 x 512 into 512 columns, 500 rows 13.1 -> 8.9, 2000 rows 19.9 -> 11.6,
// 8192 rows 31.9 -> 20.8; 3 x 256 with group norm into 256, 14200 rows 27.1 -> 13.7; 3 x 128 into 256, 400000 rows 330 -> 161.  What bounds it (8192 rows
// of 3 x 512, 256 workgroups of 64 x 256; parts left out one at a time): launch, rows, residual and result 9.7, y 2, the products 6.2, W's copies 4 on top
// (786 KB per CU at 41 B/clk, the rate of a wave's copy instructions; rows of 128 instead of 64 bytes do not change it).  The norm is made once per
// column block: from some width and rows on the norm-multiply kernel and a GEMM are faster again (output_panel_form).
#pragma once
#include "hstu_common.h"
#include "hstu_rows.h"

namespace hstu {

struct OutputPanelParams {
    NormMulParams nm;  // `joined` unused; no dropout, no activation of u
    const char* x;     // [rows, n]
    int64_t x_rs;
    const char* w;     // [blocks * D, n] row-major
    char* out;         // [rows, n] dense
    int n;             // a multiple of 32 NW
};

template <int D, int RB, int NW>
struct OutputPanel {
    static constexpr int kRows = RB * 32, kCols = NW * 32;
    static constexpr int kTile = 16 * 32 * 2;                          // a W tile: 16 k x 32 columns, one copy instruction
    static constexpr int kPanel = kRows * D * 2;
    // tiles in a wave's ring: what two workgroups per CU leave of the LDS, 8 at most
    static constexpr int kRing = kPanel + NW * 8 * kTile <= 80 * 1024 ? 8 : NW == 8 ? 8 : 4;
    static constexpr int kAhead = kRing / 2;                           // steps between asking for operands and their products
    static constexpr int kSumRow = kCols * 4 + 16;                     // a row of sums on their way to the stores
    static constexpr int kLds = kPanel + NW * kRing * kTile > kRows * kSumRow ? kPanel + NW * kRing * kTile : kRows * kSumRow;
};

// Which form takes a call, -1: none.  What counts is the XCD that gets most workgroups: row blocks go to the eight in turn, each with all its column blocks (3 x 512 into 1536 columns,
// 1341 rows, 504 workgroups of 32 x 128, 72 of them on one XCD: 27.7 us, as two rounds, where 64 are one; the library 23.0).  32 x 128 while two of its workgroups per CU hold all of it (us, against
// 64 x 256: 3 x 512 into 512 columns, 4000 rows 15.7 / 17.6, 6000 rows 23.1 / 18.5; 3 x 256 into 256, 8192 rows 10.5 / 11.6, 10000 rows 12.9 / 12.3), then the larger ones, whose W is read by fewer.
// They pay as long as the norm, made once per column block, costs less than a matrix written and read (us, the two kernels / this one):
//   width 128: to a d_out of 1152 at any rows: 400000 rows into 1024 columns 693 / 566
//   width 256: into 512 columns at any rows (200000: 294 / 273), into 1024 16384 rows 51 / 48, 32768 rows 87 / 91; where d_out is no multiple of 256 the
//     two kernels are slower: 60000 rows into 640 columns 167 / 108, into 1152 206 / 181
//   width 384, 512: a round of the CUs, and up to 768 columns the most of a second one, half of it into 1024 (256 columns, 32768 rows 62 / 51, 33000 rows 62 / 65; 512 columns, 16384 rows 50 / 42, 24000 rows 65 / 61, 32000
//     rows 80 / 81; 768 columns, 5440 rows, 33 workgroups on an XCD, 32.2 / 34.7, 6140 rows 48 / 35, 10877 rows, 66 of them, 42 / 51; 1024 columns, 6143 rows 47 / 36, 7040 rows, 56 of them, 36.5 / 41.0, 12000 rows 57 / 61; 1536 columns,
//     2690 rows, 36 on an XCD, 28.4 / 35.9, 4670 rows 35.9 / 37.3; 2048 columns, 3072 rows 31.7 / 37.5), in fp16, where the library is faster, the first round (512 columns, 9000 rows 34 / 38); where
//     d_out is no multiple of 256 only the small form fits: into 384 columns 8000 rows 33 / 26, 12000 rows 38 / 38; into 640 4000 rows 32 / 25, 6000 rows 29 / 32
enum { kPanel32x128 = 0, kPanel64x128 = 1, kPanel64x256 = 2 };
inline int output_panel_form(int64_t rows, int d, int n, bool bf16) {
    const int64_t small = ((rows + 31) / 32 + 7) / 8 * (n / 128), large = ((rows + 63) / 64 + 7) / 8 * (n / 256);  // on one XCD of 32 CUs
    if (small <= 64) return kPanel32x128;
    const bool whole = n % 256 == 0;
    if (d <= 256) {
        if (n > 1152 || (d == 256 && whole && n > 512 && rows * n > (16 << 20))) return -1;
        return whole ? kPanel64x256 : kPanel64x128;
    }
    if (!whole) return n <= 384 && small <= 96 ? kPanel32x128 : -1;
    const bool second = (bf16 || n == 256) && n <= 1024;
    return large <= 32 || (second && large >= 36 && large <= (n > 768 ? 48 : 64)) ? kPanel64x256 : -1;
}

// The form for the rows at the end of another kernel's call, at most a round of the 64 x 256 workgroups (n a multiple of 256).
inline int output_panel_tail_form(int64_t rows, int n) { return (rows + 31) / 32 * (n / 128) <= 512 ? kPanel32x128 : kPanel64x256; }

template <class TT, bool GROUP, int D, int RB, int NW>
__global__ __launch_bounds__(NW * 64, 2) void hstu_output_panel_kernel(const OutputPanelParams p) {
    typedef typename TT::vec8 vec8;
    typedef typename TT::elem elem;
    typedef OutputPanel<D, RB, NW> Geo;
    constexpr int CH = D / 8;                       // chunks of a row
    constexpr int LPR = D > 256 ? 64 : D / 8;       // lanes that a row lies across (384: the last 16 of 64 idle)
    constexpr int RPI = 64 / LPR;                   // rows a wave handles at a time
    constexpr int IT = Geo::kRows / NW / RPI;       // ... and how often
    constexpr int RING = Geo::kRing, STEPS = D / 16, AHEAD = Geo::kAhead;
    static_assert(Geo::kRows % (NW * RPI) == 0 && STEPS % RING == 0 && D % 128 == 0 && D <= 512, "whole rings per block, rows dealt evenly");
    extern __shared__ __attribute__((aligned(1024))) char smem[];
    const NormMulParams& nm = p.nm;

    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int g = lane >> 5, l32 = lane & 31;
    // the column blocks of a row block are workgroups 8 apart: on one XCD, one after the other, all but the first find the rows in its L2
    const unsigned ncb = (unsigned)p.n / Geo::kCols;
    const unsigned octet = blockIdx.x / (8 * ncb), within = blockIdx.x - octet * (8 * ncb);
    const int64_t row0 = ((int64_t)octet * 8 + (within & 7)) * Geo::kRows;
    if (row0 >= nm.rows) return;
    const int col0 = (int)(within >> 3) * Geo::kCols;

    // ---- the rows (those past the end repeat the last one)
    const int chunk = lane % LPR, rsub = lane / LPR;
    const bool holds = LPR * 8 == D || chunk < CH;
    vec8 av[IT], uv[IT];
#pragma unroll
    for (int i = 0; i < IT; ++i) {
        int64_t r = row0 + (wave * IT + i) * RPI + rsub;
        r = r < nm.rows ? r : nm.rows - 1;
        av[i] = vec8{}, uv[i] = vec8{};
        if (holds) {
            av[i] = *(const vec8*)(nm.attn + (r * nm.attn_rs + chunk * 8) * 2);
            uv[i] = *(const vec8*)(nm.u + (r * nm.u_rs + chunk * 8) * 2);
        }
    }
    vec8 wv = {}, bv = {};
    if (holds) {
        if constexpr (GROUP) {
            const int head = chunk / nm.group_lanes;
            wv[0] = ((const elem*)nm.weight)[head], bv[0] = ((const elem*)nm.bias)[head];
        } else {
            wv = *(const vec8*)(nm.weight + chunk * 16), bv = *(const vec8*)(nm.bias + chunk * 16);
        }
    }

    // ---- copies of W's tiles: 16 k rows of 64 bytes
    char* const ring = smem + Geo::kPanel + wave * RING * Geo::kTile;
    const unsigned coff = (unsigned)(lane >> 2) * (unsigned)(p.n * 2) + (lane & 3) * 16;
    const int blocks = 1 + (nm.off_u >= 0) + (nm.off_x >= 0);
    const unsigned wstep = 16u * (unsigned)p.n * 2;
    const i32x4_t wrsrc = make_buffer_rsrc(p.w, (unsigned)blocks * STEPS * wstep);
    unsigned wnext = (unsigned)(col0 + wave * 32) * 2;
    auto issue = [&](int slot) __attribute__((always_inline)) {  // (past the last tile: zeros, into a slot nobody reads)
        buffer_load_lds16(wrsrc, coff, wnext, ring + slot * Geo::kTile);
        wnext += wstep;
    };
#pragma unroll
    for (int t = 0; t < RING; ++t) issue(t);

    // ---- operand addresses
    int waddr[2];  // transposing reads of a W tile
    {
        const int i16 = lane & 15, half = (lane >> 4) & 1, jrow = i16 >> 2, q4 = i16 & 3;
#pragma unroll
        for (int sec = 0; sec < 2; ++sec) waddr[sec] = (8 * g + 4 * sec + jrow) * 64 + (2 * half + (q4 >> 1)) * 16 + (q4 & 1) * 8;
    }
    int paddr[8];  // a row of the panel, chunk 2 s + g of every 16, swizzled as 16 rows' reads of it want
#pragma unroll
    for (int s = 0; s < 8; ++s) paddr[s] = l32 * (D * 2) + (((2 * s + g) ^ (l32 & 15)) * 16);
    auto put = [&](int row, const vec8& v) __attribute__((always_inline)) {
        if (holds) *HSTU_LDS(vec8, smem + row * (D * 2) + ((chunk ^ (row & 15)) * 16)) = v;
    };
    // sums over the lanes of a row (of a head)
    auto row_sum = [&](float s) __attribute__((always_inline)) {
        const int lanes = GROUP ? nm.group_lanes : LPR;
        if constexpr (GROUP) {
            if (lanes > 1) s = add_dpp<0xB1>(s);    // quad_perm [1, 0, 3, 2]
            if (lanes > 2) s = add_dpp<0x4E>(s);    // quad_perm [2, 3, 0, 1]
            if (lanes > 4) s = add_dpp<0x141>(s);   // row_half_mirror: the other quad of 8, whose lanes agree
            if (lanes > 8) s = add_dpp<0x140>(s);   // row_mirror: the other 8 of 16
            if (LPR > 16 && lanes > 16) s = add_xor16(s);
            if (LPR > 32 && lanes > 32) s = add_xor32(s);
        } else {  // the furthest first, as the norm-multiply kernel adds; of 16 lanes, rotations by 8, 4, 2, 1
            if constexpr (LPR > 32) s = add_xor32(s);
            if constexpr (LPR > 16) s = add_xor16(s);
            s = add_dpp<0x128>(s);
            s = add_dpp<0x124>(s);
            s = add_dpp<0x122>(s);
            s = add_dpp<0x121>(s);
        }
        return s;
    };

    // ---- y, in groups of rows whose sums over the lanes go side by side.  The rows behind them stay packed meanwhile: left to itself the compiler keeps
    // all their fp32 conversions alive
    vec8 yv[IT];
    {
        const float inv_n = GROUP ? 1.0f / (float)(nm.group_lanes * 8) : 1.0f / (float)D;
        constexpr int G = IT < 4 ? IT : 4;
        float w[GROUP ? 1 : 8], b[GROUP ? 1 : 8];
#pragma unroll
        for (int j = 0; j < (GROUP ? 1 : 8); ++j) w[j] = (float)wv[j], b[j] = (float)bv[j];
#pragma unroll
        for (int i0 = 0; i0 < IT; i0 += G) {
#pragma unroll
            for (int i = i0; i < IT; ++i) asm volatile("" : "+v"(av[i]), "+v"(uv[i]));
            float v[G][8], mean[G], sq[G];
#pragma unroll
            for (int i = 0; i < G; ++i) {
                mean[i] = 0.f;
#pragma unroll
                for (int j = 0; j < 8; ++j) v[i][j] = (float)av[i0 + i][j], mean[i] += v[i][j];
            }
#pragma unroll
            for (int i = 0; i < G; ++i) mean[i] = row_sum(mean[i]) * inv_n;
#pragma unroll
            for (int i = 0; i < G; ++i) {
                sq[i] = 0.f;
#pragma unroll
                for (int j = 0; j < 8; ++j) v[i][j] -= mean[i], sq[i] += v[i][j] * v[i][j];
                if (!holds) sq[i] = 0.f;
            }
#pragma unroll
            for (int i = 0; i < G; ++i) sq[i] = row_sum(sq[i]);
#pragma unroll
            for (int i = 0; i < G; ++i) {
                const float rstd = __builtin_amdgcn_rsqf(sq[i] * inv_n + nm.eps);
#pragma unroll
                for (int j = 0; j < 8; ++j) yv[i0 + i][j] = (elem)((float)uv[i0 + i][j] * (v[i][j] * rstd * w[GROUP ? 0 : j] + b[GROUP ? 0 : j]));
                asm volatile("" : "+v"(yv[i0 + i]));
            }
        }
    }

    f32x16_t acc[RB];
#pragma unroll
    for (int rb = 0; rb < RB; ++rb)
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[rb][r] = 0.f;

    for (int blk = 0; blk < blocks; ++blk) {
        if (blk > 0) __syncthreads();  // the block before has been multiplied
        const int kind = blk == blocks - 1 ? 2 : (blk == 0 && nm.off_u >= 0) ? 0 : 1;  // u, attn, y
        if (kind == 0) {
#pragma unroll
            for (int i = 0; i < IT; ++i) put((wave * IT + i) * RPI + rsub, uv[i]);
        } else if (kind == 1) {
#pragma unroll
            for (int i = 0; i < IT; ++i) put((wave * IT + i) * RPI + rsub, av[i]);
        } else {
#pragma unroll
            for (int i = 0; i < IT; ++i) put((wave * IT + i) * RPI + rsub, yv[i]);
        }
        __syncthreads();

        // ---- the products: A = W^T (transposing reads), B = the panel's rows
        // operands are asked for AHEAD steps before their products: two waves of a SIMD hide less than the LDS takes
        vec8 wf[AHEAD], jf[AHEAD][RB];
        auto load_ops = [&](int s) __attribute__((always_inline)) {
            const char* tile = ring + (s % RING) * Geo::kTile;
            wf[s % AHEAD] = read_vt_operand<TT>(tile + waddr[0], tile + waddr[1]);
#pragma unroll
            for (int rb = 0; rb < RB; ++rb) jf[s % AHEAD][rb] = *HSTU_LDS(const vec8, smem + paddr[s % 8] + (s / 8) * 256 + rb * 32 * (D * 2));
        };
        asm volatile("s_waitcnt vmcnt(%0)" : : "n"(RING - AHEAD) : "memory");
#pragma unroll
        for (int s = 0; s < AHEAD; ++s) load_ops(s);
#pragma unroll
        for (int s = 0; s < STEPS; ++s) {
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int rb = 0; rb < RB; ++rb) acc[rb] = TT::mfma(wf[s % AHEAD], jf[s % AHEAD][rb], acc[rb]);
            __builtin_amdgcn_sched_barrier(0);
            issue(s % RING);  // (this tile's slot: its operands are in registers)
            if (s + AHEAD < STEPS) {
                // the tile AHEAD steps on has landed: the RING - AHEAD behind it may be on their way
                asm volatile("s_waitcnt vmcnt(%0)" : : "n"(RING - AHEAD) : "memory");
                load_ops(s + AHEAD);
            }
        }
    }

    // ---- the sums through LDS, the residual, whole rows out
    constexpr int CPR = Geo::kCols / 8, RPP = NW * 64 / CPR, PASSES = Geo::kRows / RPP;
    const int ochunk = threadIdx.x % CPR, orow = threadIdx.x / CPR;
    vec8 xr[PASSES];
#pragma unroll
    for (int i = 0; i < PASSES; ++i) {
        int64_t r = row0 + i * RPP + orow;
        r = r < nm.rows ? r : nm.rows - 1;
        xr[i] = *(const vec8*)(p.x + (r * p.x_rs + col0 + ochunk * 8) * 2);
    }
    asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" : : "n"(PASSES) : "memory");  // no copy is on its way, nobody reads the panel
#pragma unroll
    for (int rb = 0; rb < RB; ++rb)
#pragma unroll
        for (int r4 = 0; r4 < 4; ++r4) {
            f32x4_t s;
#pragma unroll
            for (int j = 0; j < 4; ++j) s[j] = acc[rb][r4 * 4 + j];
            *HSTU_LDS(f32x4_t, smem + (rb * 32 + l32) * Geo::kSumRow + (wave * 32 + r4 * 8 + g * 4) * 4) = s;
        }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < PASSES; ++i) {
        const int row = i * RPP + orow;
        const int64_t r = row0 + row;
        const f32x4_t lo = *HSTU_LDS(const f32x4_t, smem + row * Geo::kSumRow + ochunk * 32);
        const f32x4_t hi = *HSTU_LDS(const f32x4_t, smem + row * Geo::kSumRow + ochunk * 32 + 16);
        if (r < nm.rows) {
            vec8 o;
#pragma unroll
            for (int j = 0; j < 4; ++j) o[j] = (elem)(lo[j] + (float)xr[i][j]), o[4 + j] = (elem)(hi[j] + (float)xr[i][4 + j]);
            *(vec8*)(p.out + (r * p.n + col0 + ochunk * 8) * 2) = o;
        }
    }
}

}  // namespace hstu
