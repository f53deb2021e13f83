// The fused producer of hstu_uqvk_kernel.h for d_model 256, 384, 512 with 64 rows per wave.
//
// With 32 rows per wave every MFMA reads its 1 KB A operand from LDS, which is all the LDS can deliver, and the epilogue of
// a column block adds to the matrix phase.  Here a wave keeps 64 normalised rows in registers (256 of its 512; one
// workgroup of 4 waves per CU), an operand read from LDS feeds two MFMAs, and the epilogue of a column block of 64 runs piece
// by piece behind the MFMAs of the next one, from a second set of accumulators: a step of two MFMAs keeps the matrix pipe busy
// for 64 cycles, in which the wave issues the operand reads of a later step, one copy instruction, and one piece of the epilogue.
//
// W comes in tiles of 128 k x 64 n (16 KB, a ring, issued a column block ahead: stores lie between the copies, and a wait for a copy waits for them too).  The barrier of a tile stands four steps
// before its end, where the first operands of the next tile are requested.  Copies and stores count in one counter,
// in order: rows past the end repeat the last row down to the store (the same bits to the same place), so that the number of
// stores in flight is known wherever a copy is waited for.
//
// The work, row blocks of 256 x column blocks of 64, is one line that is cut into equal parts, one per CU; a part that crosses
// into the next row block normalises that block's rows too (12 us, three column blocks' time: 6000 vector instructions and the wait for HBM).
//
// 139264 rows of d_model 512 into 2048 columns: 408 -> 329 us (0.89 PFLOP/s); 300000 rows into 4096 columns 1593 -> 1249 us
// (1.01 PFLOP/s; a large library product reaches 1.36); 524288 rows into 2048 columns 1.20 ms, the matrix pipe busy 56 % of the
// cycles (SQ_VALU_MFMA_BUSY_CYCLES / 4 SQ_BUSY_CU_CYCLES).  On the way: the barrier without a
// wait for LDS reads 347 -> 329, no branches inside a column block and column blocks in turned order (see below) 65536 rows into
// 4096 columns 364 -> 292; the addresses of the stores computed where they are used (no spills, whose reloads wait for all
// copies) and the e4m3 copy in halves behind the store: the 8-bit layer of 16 sequences of 4096 .. 16384 rows 1.013 -> 1.064 of its
// former speed.  What is left: the rows' preparation, which nothing overlaps, 8 % of the time (with other rows of the matrix prepared
// first, as a measurement, 1.20 -> 1.31 ms at 524288 rows), and the column blocks themselves, where the matrix pipe is idle for 39 % of it.
#pragma once
#include <type_traits>
#include <utility>

#include "hstu_uqvk_kernel.h"

namespace hstu {

constexpr int kWideRows = 256, kWideCols = 64, kWideTileK = 128;
constexpr int kWideSlot = kWideTileK * kWideCols * 2;  // one W tile
constexpr int kWideStage = 32 * kUqvkStageRow;          // 32 rows of a wave
constexpr int kWideBias = 4 * 128;                      // bias values of four consecutive column blocks
// the copies run one column block (KT / 2 tiles) ahead
template <int KT>
constexpr int kWideRing = KT / 2 + 2;
template <int KT>
constexpr int kWideLds = kWideRing<KT> * kWideSlot + kWideBias + 4 * 2 * kWideStage;

// When the epilogue of the previous column block does what, in steps of the S a column block has.
template <int S>
struct WideSchedule {
    static constexpr int at(int x) { return x * S / 64; }
    static constexpr int piece(int i) { return at(3 + 11 * i / 4); }  // 16 pieces, eight per 32 rows: bias, SiLU, rounding, staging
    static constexpr int read(int i) { return at((i < 4 ? 25 : 47 - 12) + 3 * i); }  // 8: a store's rows out of the staging area
    static constexpr int store(int i) { return at((i < 4 ? 29 : 51 - 12) + 3 * i); }
    static constexpr int convert(int i, int half) { return at((i < 4 ? 30 : 52 - 12) + 3 * i + half); }  // the e4m3 copy, behind the store
    static constexpr int stores_in(int first, int last) {
        int n = 0;
        for (int i = 0; i < 8; ++i) n += store(i) >= first && store(i) <= last;
        return n;
    }
};

// At most N of the wave's copies and stores are outstanding, then the barrier.  LDS reads may be: a copy goes into the slot of the tile
// before the previous one, whose operands every wave has multiplied before the barrier that precedes the copy.
template <int N>
__device__ __forceinline__ void wide_barrier() {
    asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" : : "n"(N) : "memory");
}

template <class F, int... I>
__device__ __forceinline__ void wide_for(F&& f, std::integer_sequence<int, I...>) {
    (f(std::integral_constant<int, I>{}), ...);
}

template <class TT, int KT, int MODE>  // KT = d_model / 64; MODE: not kUqvkGradU
__global__ __launch_bounds__(256, 1) void hstu_uqvk_wide_kernel(const UqvkFusedParams p) {
    typedef typename TT::vec8 vec8;
    typedef typename TT::elem elem;
    typedef __attribute__((ext_vector_type(4))) elem elem4;
    constexpr bool OUT8 = MODE == kUqvkForward8, TRANS = MODE == kProductT;
    constexpr int KS = KT * 4, TPB = KT / 2, S = 16 * TPB, PD = 4, RING = kWideRing<KT>;
    typedef WideSchedule<S> Plan;
    extern __shared__ __attribute__((aligned(1024))) char smem[];

    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int g = lane >> 5, l32 = lane & 31;
    const int nblk = p.n_out / kWideCols;
    // this workgroup's part of the line of units
    const int extra = p.units - p.units_per_wave * (int)gridDim.x;  // parts that are one unit longer
    int unit = (int)blockIdx.x * p.units_per_wave + ((int)blockIdx.x < extra ? (int)blockIdx.x : extra);
    const int unit_end = unit + p.units_per_wave + ((int)blockIdx.x < extra ? 1 : 0);

    // copy instruction i of this wave brings rows (wave + 4 i) * 8 + lane / 8 of a tile, physical chunk lane % 8
    unsigned coff[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        if constexpr (TRANS) {  // 64 columns' rows of 256 bytes
            const int row = (wave + 4 * i) * 4 + (lane >> 4);
            coff[i] = (unsigned)row * (unsigned)(p.w_rs * 2) + ((lane & 15) ^ (row & 15)) * 16;
        } else {
            const int row = (wave + 4 * i) * 8 + (lane >> 3);
            coff[i] = (unsigned)row * (unsigned)(p.w_rs * 2) + ((lane & 7) ^ swz_w64(row)) * 16;
        }
    }
    // transposing reads: lane supplies the address of 4 consecutive n of k row 8g + 4sec + j (+ 16 per k step)
    int waddr[2][2];
    {
        const int i16 = lane & 15, half = (lane >> 4) & 1, jrow = i16 >> 2, q4 = i16 & 3;
#pragma unroll
        for (int sec = 0; sec < 2; ++sec) {
            const int row = 8 * g + 4 * sec + jrow;
#pragma unroll
            for (int dt = 0; dt < 2; ++dt) waddr[sec][dt] = row * 128 + (((dt * 4 + 2 * half + (q4 >> 1)) ^ swz_w64(row)) * 16) + (q4 & 1) * 8;
        }
    }
    int taddr[8];  // (transposed W: the lane's column, chunk 2 k step + g)
#pragma unroll
    for (int k = 0; k < 8; ++k) taddr[k] = l32 * 256 + (((2 * k + g) ^ (l32 & 15)) * 16);
    char* const stage = smem + RING * kWideSlot + kWideBias + wave * 2 * kWideStage;
    const int chunk = lane & 7, rsub = lane >> 3;  // 8 lanes cover one row's 128 bytes, 8 rows per store
    float amax[3] = {0.f, 0.f, 0.f};                 // (e4m3 output) the largest |value| this lane has stored of v, q, k

    while (unit < unit_end) {
        const int rb = __builtin_amdgcn_readfirstlane(unit / nblk);
        const int c_begin = unit - rb * nblk;
        const int n = unit_end - unit < nblk - c_begin ? unit_end - unit : nblk - c_begin;  // column blocks of this row block
        unit += n;
        const int64_t row0 = (int64_t)rb * kWideRows + wave * 64;  // first row of the wave

        // The c-th column block in the order of this workgroup.  The lines of a W tile and of a block's stores lie a row of W or of the
        // output apart, which is a multiple of the interleave of the L2's channels, so the 32 workgroups of an XCD start at different
        // blocks: in step they would all be on one channel.
        const int turn = (int)(blockIdx.x >> 3) * n / 32 % n;
        auto col_of = [&](int c) __attribute__((always_inline)) { return (c_begin + (c + turn < n ? c + turn : c + turn - n)) * kWideCols; };
        // ---- copies: tile kt of column block c into ring slot s, one instruction of the four at a time; past the last block that one's
        // tiles again, into slots nobody reads
        const int64_t tile_bytes = TRANS ? kWideTileK * 2 : (int64_t)kWideTileK * p.w_rs * 2;
        auto issue = [&](int c, int kt, int s, int i) __attribute__((always_inline)) {
            const char* src = p.w + (int64_t)col_of(c < n ? c : n - 1) * 2 * (TRANS ? p.w_rs : 1) + kt * tile_bytes;
            // (block c's bias is read at the start of block c + 1, before the copies of block c + 4 are issued)
            if (!TRANS && i == 0 && kt == 0 && wave == 0 && lane < 8 && c < n)
                global_load_lds16(p.bias + (int64_t)col_of(c) * 2 + lane * 16, smem + RING * kWideSlot + (c & 3) * 128);
            global_load_lds16_soff(src, coff[i], smem + __builtin_amdgcn_readfirstlane(s * kWideSlot + (wave + 4 * i) * 1024));
        };
#pragma unroll
        for (int t = 0; t < TPB; ++t)
#pragma unroll
            for (int i = 0; i < 4; ++i) issue(0, t, t, i);

        vec8 xreg[2][KS];
#pragma unroll
        for (int rg = 0; rg < 2; ++rg) {
            if constexpr (TRANS) {
                int64_t r = row0 + rg * 32 + l32;
                r = r < p.rows ? r : p.rows - 1;
#pragma unroll
                for (int ks = 0; ks < KS; ++ks) xreg[rg][ks] = *(const vec8*)(p.x + (r * p.x_rs + ks * 16 + 8 * g) * 2);
            } else {
                uqvk_normalised_row<TT, KS, true>(p, row0 + rg * 32 + l32, g, xreg[rg]);
            }
            // all of it here: the compiler would otherwise move the arithmetic of the second half into the first column block
#pragma unroll
            for (int ks = 0; ks < KS; ++ks) asm volatile("" : "+a"(xreg[rg][ks]));
            __builtin_amdgcn_sched_barrier(0);
        }

        // where this lane's stores go: rows past the end are the last row
        const int64_t base_row = row0 < p.rows ? row0 : p.rows - 1;
        char* const obase = p.out + base_row * p.out_rs * 2;
        unsigned char* const obase8 = OUT8 ? p.out8 + base_row * (p.n_out - p.n_silu) : nullptr;
        const int64_t below = p.rows - 1 - base_row;
        const int last = below < 63 ? (int)below : 63;
        // (computed where it is used: hoisted out of the loop, the addresses of all stores take registers that the rows need)
        auto orow = [&](int i) __attribute__((always_inline)) {
            int r = rsub;
            asm volatile("" : "+v"(r));
            return (unsigned)(i * 8 + r < last ? i * 8 + r : last);
        };

        f32x16_t acc[2][2][2];  // [set][row group][32 columns]
        elem4 b4[2][4];
        i32x4_t rd[8];
        float blockmax = 0.f;  // (e4m3 output) the largest |value| of the column block in progress
        auto read_bias = [&](int c) __attribute__((always_inline)) {
            if constexpr (TRANS) return;
            const char* b = smem + RING * kWideSlot + (c & 3) * 128 + g * 8;
#pragma unroll
            for (int dt = 0; dt < 2; ++dt)
#pragma unroll
                for (int r4 = 0; r4 < 4; ++r4) b4[dt][r4] = *HSTU_LDS(const elem4, b + dt * 64 + r4 * 16);
        };
        // the epilogue of column block c, whose sums are in `sums`
        auto piece = [&](int i, const f32x16_t(&sums)[2][2], auto Silu) __attribute__((always_inline)) {
            const int rg = i >> 3, dt = (i >> 2) & 1, r4 = i & 3;
            float v[4];
#pragma unroll
            for (int j = 0; j < 4; ++j) v[j] = TRANS ? sums[rg][dt][r4 * 4 + j] : sums[rg][dt][r4 * 4 + j] + (float)b4[dt][r4][j];
            if constexpr (decltype(Silu)::value) {
#pragma unroll
                for (int j = 0; j < 4; ++j) v[j] = v[j] * __builtin_amdgcn_rcpf(1.0f + __builtin_amdgcn_exp2f(-1.4426950408889634f * v[j]));
            }
            elem4 o;
            if constexpr (TRANS) o = round_sums<elem>(v);
            else o = round_to<elem>(v);
            *HSTU_LDS(elem4, stage + rg * kWideStage + l32 * kUqvkStageRow + (dt * 32 + r4 * 8 + g * 4) * 2) = o;
        };
        auto read_rows = [&](int i) __attribute__((always_inline)) {
            rd[i] = *HSTU_LDS(const i32x4_t, stage + (i >> 2) * kWideStage + ((i & 3) * 8 + rsub) * kUqvkStageRow + chunk * 16);
        };
        auto store_rows = [&](int i, int c) __attribute__((always_inline)) {
            const int col0 = col_of(c);
            *(i32x4_t*)(obase + (int64_t)col0 * 2 + (orow(i) * (unsigned)(p.out_rs * 2) + chunk * 16)) = rd[i];
        };
        // The rounded values of store i once more, scaled, as e4m3, in two halves (a step of two MFMAs has
        // room for about twelve vector instructions): 8 lanes cover 64 bytes of a row.
        int half8[2];
        auto convert8 = [&](int i, int h, int c) __attribute__((always_inline)) {
            const int col0 = col_of(c);
            const int tensor = col0 < 2 * p.n_silu ? 0 : col0 < 2 * p.n_silu + p.n_attn ? 1 : 2;
            const float is = p.inv_scale[tensor];
            const vec8 e = __builtin_bit_cast(vec8, rd[i]);
            float f[4];
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const float x = (float)e[4 * h + j];
                blockmax = __builtin_fmaxf(blockmax, __builtin_fabsf(x));
                f[j] = __builtin_fminf(__builtin_fmaxf(x * is, -448.0f), 448.0f);
            }
            int v = 0;
            v = __builtin_amdgcn_cvt_pk_fp8_f32(f[0], f[1], v, false);
            v = __builtin_amdgcn_cvt_pk_fp8_f32(f[2], f[3], v, true);
            half8[h] = v;
            if (h == 1) {
                typedef __attribute__((ext_vector_type(2))) int i32x2_t;
                *(i32x2_t*)(obase8 + (col0 - p.n_silu) + (orow(i) * (unsigned)(p.n_out - p.n_silu) + chunk * 8)) = i32x2_t{half8[0], half8[1]};
                if (i == 7) {
                    amax[0] = tensor == 0 ? __builtin_fmaxf(amax[0], blockmax) : amax[0];
                    amax[1] = tensor == 1 ? __builtin_fmaxf(amax[1], blockmax) : amax[1];
                    amax[2] = tensor == 2 ? __builtin_fmaxf(amax[2], blockmax) : amax[2];
                    blockmax = 0.f;
                }
            }
        };

        // ---- operands: op m of a tile = (k step, 32 columns) = (m / 2, m % 2), requested PD steps ahead
        int slot = 0;  // of the tile in progress
        vec8 fr[PD];
        auto load_op = [&](int s, int m) __attribute__((always_inline)) {
            if constexpr (TRANS) {
                fr[m % PD] = *HSTU_LDS(const vec8, smem + s * kWideSlot + (m & 1) * 8192 + taddr[m >> 1]);
                return;
            }
            const char* b = smem + s * kWideSlot + (m >> 1) * 16 * 128;
            fr[m % PD] = read_vt_operand<TT>(b + waddr[0][m & 1], b + waddr[1][m & 1]);
        };
        wide_barrier<(TPB - 1) * 4>();  // the first tile is there
#pragma unroll
        for (int m = 0; m < PD; ++m) load_op(0, m);

        // Column block c into `now`, the epilogue of block c - 1 out of `before`.
        // Silu: whether that goes through SiLU.
        auto block = [&](f32x16_t(&now)[2][2], const f32x16_t(&before)[2][2], int c, auto Prev, auto Silu) __attribute__((always_inline)) {
            constexpr bool PREV = decltype(Prev)::value;
#pragma unroll
            for (int rg = 0; rg < 2; ++rg)
#pragma unroll
                for (int dt = 0; dt < 2; ++dt)
#pragma unroll
                    for (int r = 0; r < 16; ++r) now[rg][dt][r] = 0.f;
            if constexpr (PREV) read_bias(c - 1);
            wide_for([&](auto Kt) __attribute__((always_inline)) {
                constexpr int kt = decltype(Kt)::value;
                const int next = slot + 1 == RING ? 0 : slot + 1, prev2 = slot >= 2 ? slot - 2 : slot + TPB;  // RING = TPB + 2
#pragma unroll
                for (int m = 0; m < 16; ++m) {
                    const int s = kt * 16 + m;
                    if (m == 16 - PD) {
                        // The next tile's copies were issued in steps 1 .. 10 of the tile TPB - 1 before this one.  Behind them are the copies of
                        // the tiles since, four each, and this block's stores since then (those of the block before this one
                        // are not counted, nor is an e4m3 copy's: the wait is longer than it had to be).
                        wide_barrier<4 * (TPB - 1) + (PREV ? Plan::stores_in(16 * (kt - (TPB - 1)) + 11, 16 * kt + 11) : 0)>();
                    }
                    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                    for (int rg = 0; rg < 2; ++rg) now[rg][m & 1] = TT::mfma(fr[m % PD], xreg[rg][kt * 8 + (m >> 1)], now[rg][m & 1]);
                    if (m + PD < 16) load_op(slot, m + PD);
                    else load_op(next, m + PD - 16);
                    if constexpr (PREV) {
#pragma unroll
                        for (int i = 0; i < 16; ++i)
                            if (Plan::piece(i) == s) piece(i, before, Silu);
#pragma unroll
                        for (int i = 0; i < 8; ++i)
                            if (Plan::read(i) == s) read_rows(i);
#pragma unroll
                        for (int i = 0; i < 8; ++i)
                            if (Plan::store(i) == s) store_rows(i, c - 1);
                        if constexpr (OUT8 && !decltype(Silu)::value) {
#pragma unroll
                            for (int i = 0; i < 8; ++i)
#pragma unroll
                                for (int h = 0; h < 2; ++h)
                                    if (Plan::convert(i, h) == s) convert8(i, h, c - 1);
                        }
                    }
                    if (m < 12 && m % 3 == 1) issue(c + 1, kt, prev2, m / 3);
                }
                slot = next;
            }, std::make_integer_sequence<int, TPB>{});
            __builtin_amdgcn_sched_barrier(0);
        };
        auto finish = [&](const f32x16_t(&sums)[2][2], int c, auto Silu) __attribute__((always_inline)) {
            read_bias(c);
#pragma unroll
            for (int i = 0; i < 16; ++i) piece(i, sums, Silu);
#pragma unroll
            for (int i = 0; i < 8; ++i) read_rows(i);
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                store_rows(i, c);
                if constexpr (OUT8 && !decltype(Silu)::value) convert8(i, 0, c), convert8(i, 1, c);
            }
        };

        auto next_block = [&](f32x16_t(&now)[2][2], const f32x16_t(&before)[2][2], int c) __attribute__((always_inline)) {
            if (!TRANS && col_of(c - 1) < p.n_silu) block(now, before, c, std::true_type{}, std::true_type{});
            else block(now, before, c, std::true_type{}, std::false_type{});
        };
        auto last_epilogue = [&](const f32x16_t(&sums)[2][2], int c) __attribute__((always_inline)) {
            if (!TRANS && col_of(c) < p.n_silu) finish(sums, c, std::true_type{});
            else finish(sums, c, std::false_type{});
        };
        block(acc[0], acc[1], 0, std::false_type{}, std::false_type{});
        int c = 1;
        for (; c + 1 < n; c += 2) {
            next_block(acc[1], acc[0], c);
            next_block(acc[0], acc[1], c + 1);
        }
        if (c < n) {
            next_block(acc[1], acc[0], c);
            last_epilogue(acc[1], c);
        } else {
            last_epilogue(acc[0], c - 1);
        }
        // the copies past the end have landed and every wave has read its last operands before the ring is filled anew (or given back)
        asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
    }
    if constexpr (OUT8) {
#pragma unroll
        for (int t = 0; t < 3; ++t) {
            float m = amax[t];
#pragma unroll
            for (int d = 32; d >= 1; d >>= 1) m = __builtin_fmaxf(m, __shfl_xor(m, d, 64));
            if (lane == 0 && m > 0.f) atomicMax(p.absmax + t, __builtin_bit_cast(unsigned, m));
        }
    }
}

}  // namespace hstu
