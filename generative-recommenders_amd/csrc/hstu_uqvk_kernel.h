// Fused producer of q, k, v for gfx950: layer norm + projection + bias + SiLU(u) in one kernel.
//
//     out[r, n] = act( sum_k LN(x)[r, k] * W[k, n] + bias[n] ),   act = SiLU for n < n_silu, identity otherwise
// (hstu_compute_uqvk of the reference, ops/hstu_compute.py:54-104; LN with fp32 statistics and its result rounded to the
// input type, ops/pytorch/pt_layer_norm.py:24-39).
//
// The depth of this product (d_model, at most 512) is small enough for a wave to keep its normalised rows in registers:
// they are the B operand of every MFMA (lane = row, 8 consecutive k per 16-deep step); the normalised matrix never exists
// in memory.  W is read transposed (ds_read_b64_tr_b16) out of LDS as the A operand,
//     C^T[n, r] += W^T[n, k] . LN(x)^T[k, r]
// so that a lane ends up with one output row and, per 32-column block, four runs of four consecutive columns -- the
// accumulator layout of the attention kernels.
//
// Three kernels, with the same order of all sums, so that a row's bits do not depend on which one takes it (the choice: hstu_uqvk_launch.h):
//   * hstu_uqvk_rows_kernel, for the row counts that fill the chip once: there the time is latency, not products.  A workgroup's four
//     waves share the normalisation of its 32 or 64 rows (a row lies across the lanes, so that loads are whole rows and a wave does a
//     quarter of the arithmetic), hand the result over through LDS and then go their own ways: each walks column units of its own, with
//     W's tiles in a ring of its own, and there is no barrier any more.  The ring takes over the LDS of the rows once they are in registers.
//   * hstu_uqvk_fused_kernel, 128 rows per workgroup with shared tiles: several rounds of workgroups at d_model 384 and 512.
//   * hstu_uqvk_wide_kernel (hstu_uqvk_wide_kernel.h), 64 rows per wave: many rows.
//
// The first against the second (which had every size up to the third's), us, d_model 512 into 2048 columns: 50 rows 13.9 -> 6.5, 500 rows
// 15.9 -> 7.7, 2000 rows 17.9 -> 13.8, 8192 rows 36.6 -> 30.4, 16000 rows 58.9 -> 51.9; d_model 256 into 1024: 1000 rows 11.1 -> 5.2,
// 14200 rows 26.2 -> 18.1; d_model 128, where it has every size, into 2048: 24000 rows 49.2 -> 35.4, 131072 rows 183 -> 138, 600000 rows 864 -> 652;
// into 128: 131072 rows 22.8 -> 20.6, 600000 rows 85.5 -> 86.3.  What bounds it at 8192 rows of d_model 512 (256 workgroups, one
// per CU): the matrix products take 6.8 us of the 28, the wait for the rows and their norm 6, copying W (1 MB per CU; a copy
// instruction costs the wave some 25 cycles) 3 on top of the products, the epilogue, which nothing overlaps, 8.  A build with the epilogue under
// the next unit's products took 34 us there: the products then share the issue with it piece by piece.
#pragma once
#include <type_traits>

#include "hstu_common.h"

namespace hstu {

struct UqvkFusedParams {
    const char* x;
    int64_t x_rs;  // elements
    const char* norm_weight;
    const char* norm_bias;
    float eps;
    const char* w;     // [K, n_out] row-major (the product with a transposed matrix: [n_out, K])
    int64_t w_rs;      // its row stride in elements
    const char* bias;  // [n_out]
    char* out;         // [rows, n_out]
    int64_t out_rs;    // its row stride in elements
    const char* du;    // (gradient of u) [rows, n_out]
    int64_t du_rs;
    char* normed;      // (gradient of u) NULL, or where LN(x) goes: [rows, K] dense
    int64_t rows;
    int n_out;   // multiple of 128
    int n_silu;  // multiple of 32: columns [0, n_silu) go through SiLU
    int units_per_wave;  // column units that a wave walks; 128 rows per workgroup: column blocks of a workgroup; 64 rows per wave: units of one
    int units;           // (64 rows per wave) row blocks x column blocks of 64, of which a workgroup takes units_per_wave or one more
    // Optional second output: the v | q | k columns (those from n_silu on) once more as e4m3 bytes,
    // out8[r, n - n_silu] = e4m3(rounded out[r, n] * inv_scale[t]), t = 0 (v: the next n_silu columns), 1 (q: the next
    // n_attn), 2 (k: the rest), clamped to +-448; and the largest |rounded out| of each of the three, for the scales of
    // the next batch.  NULL = off.
    unsigned char* out8;  // [rows, n_out - n_silu] dense
    float inv_scale[3];
    unsigned* absmax;     // [3]: bit patterns of non-negative floats, raised with atomicMax (the caller zeroes them)
    int n_attn;           // multiple of 64
};

constexpr int kUqvkStageRow = 64 * 2 + 16;  // staging row: 64 outputs + pad

// N values rounded to E by instructions of the compiler's: for sums as the matrix instructions leave them.
template <class E, int N>
__device__ __forceinline__ auto round_sums(const float (&x)[N]) {
    typedef __attribute__((ext_vector_type(N))) E vec;
    vec r;
#pragma unroll
    for (int j = 0; j < N; ++j) r[j] = (E)x[j];
    return r;
}
// N values as they are in fp32, rounded to E.  (fp16: left to itself the compiler makes one rounding of the last operation and this one, in
// one kernel and not in the other.)  Results of vector instructions only: the hardware does not interlock a matrix result against a
// vector instruction's read, and the compiler does not count the wait states for reads inside an asm block.
template <class E, int N>
__device__ __forceinline__ auto round_to(const float (&x)[N]) {
    if constexpr (std::is_same<E, _Float16>::value) {
        typedef __attribute__((ext_vector_type(N))) E vec;
        typedef __attribute__((ext_vector_type(N / 2))) unsigned words;
        words w;
#pragma unroll
        for (int j = 0; j < N; j += 2) {
            unsigned o;
            asm("v_cvt_pk_f16_f32 %0, %1, %2" : "=v"(o) : "v"(x[j]), "v"(x[j + 1]));
            w[j / 2] = o;
        }
        return __builtin_bit_cast(vec, w);
    } else {
        return round_sums<E>(x);
    }
}

// The layer norm's arithmetic.  A row's bits must not depend on the batch, and the kernels for few and for many rows hold a row
// differently, so the order of its sums is fixed here: 8 consecutive elements in turn, then the chunks of 8 as a binary tree in which
// chunk 2 ks + g meets chunk 2 (ks ^ 1) + g first, then ks ^ 2, ..., and the two g last.
template <class V8>
__device__ __forceinline__ float ln_chunk_sum(const V8& x) {
    float s = (float)x[0];
#pragma unroll
    for (int j = 1; j < 8; ++j) s += (float)x[j];
    return s;
}
template <class V8>
__device__ __forceinline__ float ln_chunk_squares(const V8& x, float mean) {
    float s = 0.f;
#pragma unroll
    for (int j = 0; j < 8; ++j) {
        const float d = (float)x[j] - mean;
        s = __builtin_fmaf(d, d, s);
    }
    return s;
}
template <class V8, class E>
__device__ __forceinline__ V8 ln_chunk_apply(const V8& x, float mean, float rstd, const V8& w, const V8& b) {
    float o[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) o[j] = __builtin_fmaf(((float)x[j] - mean) * rstd, (float)w[j], (float)b[j]);
    return round_to<E>(o);
}
template <int K>
__device__ __forceinline__ float ln_mean(float sum) {
    float mean = sum * (1.0f / K);
    asm volatile("" : "+v"(mean));  // (rounded here, not folded into the subtractions)
    return mean;
}
template <int K>
__device__ __forceinline__ float ln_rstd(float sq, float eps) {
    return __builtin_amdgcn_rsqf(__builtin_fmaf(sq, 1.0f / K, eps));
}

// The tree over the KS chunks that a lane holds.
template <int KS, class F>
__device__ __forceinline__ float ln_tree(F&& leaf) {
    float t[6];
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
        float s = leaf(ks);
        int l = 0;
#pragma unroll
        for (; (ks >> l) & 1; ++l) s = t[l] + s;
        t[l] = s;
    }
    if constexpr (KS == 24) return add_xor32(t[4] + t[3]);
    else return add_xor32(t[KS == 32 ? 5 : KS == 16 ? 4 : 3]);
}
// The same tree where a lane holds one chunk: ks in the low bits of its number, g in bit 5.
template <int LANES>
__device__ __forceinline__ float ln_tree_lanes(float s) {
    s = add_dpp<0xB1>(s);  // quad_perm [1, 0, 3, 2]
    s = add_dpp<0x4E>(s);  // quad_perm [2, 3, 0, 1]
    s = add_dpp<0x141>(s);  // row_half_mirror: the other quad of 8, whose lanes agree
    if constexpr (LANES > 8) s = add_dpp<0x140>(s);  // row_mirror: the other 8 of 16
    if constexpr (LANES > 16) s = add_xor16(s);
    return add_xor32(s);
}

// Row r (rows past the end repeat the last one) through the layer norm, as the B operands of a lane: 8 consecutive k of every 16,
// from 8 g on; the two half-waves share the row.  The chunks' sums are pinned in their order: left to itself the compiler moves a tree's leaves
// so far apart that two loads wait until the others have been summed, and the operands end up in the register banks of W's.  LOADS_FIRST: no
// arithmetic among the loads, as the kernel with 64 rows per wave wants it.  Left to itself / so, us: the kernel with 128 rows per workgroup,
// d_model 512 into 256 columns, 100000 rows 66.5 / 65.1, into 512, 20000 rows 34.9 / 34.6; the one with 64 rows per wave, d_model 256 into
// 1024, 100000 rows 99.9 / 96.2.
template <class TT, int KS, bool LOADS_FIRST>
__device__ __forceinline__ void uqvk_normalised_row(const UqvkFusedParams& p, int64_t r, int g, typename TT::vec8 (&xr)[KS]) {
    typedef typename TT::vec8 vec8;
    typedef typename TT::elem elem;
    constexpr int K = KS * 16;
    r = r < p.rows ? r : p.rows - 1;
    const char* xp = p.x + (r * p.x_rs + 8 * g) * 2;
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) xr[ks] = *(const vec8*)(xp + ks * 32);
    if constexpr (LOADS_FIRST) asm volatile("" : : : "memory");
    const float mean = ln_mean<K>(ln_tree<KS>([&](int ks) __attribute__((always_inline)) {
        float sum = ln_chunk_sum(xr[ks]);
        asm volatile("" : "+v"(sum));
        return sum;
    }));
    // the rows stay packed between the passes: without this the compiler keeps all their fp32 conversions alive
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) asm volatile("" : "+v"(xr[ks]));
    const float rstd =
        ln_rstd<K>(ln_tree<KS>([&](int ks) __attribute__((always_inline)) {
                       float sum = ln_chunk_squares(xr[ks], mean);
                       asm volatile("" : "+v"(sum));
                       return sum;
                   }),
                   p.eps);
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) asm volatile("" : "+v"(xr[ks]));
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
        const vec8 wv = *(const vec8*)(p.norm_weight + (ks * 16 + 8 * g) * 2);
        const vec8 bv = *(const vec8*)(p.norm_bias + (ks * 16 + 8 * g) * 2);
        xr[ks] = ln_chunk_apply<vec8, elem>(xr[ks], mean, rstd, wv, bv);
    }
}

// Chunk swizzle of a W tile (rows of 128 bytes = 8 chunks): the rows 8g + 4sec + j of a transposing read lie in different
// 64-byte bank groups (odd rows by the pitch, row bit 1 -> chunk bit 2), the two half-waves in different halves of a group
// (row bit 3 -> chunk bit 1).
__device__ __forceinline__ int swz_w64(int row) { return (((row >> 1) & 1) << 2) | (((row >> 3) & 1) << 1); }

constexpr int kUqvkMostUnits = 16;  // column units that a wave walks at most

// Geometry of the kernel for RB blocks of 32 rows per workgroup and column units of NB.
template <int KT, int RB, int NB>
struct UqvkRows {
    static constexpr int K = KT * 64;
    static constexpr int kPerCu = KT * RB <= 8 ? 2 : 1;             // workgroups per CU: what the rows leave of the registers
    static constexpr int kTile = 32 * NB * 2;                       // a W tile: 32 k of a unit
    static constexpr int kRing = 8;                                 // tiles in a wave's ring
    static constexpr int kPanel = RB * 32 * K * 2;                  // the normalised rows
    static constexpr int kEarly = kRing - kPanel / (4 * kTile);     // ring slots beside them
    static constexpr int kStageRow = NB * 2 + 16;
    static constexpr int kStage = 32 * kStageRow;                   // of a wave
    static constexpr int kBias = 4 * kRing * kTile + 4 * kStage;    // offset of the bias values of the workgroup's columns
    static_assert(kPanel % (4 * kTile) == 0 && kEarly >= 2, "the rows take whole slots of all four rings and leave some");
    static constexpr int lds(int units_per_wave) { return kBias + units_per_wave * 4 * NB * 2; }
};

// What the kernel computes from its products.
//   kUqvkForward, kUqvkForward8: the producer, without and with the e4m3 copy
//   kUqvkGradU: out = du * SiLU'(LN(x) W + bias), the gradient of the u columns' products, and LN(x) itself, an operand of W's gradient; nothing of the
//     forward is read but x
//   kProductT: out = x W^T, no norm, no bias: W's k run along its rows, so its tiles are read as they lie
enum { kUqvkForward, kUqvkForward8, kUqvkGradU, kProductT };

template <class TT, int KT, int RB, int NB, int MODE>  // KT = d_model / 64
__global__ __launch_bounds__(256, (UqvkRows<KT, RB, NB>::kPerCu)) void hstu_uqvk_rows_kernel(const UqvkFusedParams p) {
    typedef typename TT::vec8 vec8;
    typedef typename TT::elem elem;
    typedef __attribute__((ext_vector_type(4))) elem elem4;
    typedef UqvkRows<KT, RB, NB> Geo;
    constexpr bool OUT8 = MODE == kUqvkForward8, BIAS = MODE != kProductT, TRANS = MODE == kProductT;
    constexpr int K = Geo::K, KS = K / 16, DT = NB / 32, RING = Geo::kRing, TILES = K / 32;  // TILES: of a unit
    constexpr int COPIES = Geo::kTile / 1024, RPC = 1024 / (NB * 2), CH = NB / 8;             // copies of a tile, k rows of a copy, chunks of a k row
    extern __shared__ __attribute__((aligned(1024))) char smem[];

    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int g = lane >> 5, l32 = lane & 31;
    const int64_t row0 = (int64_t)blockIdx.x * (RB * 32);
    // Units: number (y units_per_wave + i) 4 + w is the i-th of wave w in workgroup y of a row block, as far as there are columns.  All lines of a
    // unit's W tiles lie a row of W apart, often a multiple of the interleave of the L2's channels: the workgroups of an XCD start at
    // different ones of their units.
    const int left = (p.n_out / NB - wave + 3) / 4 - (int)blockIdx.y * p.units_per_wave;
    const int units = left < 0 ? 0 : left < p.units_per_wave ? left : p.units_per_wave;
    const int ntiles = units * TILES;
    const int turn = units > 0 ? (int)(blockIdx.x >> 3) % units : 0;
    const int col0_wg = (int)blockIdx.y * p.units_per_wave * 4 * NB;  // first column of the workgroup
    auto col_of = [&](int u) __attribute__((always_inline)) {
        const int i = u + turn < units ? u + turn : u + turn - units;
        return col0_wg + (i * 4 + wave) * NB;
    };

    // ---- the rows, a quarter for each wave: a row lies across LANES x 2 lanes
    constexpr int LANES = KS <= 8 ? 8 : KS <= 16 ? 16 : 32, RPI = 32 / LANES, NP = RB * 8 / RPI;  // rows per instruction, instructions
    const int ks_of = lane & (LANES - 1), sub = l32 / LANES;
    const int chunk_of = 2 * ks_of + g;
    const bool holds = KS == LANES || ks_of < KS;
    vec8 xv[NP], wv, bv;
#pragma unroll
    for (int i = 0; i < NP; ++i) {
        int64_t r = row0 + (wave * NP + i) * RPI + sub;
        r = r < p.rows ? r : p.rows - 1;
        xv[i] = vec8{};
        if (holds) xv[i] = *(const vec8*)(p.x + (r * p.x_rs + chunk_of * 8) * 2);
    }
    wv = vec8{}, bv = vec8{};
    if (MODE != kProductT && holds) wv = *(const vec8*)(p.norm_weight + chunk_of * 16), bv = *(const vec8*)(p.norm_bias + chunk_of * 16);
    if constexpr (BIAS) {  // the bias values of the workgroup's columns
        const int cols = p.units_per_wave * 4 * NB;
        for (int c = threadIdx.x * 8; c < cols; c += 256 * 8) {
            if (col0_wg + c < p.n_out) *HSTU_LDS(vec8, smem + Geo::kBias + c * 2) = *(const vec8*)(p.bias + (int64_t)(col0_wg + c) * 2);
        }
    }

    // ---- copies: tile t of this wave = 32 k of one of its units; slot s of its ring
    unsigned coff[COPIES];
#pragma unroll
    for (int i = 0; i < COPIES; ++i) {
        if constexpr (TRANS) {  // NB rows of 64 bytes, swizzled for 16 rows' reads of one chunk
            const int row = i * 16 + lane / 4, c = (lane & 3) ^ ((row >> 2) & 3);
            coff[i] = (unsigned)row * (unsigned)(p.w_rs * 2) + (unsigned)(c * 16);
        } else {
            const int row = i * RPC + lane / CH, c = lane % CH;
            coff[i] = (unsigned)row * (unsigned)(p.w_rs * 2) + (unsigned)((NB == 64 ? c ^ swz_w64(row) : c) * 16);
        }
    }
    auto slot_at = [&](int slot) __attribute__((always_inline)) { return smem + (slot * 4 + wave) * Geo::kTile; };
    auto issue_one = [&](int t, int slot, int i) __attribute__((always_inline)) {
        const int u = t / TILES, kt = t - u * TILES;
        const int64_t first = TRANS ? (int64_t)col_of(u) * p.w_rs + kt * 32 : (int64_t)kt * 32 * p.w_rs + col_of(u);
        global_load_lds16_soff(p.w + first * 2, coff[i], slot_at(slot) + i * 1024);
    };
    auto issue = [&](int t) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < COPIES; ++i) issue_one(t, t, i);
    };
#pragma unroll
    for (int t = 0; t < Geo::kEarly; ++t)
        if (t < ntiles) issue(t);

    char* const panel = smem + Geo::kEarly * 4 * Geo::kTile;
#pragma unroll
    for (int i = 0; i < NP; ++i) {
        if constexpr (MODE != kProductT) {
            const float mean = ln_mean<K>(ln_tree_lanes<LANES>(ln_chunk_sum(xv[i])));
            const float sq = ln_chunk_squares(xv[i], mean);
            const float rstd = ln_rstd<K>(ln_tree_lanes<LANES>(holds ? sq : 0.f), p.eps);
            xv[i] = ln_chunk_apply<vec8, elem>(xv[i], mean, rstd, wv, bv);
        }
        const int row = (wave * NP + i) * RPI + sub;
        if constexpr (MODE == kUqvkGradU) {
            if (p.normed && blockIdx.y == 0 && holds && row0 + row < p.rows) *(vec8*)(p.normed + ((row0 + row) * K + chunk_of * 8) * 2) = xv[i];
        }
        if (holds) *HSTU_LDS(vec8, panel + row * (K * 2) + ((chunk_of ^ (row & 15)) * 16)) = xv[i];
    }
    __syncthreads();
    vec8 xreg[RB][KS];
#pragma unroll
    for (int rb = 0; rb < RB; ++rb)
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) xreg[rb][ks] = *HSTU_LDS(const vec8, panel + (rb * 32 + l32) * (K * 2) + (((2 * ks + g) ^ (l32 & 15)) * 16));
    if constexpr (RB == 2) {  // (they fill the accumulation registers: left to itself the compiler keeps some in memory)
#pragma unroll
        for (int rb = 0; rb < RB; ++rb)
#pragma unroll
            for (int ks = 0; ks < KS; ++ks) asm volatile("" : "+a"(xreg[rb][ks]));
    }
    __syncthreads();  // every wave has its rows: the rings take their place
#pragma unroll
    for (int t = Geo::kEarly; t < RING - 1; ++t)
        if (t < ntiles) issue(t);

    // ---- operands: transposing reads of a tile; the lane supplies the address of 4 consecutive n of k row 8 g + 4 sec + j (+ 16 per k step)
    int waddr[2][DT];
    {
        const int i16 = lane & 15, half = (lane >> 4) & 1, jrow = i16 >> 2, q4 = i16 & 3;
#pragma unroll
        for (int sec = 0; sec < 2; ++sec) {
            const int row = 8 * g + 4 * sec + jrow;
#pragma unroll
            for (int dt = 0; dt < DT; ++dt) {
                const int c = dt * 4 + 2 * half + (q4 >> 1);
                waddr[sec][dt] = row * (NB * 2) + ((NB == 64 ? c ^ swz_w64(row) : c) * 16) + (q4 & 1) * 8;
            }
        }
    }
    // the operands of a tile, each of which RB MFMAs use: 16 k, 32 columns
    constexpr int OPS = 2 * DT;
    vec8 fr[OPS];
    int taddr[2];  // (transposed W: the lane's column, chunk 2 kk + g of its 32 k)
#pragma unroll
    for (int kk = 0; kk < 2; ++kk) taddr[kk] = l32 * 64 + (((2 * kk + g) ^ ((l32 >> 2) & 3)) * 16);
    auto load_op = [&](int slot, int op) __attribute__((always_inline)) {
        if constexpr (TRANS) {
            fr[op] = *HSTU_LDS(const vec8, slot_at(slot) + (op % DT) * 2048 + taddr[op / DT]);
            return;
        }
        const char* tile = slot_at(slot) + (op / DT) * 16 * (NB * 2);
        fr[op] = read_vt_operand<TT>(tile + waddr[0][op % DT], tile + waddr[1][op % DT]);
    };
    char* const stage = smem + 4 * RING * Geo::kTile + wave * Geo::kStage;
    float amax[3] = {0.f, 0.f, 0.f};  // (e4m3 output) the largest |value| this lane has stored of v, q, k
    int slot = 0;                     // of the tile in progress
    if (units > 0) {
        if (ntiles >= RING - 1) asm volatile("s_waitcnt vmcnt(%0)" : : "n"(COPIES * (RING - 2)) : "memory");
        else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
#pragma unroll
        for (int op = 0; op < OPS; ++op) load_op(0, op);
    }

    // ---- the epilogue of unit u, in pieces: bias, SiLU, rounding and staging of 4 columns x 32 rows; rows out of the staging area; stores
    constexpr int CPR = NB / 8, RPS = 64 / CPR, STORES = 32 / RPS;  // lanes per row, rows per store, stores per 32 rows
    const int chunk = lane % CPR, rsub = lane / CPR;
    elem4 b4[DT][4];
    i32x4_t rd[STORES];
    auto read_bias = [&](int u) __attribute__((always_inline)) {
        const char* b = smem + Geo::kBias + (col_of(u) - col0_wg) * 2 + g * 8;
#pragma unroll
        for (int dt = 0; dt < DT; ++dt)
#pragma unroll
            for (int r4 = 0; r4 < 4; ++r4) b4[dt][r4] = *HSTU_LDS(const elem4, b + dt * 64 + r4 * 16);
    };
    auto piece = [&](int i, const f32x16_t(&sums)[RB][DT], bool silu) __attribute__((always_inline)) {
        const int rb = i / (4 * DT), dt = i / 4 % DT, r4 = i % 4;
        float v[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) v[j] = BIAS ? sums[rb][dt][r4 * 4 + j] + (float)b4[dt][r4][j] : sums[rb][dt][r4 * 4 + j];
        if (silu) {
#pragma unroll
            for (int j = 0; j < 4; ++j) v[j] = v[j] * __builtin_amdgcn_rcpf(1.0f + __builtin_amdgcn_exp2f(-1.4426950408889634f * v[j]));
        }
        elem4 o;
        if constexpr (BIAS) o = round_to<elem>(v);
        else o = round_sums<elem>(v);
        *HSTU_LDS(elem4, stage + l32 * Geo::kStageRow + (dt * 32 + r4 * 8 + g * 4) * 2) = o;
    };
    auto read_rows = [&](int i) __attribute__((always_inline)) {
        rd[i % STORES] = *HSTU_LDS(const i32x4_t, stage + (i % STORES * RPS + rsub) * Geo::kStageRow + chunk * 16);
    };
    char* const obase = p.out + row0 * p.out_rs * 2;
    const char* const dbase = MODE == kUqvkGradU ? p.du + row0 * p.du_rs * 2 : nullptr;
    unsigned char* const obase8 = OUT8 ? p.out8 + row0 * (p.n_out - p.n_silu) : nullptr;
    const int rows_here = p.rows - row0 < RB * 32 ? (int)(p.rows - row0) : RB * 32;
    // (computed where it is used: hoisted out of the loop, the addresses of all stores take registers that the rows need)
    auto orow = [&](int i) __attribute__((always_inline)) {
        int r = rsub;
        asm volatile("" : "+v"(r));
        return i * RPS + r;
    };
    vec8 dv[RB * STORES];
    auto read_du = [&](int i, int col0) __attribute__((always_inline)) {
        int r = orow(i);
        r = r < rows_here ? r : rows_here - 1;
        dv[i] = *(const vec8*)(dbase + (int64_t)col0 * 2 + ((unsigned)r * (unsigned)(p.du_rs * 2) + chunk * 16));
    };
    auto store_rows = [&](int i, int col0) __attribute__((always_inline)) {
        const int r = orow(i);
        if constexpr (MODE == kUqvkGradU) {  // (the rounded sums, as a product of its own would leave them)
            const vec8 f8 = __builtin_bit_cast(vec8, rd[i % STORES]);
            vec8 o;
#pragma unroll
            for (int j = 0; j < 8; ++j) {
                const float f = (float)f8[j], sg = __builtin_amdgcn_rcpf(1.0f + __builtin_amdgcn_exp2f(-1.4426950408889634f * f));
                o[j] = (elem)((float)dv[i][j] * sg * (1.f + f * (1.f - sg)));
            }
            rd[i % STORES] = __builtin_bit_cast(i32x4_t, o);
        }
        if (r < rows_here) *(i32x4_t*)(obase + (int64_t)col0 * 2 + ((unsigned)r * (unsigned)(p.out_rs * 2) + chunk * 16)) = rd[i % STORES];
    };
    // the rounded values once more, scaled, as e4m3
    auto convert8 = [&](int i, int col0) __attribute__((always_inline)) {
        const int r = orow(i);
        if (col0 < p.n_silu || r >= rows_here) return;
        const int tensor = col0 < 2 * p.n_silu ? 0 : col0 < 2 * p.n_silu + p.n_attn ? 1 : 2;
        const vec8 e = __builtin_bit_cast(vec8, rd[i % STORES]);
        const float is = p.inv_scale[tensor];
        float f[8], m8 = 0.f;
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            const float x = (float)e[j];
            m8 = __builtin_fmaxf(m8, __builtin_fabsf(x));
            f[j] = __builtin_fminf(__builtin_fmaxf(x * is, -448.0f), 448.0f);
        }
#pragma unroll
        for (int t = 0; t < 3; ++t) amax[t] = tensor == t ? __builtin_fmaxf(amax[t], m8) : amax[t];
        int lo = 0, hi = 0;
        lo = __builtin_amdgcn_cvt_pk_fp8_f32(f[0], f[1], lo, false);
        lo = __builtin_amdgcn_cvt_pk_fp8_f32(f[2], f[3], lo, true);
        hi = __builtin_amdgcn_cvt_pk_fp8_f32(f[4], f[5], hi, false);
        hi = __builtin_amdgcn_cvt_pk_fp8_f32(f[6], f[7], hi, true);
        *(i32x2_t*)(obase8 + (col0 - p.n_silu) + ((unsigned)r * (unsigned)(p.n_out - p.n_silu) + chunk * 8)) = i32x2_t{lo, hi};
    };
    auto finish = [&](const f32x16_t(&sums)[RB][DT], int u) __attribute__((always_inline)) {
        const int col0 = col_of(u);
        if constexpr (BIAS) read_bias(u);
        if constexpr (MODE == kUqvkGradU) {
#pragma unroll
            for (int i = 0; i < RB * STORES; ++i) read_du(i, col0);
        }
#pragma unroll
        for (int rb = 0; rb < RB; ++rb) {
            if ((MODE == kUqvkForward || MODE == kUqvkForward8) && col0 < p.n_silu) {  // (a unit's columns are all u's or none)
#pragma unroll
                for (int i = 0; i < 4 * DT; ++i) piece(rb * 4 * DT + i, sums, true);
            } else {
#pragma unroll
                for (int i = 0; i < 4 * DT; ++i) piece(rb * 4 * DT + i, sums, false);
            }
#pragma unroll
            for (int i = 0; i < STORES; ++i) read_rows(rb * STORES + i);
#pragma unroll
            for (int i = 0; i < STORES; ++i) {
                store_rows(rb * STORES + i, col0);
                if constexpr (OUT8) convert8(rb * STORES + i, col0);
            }
        }
    };

    for (int u = 0; u < units; ++u) {
        f32x16_t acc[RB][DT];
#pragma unroll
        for (int rb = 0; rb < RB; ++rb)
#pragma unroll
            for (int dt = 0; dt < DT; ++dt)
#pragma unroll
                for (int r = 0; r < 16; ++r) acc[rb][dt][r] = 0.f;
#pragma unroll
        for (int kt = 0; kt < TILES; ++kt) {
            const int t = u * TILES + kt;
            const int next = slot + 1 == RING ? 0 : slot + 1, before = slot == 0 ? RING - 1 : slot - 1;
            // The next tile has landed: at most the copies of the RING - 3 behind it are outstanding (stores in between make the wait longer
            // than it had to be, never shorter).
            if (t + RING - 2 < ntiles) asm volatile("s_waitcnt vmcnt(%0)" : : "n"(COPIES * (RING - 3)) : "memory");
            else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
            const bool more = t + RING - 1 < ntiles;
            // Behind each operand's products: the same operand of the next tile, and copies into the slot of the tile before this one, whose
            // operands have been multiplied.
#pragma unroll
            for (int op = 0; op < OPS; ++op) {
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int rb = 0; rb < RB; ++rb) acc[rb][op % DT] = TT::mfma(fr[op], xreg[rb][kt * 2 + op / DT], acc[rb][op % DT]);
                load_op(next, op);
                __builtin_amdgcn_sched_barrier(0);
                if (more) {
#pragma unroll
                    for (int i = op * COPIES / OPS; i < (op + 1) * COPIES / OPS; ++i) issue_one(t + RING - 1, before, i);
                }
            }
            slot = next;
        }
        __builtin_amdgcn_sched_barrier(0);
        finish(acc, u);
    }
    if constexpr (OUT8) {  // one maximum per workgroup and tensor: hundreds of workgroups end together, on three addresses
#pragma unroll
        for (int t = 0; t < 3; ++t) {
            float m = amax[t];
#pragma unroll
            for (int d = 32; d >= 1; d >>= 1) m = __builtin_fmaxf(m, __shfl_xor(m, d, 64));
            if (lane == 0) *HSTU_LDS(float, stage + t * 4) = m;
        }
        __syncthreads();
        if (threadIdx.x < 3) {
            float m = 0.f;
#pragma unroll
            for (int w = 0; w < 4; ++w) m = __builtin_fmaxf(m, *HSTU_LDS(const float, smem + 4 * RING * Geo::kTile + w * Geo::kStage + threadIdx.x * 4));
            if (m > 0.f) atomicMax(p.absmax + threadIdx.x, __builtin_bit_cast(unsigned, m));
        }
    }
}

constexpr int kUqvkWaves = 4, kUqvkRowsPerWave = 32;
constexpr int kUqvkTileK = 64, kUqvkTileN = 128;
constexpr int kUqvkSlot = kUqvkTileK * kUqvkTileN * 2;  // one W tile
constexpr int kUqvkBiasRing = 4 * 256;                  // the bias values of four consecutive column blocks
constexpr int kUqvkLds = 3 * kUqvkSlot + kUqvkBiasRing + kUqvkWaves * 32 * kUqvkStageRow;

// The kernel with 32 rows per wave: a workgroup of 4 waves owns 128 rows and walks its share of W's columns once, W's tiles shared by its
// waves (three slots, one barrier per tile; two workgroups per CU).  For each block of 128 output columns, d_model / 64 k tiles of 16
// MFMAs per wave, then the epilogue.  Stores count in the same counter as the copies (vmcnt), so the wait after an epilogue
// leaves room for them.
template <class TT, int KT>  // KT = d_model / 64: k tiles per column block
__global__ __launch_bounds__(kUqvkWaves * 64, 2) void hstu_uqvk_fused_kernel(const UqvkFusedParams p) {
    typedef typename TT::vec8 vec8;
    typedef typename TT::elem elem;
    constexpr int K = KT * kUqvkTileK, KS = K / 16;
    constexpr int NOPS = kUqvkTileK / 16 * 4;                  // A operands per tile: (kk, dt)
    constexpr int NPW = (kUqvkTileK * 16 / 64) / kUqvkWaves;  // copy instructions per wave and tile: 4
    constexpr int RG = kUqvkRowsPerWave / 32;                  // blocks of 32 rows per wave
    constexpr int PD = 3;
    extern __shared__ __attribute__((aligned(1024))) char smem[];

    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int g = lane >> 5, l32 = lane & 31;
    const int64_t row0 = ((int64_t)blockIdx.x * kUqvkWaves + wave) * kUqvkRowsPerWave;  // first row of the wave
    // the column blocks of this workgroup: [c_begin, c_begin + nchunks)
    const int c_begin = blockIdx.y * p.units_per_wave;
    const int left = p.n_out / kUqvkTileN - c_begin;
    const int nchunks = left < p.units_per_wave ? left : p.units_per_wave;
    const int ntiles = nchunks * KT;

    // copy of tile t = (column block c, k tile kt) into slot t % 3; wave 0 adds the block's bias values with the first k tile
    unsigned coff[NPW];
#pragma unroll
    for (int i = 0; i < NPW; ++i) {
        const int pidx = (wave + kUqvkWaves * i) * 64 + lane;
        const int row = pidx >> 4;
        const int logical = (pidx & 15) ^ swz_w(row);
        coff[i] = (unsigned)row * (unsigned)(p.n_out * 2) + logical * 16;
    }
    auto issue_copy = [&](int t) {
        const int c = t / KT, kt = t - c * KT;
        char* slot = smem + (t % 3) * kUqvkSlot;
        const char* src = p.w + ((int64_t)kt * kUqvkTileK * p.n_out + (int64_t)(c_begin + c) * kUqvkTileN) * 2;
#pragma unroll
        for (int i = 0; i < NPW; ++i) global_load_lds16_soff(src, coff[i], slot + (wave + kUqvkWaves * i) * 1024);
        // block c's bias is read after its last k tile, when at most the copies of block c + 1 have been issued
        if (kt == 0 && wave == 0 && lane < 16)
            global_load_lds16(p.bias + (int64_t)(c_begin + c) * kUqvkTileN * 2 + lane * 16, smem + 3 * kUqvkSlot + (c & 3) * 256);
    };
    issue_copy(0);
    if (ntiles > 1) issue_copy(1);

    // ---- this wave's rows: load, normalise, keep as B operands
    vec8 xreg[RG][KS];
#pragma unroll
    for (int rg = 0; rg < RG; ++rg) uqvk_normalised_row<TT, KS, false>(p, row0 + rg * 32 + l32, g, xreg[rg]);

    // transposing reads of a W tile: lane supplies the address of 4 consecutive n of k row 8g + 4sec + j
    int waddr[2][4];
    {
        const int i16 = lane & 15, half = (lane >> 4) & 1, jrow = i16 >> 2, q4 = i16 & 3;
#pragma unroll
        for (int sec = 0; sec < 2; ++sec) {
            const int row = 8 * g + 4 * sec + jrow;  // + 16 kk
#pragma unroll
            for (int dt = 0; dt < 4; ++dt) {
                const int chunk = dt * 4 + 2 * half + (q4 >> 1);
                waddr[sec][dt] = row * 256 + ((chunk ^ swz_w(row)) * 16) + (q4 & 1) * 8;
            }
        }
    }
    char* stage = smem + 3 * kUqvkSlot + kUqvkBiasRing + wave * 32 * kUqvkStageRow;

    f32x16_t acc[RG][4];
    float amax[3] = {0.f, 0.f, 0.f};  // (e4m3 output) the largest |value| this lane has stored of v, q, k
    for (int c = 0; c < nchunks; ++c) {
#pragma unroll
        for (int rg = 0; rg < RG; ++rg)
#pragma unroll
            for (int dt = 0; dt < 4; ++dt)
#pragma unroll
                for (int r = 0; r < 16; ++r) acc[rg][dt][r] = 0.f;
        const char* bias_lds = smem + 3 * kUqvkSlot + (c & 3) * 256;
#pragma unroll
        for (int kt = 0; kt < KT; ++kt) {
            const int t = c * KT + kt;
            // everything but the newest batch of copies (tile t + 1) -- and, after an epilogue, its stores, which
            // count in the same counter -- has landed for this wave ...
            constexpr int STORES = RG * 8;
            if (t + 1 >= ntiles) __builtin_amdgcn_s_waitcnt(0x0F70);
            else if (kt == 0 && c > 0) __builtin_amdgcn_s_waitcnt(0x0F70 | ((NPW + STORES) & 15) | (((NPW + STORES) >> 4) << 14));
            else __builtin_amdgcn_s_waitcnt(0x0F70 | NPW);
            __syncthreads();  // ... and for every wave; nobody reads tile t - 1 any more, whose slot tile t + 2 takes
            if (t + 2 < ntiles) issue_copy(t + 2);
            const char* tile = smem + (t % 3) * kUqvkSlot;
            // NOPS A operands, each used for the wave's RG row blocks: op m = (kk, dt) = (m / 4, m % 4), requested PD ahead
            auto load_op = [&](int m) __attribute__((always_inline)) -> vec8 {
                const char* b = tile + (m >> 2) * 16 * 256;
                return read_vt_operand<TT>(b + waddr[0][m & 3], b + waddr[1][m & 3]);
            };
            vec8 fr[PD];
#pragma unroll
            for (int m = 0; m < PD; ++m) fr[m] = load_op(m);
#pragma unroll
            for (int m = 0; m < NOPS; ++m) {
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int rg = 0; rg < RG; ++rg) acc[rg][m & 3] = TT::mfma(fr[m % PD], xreg[rg][kt * (kUqvkTileK / 16) + (m >> 2)], acc[rg][m & 3]);
                if (m + PD < NOPS) fr[m % PD] = load_op(m + PD);
            }
            __builtin_amdgcn_sched_barrier(0);
        }
        // ---- epilogue of the column block: bias, SiLU for the u columns, rounding, transposition through LDS, stores
        const int col_block = (c_begin + c) * kUqvkTileN;
#pragma unroll
        for (int rg = 0; rg < RG; ++rg)
#pragma unroll
        for (int hf = 0; hf < 2; ++hf) {
#pragma unroll
            for (int d2 = 0; d2 < 2; ++d2) {
                const int dt = hf * 2 + d2;
                const bool silu = col_block + dt * 32 < p.n_silu;
#pragma unroll
                for (int r4 = 0; r4 < 4; ++r4) {
                    typedef __attribute__((ext_vector_type(4))) elem elem4;
                    const elem4 b4 = *HSTU_LDS(const elem4, bias_lds + (dt * 32 + r4 * 8 + g * 4) * 2);
                    float v[4];
#pragma unroll
                    for (int i = 0; i < 4; ++i) {
                        v[i] = acc[rg][dt][r4 * 4 + i] + (float)b4[i];
                        if (silu) v[i] = v[i] * __builtin_amdgcn_rcpf(1.0f + __builtin_amdgcn_exp2f(-1.4426950408889634f * v[i]));
                    }
                    *HSTU_LDS(elem4, stage + l32 * kUqvkStageRow + (d2 * 32 + r4 * 8 + g * 4) * 2) = round_to<elem>(v);
                }
            }
            // 8 lanes cover one row's 128 bytes, 8 rows per instruction
            const int chunk = lane & 7, rsub = lane >> 3;
            const int col0 = col_block + hf * 64;  // first column of this half block
            const bool to8 = p.out8 != nullptr && col0 >= p.n_silu;
            const int tensor = col0 < 2 * p.n_silu ? 0 : col0 < 2 * p.n_silu + p.n_attn ? 1 : 2;
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int row = i * 8 + rsub;
                const i32x4_t v = *HSTU_LDS(const i32x4_t, stage + row * kUqvkStageRow + chunk * 16);
                // rows past the end are the last row once more, the same bits to the same place: a store that is left out where no lane has
                // a row would be missing from the number of instructions in flight that the next tile's wait counts with
                int64_t r = row0 + rg * 32 + row;
                r = r < p.rows ? r : p.rows - 1;
                *(i32x4_t*)(p.out + (r * p.n_out + col0) * 2 + chunk * 16) = v;
                if (to8) {
                    // the rounded values once more, scaled, as e4m3: 8 lanes cover 64 bytes of a row
                    const vec8 e = __builtin_bit_cast(vec8, v);
                    const float is = p.inv_scale[tensor];
                    float f[8], m8 = 0.f;
#pragma unroll
                    for (int j = 0; j < 8; ++j) {
                        const float x = (float)e[j];
                        m8 = __builtin_fmaxf(m8, __builtin_fabsf(x));
                        f[j] = __builtin_fminf(__builtin_fmaxf(x * is, -448.0f), 448.0f);
                    }
                    // (rows past the end repeat the last row: they change no maximum)
                    amax[0] = tensor == 0 ? __builtin_fmaxf(amax[0], m8) : amax[0];
                    amax[1] = tensor == 1 ? __builtin_fmaxf(amax[1], m8) : amax[1];
                    amax[2] = tensor == 2 ? __builtin_fmaxf(amax[2], m8) : amax[2];
                    int lo = 0, hi = 0;
                    lo = __builtin_amdgcn_cvt_pk_fp8_f32(f[0], f[1], lo, false);
                    lo = __builtin_amdgcn_cvt_pk_fp8_f32(f[2], f[3], lo, true);
                    hi = __builtin_amdgcn_cvt_pk_fp8_f32(f[4], f[5], hi, false);
                    hi = __builtin_amdgcn_cvt_pk_fp8_f32(f[6], f[7], hi, true);
                    typedef __attribute__((ext_vector_type(2))) int i32x2_t;
                    *(i32x2_t*)(p.out8 + r * (int64_t)(p.n_out - p.n_silu) + (col0 - p.n_silu) + chunk * 8) = i32x2_t{lo, hi};
                }
            }
        }
    }
    if (p.out8 != nullptr) {
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
