// The output step in one kernel for rows that fill the chip and d_out a multiple of 512 (gfx950):
//
//     out[r, n] = x[r, n] + sum_k joined[r, k] * W[k, n],   joined = [u | attn | y],  y = u * norm(attn)
// (hstu_compute_output of the reference, ops/hstu_compute.py:107-170).
//
// A workgroup of 8 waves, one per CU, owns 128 rows and 512 columns at a time, wave w columns 64 w .. 64 w + 63 in 128 accumulator registers: the rows are
// read and normalised once, and 128 rows share a pass over W.  The depth is walked in slices of 32 columns of u, attn and y, six steps of 16: u and attn
// come into LDS by copies issued a slice and a half ahead, and of its own 16 rows every wave makes y there while the slice before is multiplied, so that
// one barrier per slice is enough.  W's tiles (16 k x 64 columns) come through a private ring of six per wave, whose copies no barrier concerns.  The norm's
// sums are taken first, from the rows of attn in registers; the first slices of the next rows are on their way meanwhile, through the epilogue.
// Copies complete in order, so a copy from HBM between two of W's tiles holds the second one's wait up: the ring is deep enough for that.
#pragma once
#include <type_traits>

#include "hstu_output_panel_kernel.h"
#include "hstu_uqvk_kernel.h"

namespace hstu {

constexpr int kOutWideRows = 128, kOutWideCols = 512, kOutWideWaves = 8;
constexpr int kOutWideRing = 6, kOutWideTile = 16 * 64 * 2;
constexpr int kOutWidePanel = kOutWideRows * 64;                 // 32 columns of the rows
constexpr int kOutWideHeads = 8;                                 // group norm: heads whose sums fit
constexpr int kOutWideStats = kOutWideHeads * kOutWideRows * 8;  // mean and 1 / deviation of a row (of a head of it)
constexpr int kOutWideLds = kOutWideWaves * kOutWideRing * kOutWideTile + 6 * kOutWidePanel + kOutWideStats + 2 * 1024 * 2;
constexpr int kOutWideStageRow = 64 * 4 + 16;                    // a row of a wave's sums on their way to the stores
static_assert(32 * kOutWideStageRow <= kOutWideRing * kOutWideTile, "32 rows of sums fit a wave's ring");

template <class TT, bool GROUP, int D>
__global__ __launch_bounds__(kOutWideWaves * 64, 2) void hstu_output_wide_kernel(const OutputPanelParams p) {
    typedef typename TT::vec8 vec8;
    typedef typename TT::elem elem;
    typedef __attribute__((ext_vector_type(2))) float f32x2_t;
    constexpr int CH = D / 8;                        // chunks of a row
    constexpr int LPR = D > 256 ? 64 : D / 8;        // lanes that a row lies across
    constexpr int CPL = D > 512 ? D / 512 : 1;       // chunks of it per lane
    constexpr int RPI = 64 / LPR;                    // rows a wave handles at a time
    constexpr int IT = 16 / RPI;                     // ... and how often
    constexpr int NS = D / 32, PANEL = kOutWidePanel, RING = kOutWideRing, TILE = kOutWideTile;
    static_assert(D % 128 == 0 && (D <= 512 || D == 1024), "an even number of slices, whole chunks per lane");
    extern __shared__ __attribute__((aligned(1024))) char smem[];
    const NormMulParams& nm = p.nm;

    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int g = lane >> 5, l32 = lane & 31;
    const unsigned row_blocks = (unsigned)((nm.rows + kOutWideRows - 1) / kOutWideRows);
    const unsigned items = row_blocks * ((unsigned)p.n / kOutWideCols);

    char* const ring = smem + wave * RING * TILE;
    char* const panels = smem + kOutWideWaves * RING * TILE;  // u, attn, y of even slices, of odd slices
    char* const stats = panels + 6 * PANEL;
    char* const table = stats + kOutWideStats;                // the norm's weight and bias

    // ---- copies of W's tiles: instruction i brings 8 k rows of 128 bytes
    unsigned coff[2];
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        const int row = 8 * i + (lane >> 3);
        coff[i] = (unsigned)row * (unsigned)(p.n * 2) + (unsigned)wave * 128 + ((lane & 7) ^ swz_w64(row)) * 16;
    }
    const unsigned wrow16 = 16u * (unsigned)p.n * 2, wblock = D / 16 * wrow16;
    const i32x4_t wrsrc = make_buffer_rsrc(p.w, 3 * wblock);
    auto issue_w = [&](unsigned at, int j, int i) __attribute__((always_inline)) {  // tile j of the slice whose first row of u's part of W lies at `at`
        buffer_load_lds16(wrsrc, coff[i], at + (j >> 1) * wblock + (j & 1) * wrow16, ring + j * TILE + i * 1024);
    };
    // ---- copies of u and attn: a wave brings its own 16 rows, 64 bytes each, the four chunks swizzled as the operands' reads want.  (Rows past the end: zeros)
    const int prow = wave * 16 + (lane >> 2), pchunk = (lane & 3) ^ swz_k<4>(lane >> 2);
    const unsigned uoff = (unsigned)prow * (unsigned)(nm.u_rs * 2) + pchunk * 16, aoff = (unsigned)prow * (unsigned)(nm.attn_rs * 2) + pchunk * 16;
    struct Rows { i32x4_t u, a; };
    auto rows_of = [&](unsigned item) __attribute__((always_inline)) {
        const int64_t row0 = (int64_t)(item % row_blocks) * kOutWideRows;
        const unsigned last = (unsigned)(nm.rows - 1 - row0 < kOutWideRows - 1 ? nm.rows - 1 - row0 : kOutWideRows - 1);
        return Rows{make_buffer_rsrc(nm.u + row0 * nm.u_rs * 2, last * (unsigned)(nm.u_rs * 2) + D * 2),
                    make_buffer_rsrc(nm.attn + row0 * nm.attn_rs * 2, last * (unsigned)(nm.attn_rs * 2) + D * 2)};
    };
    auto issue_rows = [&](const Rows& r, int s, int par) __attribute__((always_inline)) {
        buffer_load_lds16(r.u, uoff, (unsigned)s * 64, panels + (par * 3 + 0) * PANEL + wave * 1024);
        buffer_load_lds16(r.a, aoff, (unsigned)s * 64, panels + (par * 3 + 1) * PANEL + wave * 1024);
    };

    // ---- operand addresses
    int waddr[2][2];  // transposing reads of a W tile
    {
        const int i16 = lane & 15, half = (lane >> 4) & 1, jrow = i16 >> 2, q4 = i16 & 3;
#pragma unroll
        for (int sec = 0; sec < 2; ++sec) {
            const int row = 8 * g + 4 * sec + jrow;
#pragma unroll
            for (int dt = 0; dt < 2; ++dt) waddr[sec][dt] = row * 128 + (((dt * 4 + 2 * half + (q4 >> 1)) ^ swz_w64(row)) * 16) + (q4 & 1) * 8;
        }
    }
    int paddr[2];
#pragma unroll
    for (int st = 0; st < 2; ++st) paddr[st] = l32 * 64 + (((2 * st + g) ^ swz_k<4>(l32)) * 16);

    // ---- the norm's weight and bias (group norm: one of each per head)
    {
        const int count = GROUP ? CH / nm.group_lanes : D;
        for (int i = threadIdx.x; i < count; i += kOutWideWaves * 64) {
            HSTU_LDS(elem, table)[i] = ((const elem*)nm.weight)[i];
            HSTU_LDS(elem, table + 2048)[i] = ((const elem*)nm.bias)[i];
        }
    }
    __syncthreads();

    const int chunk = lane % LPR, rsub = lane / LPR;
    const bool holds = LPR * 8 * CPL == D || chunk < CH;
    // sums over the lanes of a row (of a head), added as the norm-multiply kernel adds
    auto row_sum = [&](float s) __attribute__((always_inline)) {
        if constexpr (GROUP) {
            const int lanes = nm.group_lanes;
            if (lanes > 1) s = add_dpp<0xB1>(s);    // quad_perm [1, 0, 3, 2]
            if (lanes > 2) s = add_dpp<0x4E>(s);    // quad_perm [2, 3, 0, 1]
            if (lanes > 4) s = add_dpp<0x141>(s);   // row_half_mirror: the other quad of 8, whose lanes agree
            if (lanes > 8) s = add_dpp<0x140>(s);   // row_mirror: the other 8 of 16
            if (LPR > 16 && lanes > 16) s = add_xor16(s);
            if (LPR > 32 && lanes > 32) s = add_xor32(s);
        } else {
            if constexpr (LPR > 32) s = add_xor32(s);
            if constexpr (LPR > 16) s = add_xor16(s);
            s = add_dpp<0x128>(s);
            s = add_dpp<0x124>(s);
            s = add_dpp<0x122>(s);
            s = add_dpp<0x121>(s);
        }
        return s;
    };
    // mean and 1 / deviation of this wave's 16 rows, into LDS (nobody else reads them)
    auto make_stats = [&](int64_t row0) __attribute__((always_inline)) {
        constexpr int LOADS = IT * CPL <= 16 ? IT : 16 / CPL;  // rows of registers at a time
        const float inv_n = GROUP ? 1.0f / (float)(nm.group_lanes * 8) : 1.0f / (float)D;
#pragma unroll
        for (int i0 = 0; i0 < IT; i0 += LOADS) {
            vec8 av[LOADS][CPL];
#pragma unroll
            for (int i = 0; i < LOADS; ++i) {
                int64_t r = row0 + wave * 16 + (i0 + i) * RPI + rsub;
                r = r < nm.rows ? r : nm.rows - 1;
#pragma unroll
                for (int c = 0; c < CPL; ++c) {
                    av[i][c] = vec8{};
                    if (holds) av[i][c] = *(const vec8*)(nm.attn + (r * nm.attn_rs + (c * 64 + chunk) * 8) * 2);
                }
            }
            constexpr int G = LOADS < 4 ? LOADS : 4;
#pragma unroll
            for (int i1 = 0; i1 < LOADS; i1 += G) {
#pragma unroll
                for (int i = i1; i < LOADS; ++i)
#pragma unroll
                    for (int c = 0; c < CPL; ++c) asm volatile("" : "+v"(av[i][c]));  // (they stay packed until their turn)
#pragma unroll
                for (int c0 = 0; c0 < (GROUP ? CPL : 1); ++c0) {  // (a head lies within one chunk column of the lanes)
                    constexpr int CN = GROUP ? 1 : CPL;
                    float v[G][CN][8], mean[G], sq[G];
#pragma unroll
                    for (int i = 0; i < G; ++i) {
                        mean[i] = 0.f;
#pragma unroll
                        for (int c = 0; c < CN; ++c)
#pragma unroll
                            for (int j = 0; j < 8; ++j) v[i][c][j] = (float)av[i1 + i][c0 + c][j], mean[i] += v[i][c][j];
                    }
#pragma unroll
                    for (int i = 0; i < G; ++i) mean[i] = row_sum(mean[i]) * inv_n;
#pragma unroll
                    for (int i = 0; i < G; ++i) {
                        sq[i] = 0.f;
#pragma unroll
                        for (int c = 0; c < CN; ++c)
#pragma unroll
                            for (int j = 0; j < 8; ++j) v[i][c][j] -= mean[i], sq[i] += v[i][c][j] * v[i][c][j];
                        if (!holds) sq[i] = 0.f;
                    }
#pragma unroll
                    for (int i = 0; i < G; ++i) sq[i] = row_sum(sq[i]);
#pragma unroll
                    for (int i = 0; i < G; ++i) {
                        const float rstd = __builtin_amdgcn_rsqf(sq[i] * inv_n + nm.eps);
                        const int row = wave * 16 + (i0 + i1 + i) * RPI + rsub;
                        if constexpr (GROUP) {
                            const int at = c0 * 64 + chunk;
                            if (holds && (at & (nm.group_lanes - 1)) == 0)
                                *HSTU_LDS(f32x2_t, stats + (at / nm.group_lanes * kOutWideRows + row) * 8) = f32x2_t{mean[i], rstd};
                        } else if (chunk == 0) {
                            *HSTU_LDS(f32x2_t, stats + row * 8) = f32x2_t{mean[i], rstd};
                        }
                    }
                }
            }
        }
    };
    const int head_shift = GROUP ? 3 + __builtin_ctz(nm.group_lanes) : 0;
    // y of a slice, this wave's rows: a lane makes the chunk that its copies brought, fetched in step 3 of the slice before, an element behind each product of
    // step 4 (in one piece it held the matrix pipe up: 131072 rows 241 us, so 236)
    vec8 yu, ya, yw, yb;
    f32x2_t yst;
    auto fetch_y = [&](int s, int par) __attribute__((always_inline)) {
        const char* const at = panels + par * 3 * PANEL + wave * 1024 + lane * 16;
        yu = *HSTU_LDS(const vec8, at), ya = *HSTU_LDS(const vec8, at + PANEL);
        const int col = s * 32 + pchunk * 8;
        if constexpr (GROUP) {
            const int head = col >> head_shift;
            yst = *HSTU_LDS(const f32x2_t, stats + (head * kOutWideRows + prow) * 8);
            yw[0] = *HSTU_LDS(const elem, table + head * 2), yb[0] = *HSTU_LDS(const elem, table + 2048 + head * 2);
        } else {
            yst = *HSTU_LDS(const f32x2_t, stats + prow * 8);
            yw = *HSTU_LDS(const vec8, table + col * 2), yb = *HSTU_LDS(const vec8, table + 2048 + col * 2);
        }
    };
    auto make_y = [&](int j) __attribute__((always_inline)) {
        const float v = (float)ya[j] - yst[0];
        yu[j] = (elem)((float)yu[j] * (v * yst[1] * (float)yw[GROUP ? 0 : j] + (float)yb[GROUP ? 0 : j]));
    };
    auto put_y = [&](int par) __attribute__((always_inline)) {
        *HSTU_LDS(vec8, panels + (par * 3 + 2) * PANEL + wave * 1024 + lane * 16) = yu;
    };

    unsigned item = blockIdx.x;
    if (item >= items) return;
    Rows rows = rows_of(item);
    issue_rows(rows, 0, 0);
    issue_rows(rows, 1, 1);
    while (true) {
        const int64_t row0 = (int64_t)(item % row_blocks) * kOutWideRows;
        const int col0 = (int)(item / row_blocks) * kOutWideCols;
        const unsigned next = item + gridDim.x;
        const Rows next_rows = rows_of(next < items ? next : item);  // (past the last item: this one's rows, which nobody reads)
        unsigned wat = (unsigned)col0 * 2;  // u's part of W, the slice in progress
#pragma unroll
        for (int j = 0; j < RING; ++j) issue_w(wat, j, 0), issue_w(wat, j, 1);
        make_stats(row0);
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // (the copies above are older than the rows just used)
        fetch_y(0, 0);
#pragma unroll
        for (int j = 0; j < 8; ++j) make_y(j);
        put_y(0);

        f32x16_t acc[4][2];
#pragma unroll
        for (int rb = 0; rb < 4; ++rb)
#pragma unroll
            for (int dt = 0; dt < 2; ++dt)
#pragma unroll
                for (int r = 0; r < 16; ++r) acc[rb][dt][r] = 0.f;

        vec8 wf[2][2], jf[2][4];
        auto load_w = [&](int b, int j, int dt) __attribute__((always_inline)) {
            wf[b][dt] = read_vt_operand<TT>(ring + j * TILE + waddr[0][dt], ring + j * TILE + waddr[1][dt]);
        };
        auto load_rows = [&](int b, int j, int par, int rb) __attribute__((always_inline)) {
            jf[b][rb] = *HSTU_LDS(const vec8, panels + (par * 3 + (j >> 1)) * PANEL + paddr[j & 1] + rb * 2048);
        };
        asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
#pragma unroll
        for (int dt = 0; dt < 2; ++dt) load_w(0, 0, dt);
#pragma unroll
        for (int rb = 0; rb < 4; ++rb) load_rows(0, 0, 0, rb);

        // the residual's rows, two of the four row blocks asked for in the last slice
        const int orow = lane >> 3, ochunk = lane & 7;
        const int64_t ocol = col0 + wave * 64 + ochunk * 8;
        vec8 xr[4][4];
        auto load_x = [&](int rb) __attribute__((always_inline)) {
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                int64_t r = row0 + rb * 32 + i * 8 + orow;
                r = r < nm.rows ? r : nm.rows - 1;
                xr[rb][i] = *(const vec8*)(p.x + (r * p.x_rs + ocol) * 2);
            }
        };

        // Slice s in parity PAR.  LAST: the item's last, behind which W's tiles are not asked for (the ring becomes the stage of the epilogue).
        auto slice = [&](int s, auto Par, auto Last, const Rows& ahead, int ahead_s) __attribute__((always_inline)) {
            constexpr int PAR = decltype(Par)::value;
            constexpr bool LAST = decltype(Last)::value;
            constexpr int XL = 8;
            wat += 2 * wrow16;
#pragma unroll
            for (int j = 0; j < 6; ++j) {
                // The next step's tile has landed.  Behind it are four more tiles, two copies each (in the last slice: those there are), and in front of the
                // last tile of the slice before the two copies of u and attn: in steps 0 .. 2 they may be on their way, in step 3 they are waited for.
                if (!LAST) {
                    if (j < 3) asm volatile("s_waitcnt vmcnt(10)" ::: "memory");
                    else asm volatile("s_waitcnt vmcnt(8)" ::: "memory");
                } else if (j == 0) asm volatile("s_waitcnt vmcnt(10)" ::: "memory");
                else if (j == 1) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(8 + XL) : "memory");
                else if (j == 2) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(6 + XL) : "memory");
                else if (j == 3) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(4 + XL) : "memory");
                else if (j == 4) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(XL) : "memory");
                if (LAST && j == 0) load_x(0), load_x(1);
                if (j == 5) {
                    // every wave has its rows of the next slice in place, y among them, and its operands of this one in registers
                    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
                    issue_rows(ahead, ahead_s, PAR);
                }
                const int b = j & 1, jn = j == 5 ? 0 : j + 1, parn = j == 5 ? 1 - PAR : PAR;
                const bool more = !(LAST && j == 5);
#pragma unroll
                for (int m = 0; m < 8; ++m) {
                    __builtin_amdgcn_sched_barrier(0);
                    acc[m >> 1][m & 1] = TT::mfma(wf[b][m & 1], jf[b][m >> 1], acc[m >> 1][m & 1]);
                    __builtin_amdgcn_sched_barrier(0);
                    if (!LAST && j == 3 && m == 7) fetch_y(s + 1, 1 - PAR);
                    if (!LAST && j == 4) make_y(m);
                    if (!LAST && j == 4 && m == 7) put_y(1 - PAR);
                    if (more && (m == 0 || m == 2)) load_w(1 - b, jn, m / 2);
                    if (more && (m == 1 || (m >= 3 && m < 6))) load_rows(1 - b, jn, parn, m == 1 ? 0 : m - 2);
                    if (!LAST && m >= 6) issue_w(wat, j, m - 6);
                }
            }
        };
        typedef std::integral_constant<int, 0> P0;
        typedef std::integral_constant<int, 1> P1;
        int s = 0;
        for (; s < NS - 2; s += 2) {
            slice(s, P0{}, std::false_type{}, rows, s + 2);
            slice(s + 1, P1{}, std::false_type{}, rows, s + 3);
        }
        slice(s, P0{}, std::false_type{}, next_rows, 0);
        slice(s + 1, P1{}, std::true_type{}, next_rows, 1);

        // ---- the sums through this wave's ring, the residual, whole lines out
        load_x(2), load_x(3);
#pragma unroll
        for (int rb = 0; rb < 4; ++rb) {
#pragma unroll
            for (int dt = 0; dt < 2; ++dt)
#pragma unroll
                for (int r4 = 0; r4 < 4; ++r4) {
                    f32x4_t v;
#pragma unroll
                    for (int j = 0; j < 4; ++j) v[j] = acc[rb][dt][r4 * 4 + j];
                    *HSTU_LDS(f32x4_t, ring + l32 * kOutWideStageRow + (dt * 32 + r4 * 8 + g * 4) * 4) = v;
                }
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const char* const at = ring + (i * 8 + orow) * kOutWideStageRow + ochunk * 32;
                const f32x4_t lo = *HSTU_LDS(const f32x4_t, at), hi = *HSTU_LDS(const f32x4_t, at + 16);
                const int64_t r = row0 + rb * 32 + i * 8 + orow;
                if (r < nm.rows) {
                    vec8 o;
#pragma unroll
                    for (int j = 0; j < 4; ++j) o[j] = (elem)(lo[j] + (float)xr[rb][i][j]), o[4 + j] = (elem)(hi[j] + (float)xr[rb][i][4 + j]);
                    *(vec8*)(p.out + (r * p.n + ocol) * 2) = o;
                }
            }
        }
        if (next >= items) break;
        item = next;
        rows = next_rows;
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // the stage has been read: W's tiles go there now
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // (the copies that nobody reads have landed before the LDS is given back)
}

}  // namespace hstu
