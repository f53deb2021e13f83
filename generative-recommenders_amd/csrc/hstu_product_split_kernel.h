// out[r, n] = sum_k a[r, k] W[n, k] for few rows of any depth (a multiple of 64): the gradient of the layer's input behind the producer, whose depth is the
// width of u, v, q, k (gfx950).
//
// A workgroup owns 32 rows and 64 columns, and its four waves share the depth in blocks of 64: few rows have too few blocks of the result to fill the chip, and a chain
// of the whole depth is long.  A wave's blocks of both operands come through a ring of its own, whole 128-byte lines, three blocks deep, without a barrier; the waves' sums
// meet in LDS and are added in order.  What bounds it: 192 bytes of operands per column of the depth at the 64 bytes a clock of a CU's copies, and the launch (768 deep 4.5 us, 2048
// 6.6, 4096 9.7; with operands loaded from memory to registers, 16 bytes of 32 rows at a time, 5.9, 12.0, 21.8).
#pragma once
#include "hstu_uqvk_kernel.h"

namespace hstu {

constexpr int kSplitRows = 32, kSplitCols = 64, kSplitWaves = 4, kSplitRing = 3;
constexpr int kSplitBlock = (kSplitRows + kSplitCols) * 128;  // 64 of the depth of both operands
constexpr int kSplitCopies = kSplitBlock / 1024;
constexpr int kSplitLds = kSplitWaves * kSplitRing * kSplitBlock;
constexpr int kSplitSumRow = kSplitCols * 4 + 16;             // a row of a wave's sums
static_assert(kSplitRows * kSplitSumRow <= kSplitRing * kSplitBlock, "a wave's sums fit its ring");

struct ProductSplitParams {
    const char* a;  // [rows, k], strides in elements, below 2^22
    const char* w;  // [n, k]
    char* out;
    int64_t a_rs, w_rs, out_rs, rows;
    int k;          // a multiple of 64
};

template <class TT>
__global__ __launch_bounds__(kSplitWaves * 64, 1) void hstu_product_split_kernel(const ProductSplitParams p) {
    typedef typename TT::vec8 vec8;
    typedef typename TT::elem elem;
    extern __shared__ __attribute__((aligned(1024))) char smem[];
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int g = lane >> 5, l32 = lane & 31;
    const int64_t row0 = (int64_t)blockIdx.y * kSplitRows;
    const int col0 = blockIdx.x * kSplitCols;
    char* const ring = smem + wave * kSplitRing * kSplitBlock;

    // copy instruction i brings 8 rows of 128 bytes, the eight chunks swizzled as the operands' reads want: a's 32 rows (past the end the last one again), then W's 64
    const int64_t below = p.rows - 1 - row0;
    unsigned off[kSplitCopies];
#pragma unroll
    for (int i = 0; i < kSplitCopies; ++i) {
        const int row = i * 8 + (lane >> 3), chunk = (lane & 7) ^ swz_k<8>(row);
        if (i < kSplitRows / 8) off[i] = (unsigned)(row < below ? row : (int)below) * (unsigned)(p.a_rs * 2) + chunk * 16;
        else off[i] = (unsigned)(row - kSplitRows) * (unsigned)(p.w_rs * 2) + chunk * 16;
    }
    const char* const abase = p.a + row0 * p.a_rs * 2;
    const char* const wbase = p.w + (int64_t)col0 * p.w_rs * 2;
    const int blocks = p.k / 64, mine = (blocks - wave + kSplitWaves - 1) / kSplitWaves;  // this wave's: wave, wave + 4, ...
    auto issue = [&](int i, int slot) __attribute__((always_inline)) {  // (behind the last one that one again, into a slot nobody reads)
        const int64_t at = (int64_t)(wave + kSplitWaves * (i < mine ? i : mine - 1)) * 128;
#pragma unroll
        for (int c = 0; c < kSplitCopies; ++c)
            global_load_lds16_soff((c < kSplitRows / 8 ? abase : wbase) + at, off[c], ring + slot * kSplitBlock + c * 1024);
    };
    f32x16_t acc[2];
#pragma unroll
    for (int dt = 0; dt < 2; ++dt)
#pragma unroll
        for (int i = 0; i < 16; ++i) acc[dt][i] = 0.f;
    if (mine > 0) {
#pragma unroll
        for (int i = 0; i < kSplitRing; ++i) issue(i, i);
        int slot = 0;
        for (int i = 0; i < mine; ++i) {
            asm volatile("s_waitcnt vmcnt(%0)" : : "n"((kSplitRing - 1) * kSplitCopies) : "memory");
            const char* const at = ring + slot * kSplitBlock;
            vec8 f[4][3];
#pragma unroll
            for (int s = 0; s < 4; ++s)
#pragma unroll
                for (int o = 0; o < 3; ++o) f[s][o] = *HSTU_LDS(const vec8, at + o * 4096 + l32 * 128 + (((2 * s + g) ^ swz_k<8>(l32)) * 16));
#pragma unroll
            for (int s = 0; s < 4; ++s)
#pragma unroll
                for (int dt = 0; dt < 2; ++dt) acc[dt] = TT::mfma(f[s][1 + dt], f[s][0], acc[dt]);
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // the slot has been read
            issue(i + kSplitRing, slot);
            slot = slot + 1 == kSplitRing ? 0 : slot + 1;
        }
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // (the copies that nobody reads have landed)
    }
#pragma unroll
    for (int dt = 0; dt < 2; ++dt)
#pragma unroll
        for (int r4 = 0; r4 < 4; ++r4) {
            f32x4_t s;
#pragma unroll
            for (int j = 0; j < 4; ++j) s[j] = acc[dt][r4 * 4 + j];
            *HSTU_LDS(f32x4_t, ring + l32 * kSplitSumRow + (dt * 32 + r4 * 8 + g * 4) * 4) = s;
        }
    __syncthreads();
    const int row = threadIdx.x >> 3, chunk = threadIdx.x & 7;
    float v[8];
#pragma unroll
    for (int w = 0; w < kSplitWaves; ++w) {
        const char* const at = smem + w * kSplitRing * kSplitBlock + row * kSplitSumRow + chunk * 32;
        const f32x4_t lo = *HSTU_LDS(const f32x4_t, at), hi = *HSTU_LDS(const f32x4_t, at + 16);
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            v[j] = w == 0 ? lo[j] : v[j] + lo[j];
            v[4 + j] = w == 0 ? hi[j] : v[4 + j] + hi[j];
        }
    }
    if (row0 + row < p.rows) {
        vec8 o;
#pragma unroll
        for (int j = 0; j < 8; ++j) o[j] = (elem)v[j];
        *(vec8*)(p.out + ((row0 + row) * p.out_rs + col0 + chunk * 8) * 2) = o;
    }
}

}  // namespace hstu
