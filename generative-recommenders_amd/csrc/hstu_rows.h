// What the row-wise kernels of the dense steps share, forward (hstu_linear.hip) and backward (hstu_linear_bwd.hip): vector types,
// sums over a wave, the arguments of the norm-multiply step and the dropout of its output.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "hstu_linear.h"
#include "hstu_philox.h"

namespace hstu {

typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8_t;
typedef __attribute__((ext_vector_type(8))) _Float16 f16x8_t;

// Sum over the 64 lanes of a wave, result in every lane.
__device__ __forceinline__ float wave_sum(float v) {
#pragma unroll
    for (int d = 32; d >= 1; d >>= 1) v += __shfl_xor(v, d, 64);
    return v;
}

__device__ __forceinline__ float sigmoid_f(float x) { return __builtin_amdgcn_rcpf(1.0f + __expf(-x)); }

// The norm-multiply step: out = [u' | attn | y] with y = act(u) * norm(attn), blocks as the flags say.
struct NormMulParams {
    const char *attn, *u, *weight, *bias;
    char* joined;
    int64_t attn_rs, u_rs, joined_rs, rows;  // strides in elements
    float eps;
    int d, group_lanes;                      // row width; lanes per head (group norm)
    int off_u, off_x, off_y;                 // column offsets of the blocks in `joined`, -1 = block absent
    int silu_u, mul_act;
    DropoutParams drop;                // thresh 0: no dropout
    int64_t width;                           // logical width of `joined` (all blocks): the mask's row pitch
};

// Eight consecutive elements starting at column `col` (a multiple of 8) of row r: dropped or scaled, in fp32.
template <class V8, class E>
__device__ __forceinline__ V8 dropout8(const DropoutParams& d, int64_t r, int64_t width, int64_t col, const float (&x)[8]) {
    const uint64_t group = (uint64_t)(r * width + col) >> 2;
    const PhiloxWords a = dropout_words(d, group), b = dropout_words(d, group + 1);
    V8 out;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        out[j] = (E)(a.w[j] >= d.thresh ? x[j] * d.scale : 0.f);
        out[4 + j] = (E)(b.w[j] >= d.thresh ? x[4 + j] * d.scale : 0.f);
    }
    return out;
}

// False: the ratio is not in [0, 1).
inline bool dropout_params(float ratio, uint64_t seed, uint64_t offset, DropoutParams& d) {
    if (!(ratio >= 0.f && ratio < 1.f)) return false;
    d.seed = seed, d.offset = offset;
    d.thresh = (uint32_t)((double)ratio * 4294967296.0);
    d.scale = 1.0f / (1.0f - ratio);
    return true;
}

inline int output_blocks(const HstuOutputArgs* a) {
    if (a->group_norm) return (a->concat_u && a->concat_x) ? 3 : 1;
    return 1 + (a->concat_u ? 1 : 0) + (a->concat_x ? 1 : 0);
}

// Checks the norm-multiply step's arguments and gathers them; `joined` may be null where the caller has no use for it.
// 0, or the status the entry point returns (rows == 0 is 0 as well: nothing to launch).
inline int norm_mul_params(const HstuOutputArgs* a, void* joined, int64_t joined_rs, bool joined_needed, NormMulParams& p) {
    if (a->rows < 0 || a->heads <= 0 || a->linear_dim <= 0) return -5;
    const int64_t d64 = (int64_t)a->heads * a->linear_dim;
    if (d64 > 4096 || (d64 & 7) != 0) return -5;
    const int d = (int)d64, blocks = output_blocks(a);
    if (a->attn_row_stride < d || a->u_row_stride < d || joined_rs < (int64_t)blocks * d) return -5;
    if (((a->attn_row_stride | a->u_row_stride | joined_rs) & 7) != 0) return -4;
    if (a->dtype != 0 && a->dtype != 1) return -2;
    if (a->mul_u_activation < 0 || a->mul_u_activation > 2) return -5;
    int group_lanes = 0;
    if (a->group_norm) {
        group_lanes = a->linear_dim / 8;
        if ((a->linear_dim & 7) != 0 || group_lanes > 64 || (group_lanes & (group_lanes - 1)) != 0) return -6;
    }
    if (a->rows == 0) return 0;
    if (!a->attn || !a->u || !a->norm_weight || !a->norm_bias || (joined_needed && !joined)) return -1;
    if ((((uintptr_t)a->attn | (uintptr_t)a->u | (uintptr_t)joined) & 15) != 0) return -4;
    if (!a->group_norm && (((uintptr_t)a->norm_weight | (uintptr_t)a->norm_bias) & 15) != 0) return -4;
    p.attn = (const char*)a->attn, p.u = (const char*)a->u, p.weight = (const char*)a->norm_weight, p.bias = (const char*)a->norm_bias;
    p.joined = (char*)joined;
    p.attn_rs = a->attn_row_stride, p.u_rs = a->u_row_stride, p.joined_rs = joined_rs, p.rows = a->rows;
    p.eps = a->norm_eps, p.d = d, p.group_lanes = group_lanes;
    const bool cu = blocks == 3 || (!a->group_norm && a->concat_u), cx = blocks == 3 || (!a->group_norm && a->concat_x);
    p.off_u = cu ? 0 : -1;
    p.off_x = cx ? (cu ? d : 0) : -1;
    p.off_y = (blocks - 1) * d;
    p.silu_u = a->silu_u ? 1 : 0, p.mul_act = a->mul_u_activation;
    p.width = (int64_t)blocks * d;
    if (!dropout_params(a->dropout_ratio, a->dropout_seed, a->dropout_offset, p.drop)) return -5;
    return 0;
}

}  // namespace hstu
