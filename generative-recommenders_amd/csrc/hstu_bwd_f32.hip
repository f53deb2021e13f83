// C ABI of the backward pass with fp32 tensors (hstu_hip_mha_bwd_f32): the kernels take 16-bit operands, so q, k, v and dout are rounded to bf16 (fp32's
// range: dout can be tiny) by one launch, and dq, dk, dv are stored from the fp32 sums as they are.  Done by the caller that is four
// casts before and three behind, at 3 to 5 us each in a call whose kernels take 57 (16 sequences of 100 .. 768 rows).
#include "hstu_bwd_launch.h"

namespace {

// bf16 operands, fp32 gradients
struct Bf16F32 : hstu::Bf16 {
    typedef float out_elem;
};

// dst[row][h][0 .. d) (dense) = src[row * rs + h * hs + 0 .. d) (strides in elements), 8 elements per thread; the workgroups of an operand behind
// those of the one before it.
struct RoundParams {
    const float* src[4];
    __bf16* dst[4];
    int64_t rs[4], hs[4], rows[4];
    int d8[4];  // groups of 8 in a head
    unsigned first[4];
    int H;
};

template <class INDEX>
__global__ __launch_bounds__(256) void hstu_round_bf16_kernel(const RoundParams p) {
    const int which = blockIdx.x >= p.first[3] ? 3 : blockIdx.x >= p.first[2] ? 2 : blockIdx.x >= p.first[1] ? 1 : 0;
    const INDEX idx = (INDEX)(blockIdx.x - p.first[which]) * 256 + threadIdx.x, d8 = (INDEX)p.d8[which], H = (INDEX)p.H;
    if (idx >= (INDEX)p.rows[which] * H * d8) return;
    const INDEX rh = idx / d8, c = idx - rh * d8, row = rh / H, h = rh - row * H;
    const float* s = p.src[which] + (int64_t)row * p.rs[which] + (int64_t)h * p.hs[which] + (int64_t)c * 8;
    const hstu::f32x4_t a = *(const hstu::f32x4_t*)s, b = *(const hstu::f32x4_t*)(s + 4);
    hstu::bf16x8_t o;
#pragma unroll
    for (int i = 0; i < 4; ++i) o[i] = (__bf16)a[i], o[4 + i] = (__bf16)b[i];
    *(hstu::bf16x8_t*)(p.dst[which] + (int64_t)idx * 8) = o;
}

size_t align256(size_t x) { return (x + 255) & ~(size_t)255; }

}  // namespace

extern "C" size_t hstu_hip_mha_bwd_f32_copies_bytes(const HstuFwdArgs* a) {
    if (!a || a->heads <= 0 || a->dqk <= 0 || a->dv <= 0 || a->total_q <= 0 || a->total_kv <= 0) return 0;
    const size_t q = (size_t)a->total_q * a->heads * 2, kv = (size_t)a->total_kv * a->heads * 2;
    return align256(q * a->dqk) + align256(kv * a->dqk) + align256(kv * a->dv) + align256(q * a->dv);
}

extern "C" int hstu_hip_mha_bwd_f32(const HstuFwdArgs* a, const HstuBwdGrads* g, void* copies, int64_t copies_bytes, void* stream_) {
    if (!a || !g) return HSTU_ERR_NULL_POINTER;
    HstuFwdArgs c = *a;  // the forward's own checks, with the unused output standing in as any aligned pointer
    c.out = const_cast<void*>(a->q);
    c.o_row_stride = c.o_head_stride = 0;
    c.tile_config = c.kv_splits = 0;
    int rc = hstu_hip_check_args(&c);
    if (rc != HSTU_OK) return rc;
    if (a->dtype != HSTU_FP32 || a->delta_size != 0 || a->attn_scale) return HSTU_ERR_UNSUPPORTED;
    if (a->total_q == 0 || a->batch == 0) return HSTU_OK;
    if (!g->dout || !g->dq || !g->dk || !g->dv || !copies) return HSTU_ERR_NULL_POINTER;
    if (((reinterpret_cast<uintptr_t>(g->dout) | reinterpret_cast<uintptr_t>(copies)) & 15) != 0) return HSTU_ERR_MISALIGNED;
    if (g->do_row_stride < 0 || g->do_head_stride < 0 || ((g->do_row_stride | g->do_head_stride) & 3) != 0) return HSTU_ERR_MISALIGNED;
    if (copies_bytes < (int64_t)hstu_hip_mha_bwd_f32_copies_bytes(a)) return HSTU_ERR_BAD_SHAPE;
    hipStream_t stream = (hipStream_t)stream_;

    RoundParams p;
    const void* const src[4] = {a->q, a->k, a->v, g->dout};
    const int64_t rs[4] = {a->q_row_stride, a->k_row_stride, a->v_row_stride, g->do_row_stride};
    const int64_t hs[4] = {a->q_head_stride, a->k_head_stride, a->v_head_stride, g->do_head_stride};
    const int64_t rows[4] = {a->total_q, a->total_kv, a->total_kv, a->total_q};
    const int d[4] = {a->dqk, a->dqk, a->dv, a->dv};
    char* at = (char*)copies;
    long long blocks = 0;
    bool small = true;
    for (int i = 0; i < 4; ++i) {
        const int64_t groups = rows[i] * a->heads * (d[i] / 8);
        p.src[i] = (const float*)src[i], p.dst[i] = (__bf16*)at, p.rs[i] = rs[i], p.hs[i] = hs[i], p.rows[i] = rows[i], p.d8[i] = d[i] / 8;
        p.first[i] = (unsigned)blocks;
        blocks += (groups + 255) / 256;
        small = small && groups < 0x7fffffffLL;
        at += align256((size_t)rows[i] * a->heads * d[i] * 2);
    }
    if (blocks > 0x7fffffffLL) return HSTU_ERR_BAD_SHAPE;
    p.H = a->heads;

    c = *a;
    c.dtype = HSTU_BF16;
    c.q = p.dst[0], c.k = p.dst[1], c.v = p.dst[2];
    c.q_row_stride = c.k_row_stride = (int64_t)a->heads * a->dqk, c.q_head_stride = c.k_head_stride = a->dqk;
    c.v_row_stride = (int64_t)a->heads * a->dv, c.v_head_stride = a->dv;
    HstuBwdGrads g16 = *g;
    g16.dout = p.dst[3], g16.do_row_stride = c.v_row_stride, g16.do_head_stride = a->dv;
    hstu::BwdParams bp;
    bool nothing;
    rc = hstu_bwd_params(&c, &g16, 3, bp, nothing, stream_);
    if (rc != HSTU_OK || nothing) return rc;
    if (small) hipLaunchKernelGGL(hstu_round_bf16_kernel<unsigned>, dim3((unsigned)blocks), dim3(256), 0, stream, p);
    else hipLaunchKernelGGL(hstu_round_bf16_kernel<uint64_t>, dim3((unsigned)blocks), dim3(256), 0, stream, p);
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) {
        hstu_hip_set_last_error("rounding kernel launch", (int)e);
        return HSTU_ERR_LAUNCH;
    }
    return launch_bwd_dim<Bf16F32>(bp, a->dqk, a->dv, stream);
}
