// C ABI of the backward pass (hstu_hip_mha_bwd): validation and launch of the two kernels of hstu_bwd_kernel.h.
// A translation unit of its own so that it compiles in parallel with the forward kernels.
#include "hstu_bwd_launch.h"

#include <cstdio>
#include <cstring>

extern "C" __attribute__((visibility("hidden"))) int hstu_hip_launch_rank(const void* offsets, int offsets_i64, int batch, int* order,
                                                                          void* stream);

namespace {

size_t align256(size_t x) { return (x + 255) & ~(size_t)255; }

// Bytes of the dS blocks: (total rows + 32 per sequence) x H x pitch32 x 64, pitch32 = 4 * ceil(max_seq_len / 128).
size_t ds_bytes(const HstuFwdArgs* a) {
    const size_t pitch32 = 4 * (((size_t)a->max_seq_len + 127) / 128);
    return ((size_t)a->total_q + 32 * (size_t)a->batch) * (size_t)a->heads * pitch32 * 64;
}

}  // namespace

extern "C" size_t hstu_hip_mha_bwd_workspace_bytes(const HstuFwdArgs* a) {
    if (!a || a->batch <= 0 || a->heads <= 0 || a->max_seq_len <= 0 || a->total_q <= 0) return 0;
    return align256((size_t)a->batch * sizeof(int)) + ds_bytes(a);
}

__attribute__((visibility("hidden"))) int hstu_bwd_params(const HstuFwdArgs* a, const HstuBwdGrads* g, int64_t grad_mask, hstu::BwdParams& bp, bool& nothing,
                                                          void* stream_) {
    nothing = true;
    if (!a || !g) return HSTU_ERR_NULL_POINTER;
    HstuFwdArgs c = *a;  // the forward's own checks, with the unused output standing in as any aligned pointer
    c.out = const_cast<void*>(a->q);
    c.o_row_stride = c.o_head_stride = 0;
    c.tile_config = 0;
    c.kv_splits = 0;
    int rc = hstu_hip_check_args(&c);
    if (rc != HSTU_OK) return rc;
    if (a->delta_size != 0) return HSTU_ERR_UNSUPPORTED;
    if (a->dtype != HSTU_BF16 && a->dtype != HSTU_FP16) return HSTU_ERR_UNSUPPORTED;
    // the kernels scale by 1 / max_seq_len: a caller with an attn_scale multiplies dout by attn_scale * max_seq_len
    // itself (a per-row factor commutes with everything behind it) and calls with attn_scale = NULL
    if (a->attn_scale) return HSTU_ERR_UNSUPPORTED;
    if (a->total_q == 0 || a->batch == 0) return HSTU_OK;
    if (!g->dout || !g->dq || !g->dk || !g->dv) return HSTU_ERR_NULL_POINTER;
    const uintptr_t ptrs = reinterpret_cast<uintptr_t>(g->dout) | reinterpret_cast<uintptr_t>(g->dq) |
                           reinterpret_cast<uintptr_t>(g->dk) | reinterpret_cast<uintptr_t>(g->dv);
    if ((ptrs & 15) != 0) return HSTU_ERR_MISALIGNED;
    const int64_t strides[8] = {g->do_row_stride, g->do_head_stride, g->dq_row_stride, g->dq_head_stride,
                                g->dk_row_stride, g->dk_head_stride, g->dv_row_stride, g->dv_head_stride};
    for (int i = 0; i < 8; ++i)
        if (strides[i] < 0 || (strides[i] & (i < 2 ? 7 : grad_mask)) != 0) return HSTU_ERR_MISALIGNED;
    if (!hstu_hip_device_is_gfx950()) return HSTU_ERR_BAD_DEVICE;
    nothing = false;

    memset(&bp, 0, sizeof(bp));
    hstu::FwdParams& p = bp.f;
    p.q = (const char*)a->q;
    p.k = (const char*)a->k;
    p.v = (const char*)a->v;
    p.q_rs = a->q_row_stride, p.q_hs = a->q_head_stride;
    p.k_rs = a->k_row_stride, p.k_hs = a->k_head_stride;
    p.v_rs = a->v_row_stride, p.v_hs = a->v_head_stride;
    p.offsets = a->seq_offsets;
    p.targets = a->num_targets;
    p.offsets_i64 = a->seq_offsets_i64;
    p.targets_i64 = a->num_targets_i64;
    p.B = a->batch;
    p.H = a->heads;
    p.max_seq_len = a->max_seq_len;
    p.w = a->max_attn_len;
    p.c = a->contextual_seq_len;
    p.f = a->min_full_attn_seq_len;
    p.kv_splits = 1;
    p.c1 = -a->alpha * 1.4426950408889634f;
    bp.gscale = a->alpha / (float)a->max_seq_len;
    bp.pscale = a->alpha == 0.0f ? 0.0f : -1.0f / ((float)a->max_seq_len * 1.4426950408889634f);
    bp.total_q = a->total_q;
    bp.dout = (const char*)g->dout;
    bp.dq = (char*)g->dq, bp.dk = (char*)g->dk, bp.dv = (char*)g->dv;
    bp.do_rs = g->do_row_stride, bp.do_hs = g->do_head_stride;
    bp.dq_rs = g->dq_row_stride, bp.dq_hs = g->dq_head_stride;
    bp.dk_rs = g->dk_row_stride, bp.dk_hs = g->dk_head_stride;
    bp.dv_rs = g->dv_row_stride, bp.dv_hs = g->dv_head_stride;

    p.num_mb = (a->max_seq_len + kBwdRows - 1) / kBwdRows;
    const long long pairs_per_xcd = ((long long)a->batch * a->heads + 7) / 8;
    const long long slots = pairs_per_xcd * p.num_mb;
    if (slots * 8 > 0x7fffffffLL) return HSTU_ERR_BAD_SHAPE;
    p.pairs_per_xcd = (int)pairs_per_xcd;
    p.slots_per_xcd = (int)slots;

    // `sort_by_length`: long sequences first (their blocks are the long-running ones); needs 4 * batch bytes of workspace
    // (not where all blocks start together, one workgroup per CU: 8 sequences of 150 rows, 2 heads, save the launch)
    if (a->sort_by_length && a->batch >= 2 && a->batch <= 8192 && slots * 8 > 256 && a->workspace &&
        (size_t)a->workspace_bytes >= (size_t)a->batch * sizeof(int)) {
        rc = hstu_hip_launch_rank(a->seq_offsets, a->seq_offsets_i64, a->batch, (int*)a->workspace, stream_);
        if (rc != HSTU_OK) return rc;
        p.order = (const int*)a->workspace;
    }
    // enough workspace for the dS blocks: the key-stationary kernel stores them and dQ is formed from them
    if (a->workspace && (size_t)a->workspace_bytes >= hstu_hip_mha_bwd_workspace_bytes(a) &&
        (reinterpret_cast<uintptr_t>(a->workspace) & 255) == 0) {
        bp.ds = (char*)a->workspace + align256((size_t)a->batch * sizeof(int));
        bp.ds_pitch32 = 4 * ((a->max_seq_len + 127) / 128);
    }
    return HSTU_OK;
}

extern "C" int hstu_hip_mha_bwd(const HstuFwdArgs* a, const HstuBwdGrads* g, void* stream) {
    hstu::BwdParams bp;
    bool nothing;
    const int rc = hstu_bwd_params(a, g, 7, bp, nothing, stream);
    if (rc != HSTU_OK || nothing) return rc;
    if (a->dtype == HSTU_BF16) return launch_bwd_dim<hstu::Bf16>(bp, a->dqk, a->dv, (hipStream_t)stream);
    return launch_bwd_dim<hstu::Fp16>(bp, a->dqk, a->dv, (hipStream_t)stream);
}
