// Native front of the operators: a Python module (`hstu_native`) that takes torch tensors, checks them, allocates the
// result and the scratch memory and calls the C ABI (hstu_hip.h, hstu_linear.h) -- the work that ops/*.py does through
// ctypes for every argument it has to look at, in a few microseconds instead of ten to thirty.
//
// The operators that are differentiable record a backward node of their own here (torch::autograd::Function): nothing but inputs
// is saved, the gradients come from the library's backward kernels and plain products.
//
// Every function serves the usual call only and returns nothing (None) for any other: tensors that need a copy first
// (rows not dense or not 16-byte aligned), dtypes it does not know, gradients it does not form, arguments the caller got
// wrong, HSTU_HIP_CHECK_CONTRACT, a status other than 0.  The Python operator then goes through its own checks and raises,
// copies or computes, so that every message and every rare case has one place.  Nothing is kept between calls.
#include <torch/extension.h>

#include <ATen/record_function.h>
#include <c10/core/DeviceGuard.h>
#include <c10/hip/HIPStream.h>

#include <cstdlib>
#include <optional>
#include <tuple>

#include "hstu_hip.h"
#include "hstu_linear.h"

namespace {

using at::Tensor;
using OptTensor = std::optional<Tensor>;
using torch::autograd::AutogradContext;
using torch::autograd::variable_list;

// Every backward node runs in one.  No graph, with create_graph too: the kernels' gradients are not differentiable.  And no autocast: the
// kernels read a product as the inputs' type, which autocast to another one would change.
struct BackwardScope {
    torch::NoGradGuard no_graph;
    c10::impl::ExcludeDispatchKeyGuard no_autocast{c10::autocast_dispatch_keyset};
};

struct Declined {};  // thrown where a call turns out, on the way, to be the Python operator's

void* stream_of(const Tensor& t) { return (void*)c10::hip::getCurrentHIPStream(t.get_device()).stream(); }

bool index_tensor(const Tensor& t) {
    return t.is_cuda() && t.is_contiguous() && (t.scalar_type() == at::kLong || t.scalar_type() == at::kInt);
}

bool wants_grad(std::initializer_list<const Tensor*> ts) {
    if (!at::GradMode::is_enabled()) return false;
    for (const Tensor* t : ts)
        if (t->requires_grad()) return true;
    return false;
}

bool contract_checks() {
    const char* e = getenv("HSTU_HIP_CHECK_CONTRACT");
    return e && e[0] && !(e[0] == '0' && !e[1]);
}

int attention_dtype(at::ScalarType t) {
    switch (t) {
        case at::kBFloat16: return HSTU_BF16;
        case at::kHalf: return HSTU_FP16;
        case at::kFloat8_e4m3fn: return HSTU_FP8_E4M3;
        case at::kFloat: return HSTU_FP32;
        default: return -1;
    }
}

// [rows, heads, dim] as the kernels read it: dense innermost, rows and heads on 16-byte boundaries
bool kernel_layout(const Tensor& t) {
    const int64_t per16 = 16 / t.element_size();
    return t.stride(2) == 1 && (reinterpret_cast<uintptr_t>(t.const_data_ptr()) & 15) == 0 && t.stride(0) % per16 == 0 &&
           t.stride(1) % per16 == 0 && t.stride(0) >= 0 && t.stride(1) >= 0;
}

struct AttentionCall {
    int64_t max_seq_len, delta, w, c, f;
    double alpha, q_scale, k_scale, v_scale;
    int64_t tile_config, kv_splits;
    bool sort;
};

// The operands' part of the argument block; `args` arrives zeroed.
void fill_attention(HstuFwdArgs& a, const Tensor& q, const Tensor& k, const Tensor& v, const Tensor& offsets, const OptTensor& targets,
                    const AttentionCall& call) {
    a.q = q.const_data_ptr(), a.k = k.const_data_ptr(), a.v = v.const_data_ptr();
    a.q_row_stride = q.stride(0), a.q_head_stride = q.stride(1);
    a.k_row_stride = k.stride(0), a.k_head_stride = k.stride(1);
    a.v_row_stride = v.stride(0), a.v_head_stride = v.stride(1);
    a.seq_offsets = offsets.const_data_ptr(), a.seq_offsets_i64 = offsets.scalar_type() == at::kLong;
    if (targets) a.num_targets = targets->const_data_ptr(), a.num_targets_i64 = targets->scalar_type() == at::kLong;
    a.batch = (int32_t)(offsets.numel() - 1);
    a.heads = (int32_t)q.size(1), a.dqk = (int32_t)q.size(2), a.dv = (int32_t)v.size(2);
    a.total_q = q.size(0), a.total_kv = k.size(0);
    a.max_seq_len = (int32_t)call.max_seq_len, a.delta_size = (int32_t)call.delta, a.alpha = (float)call.alpha;
    a.max_attn_len = (int32_t)call.w, a.contextual_seq_len = (int32_t)call.c, a.min_full_attn_seq_len = (int32_t)call.f;
    a.dtype = attention_dtype(q.scalar_type());
    a.q_scale = (float)call.q_scale, a.k_scale = (float)call.k_scale, a.v_scale = (float)call.v_scale;
    a.tile_config = (int32_t)call.tile_config, a.kv_splits = (int32_t)call.kv_splits, a.sort_by_length = call.sort;
}

// Launches the forward into `out`; the status of the C ABI.
int attention_forward(const Tensor& q, const Tensor& k, const Tensor& v, const Tensor& out, const Tensor& offsets, const OptTensor& targets,
                      const AttentionCall& call) {
    HstuFwdArgs a{};
    fill_attention(a, q, k, v, offsets, targets, call);
    a.out = out.data_ptr(), a.o_row_stride = out.stride(0), a.o_head_stride = out.stride(1);
    const size_t need = hstu_hip_workspace_bytes(&a);
    Tensor scratch;  // (the caching allocator keeps it from other streams' work until this stream has consumed it)
    if (need > 0) {
        scratch = at::empty({(int64_t)need}, q.options().dtype(at::kByte));
        a.workspace = scratch.data_ptr(), a.workspace_bytes = (int64_t)need;
    }
    const c10::DeviceGuard guard(q.device());
    return hstu_hip_mha_fwd(&a, stream_of(q));
}

bool index_operands(const Tensor& offsets, const OptTensor& targets) {
    if (!index_tensor(offsets) || offsets.dim() != 1 || offsets.numel() < 2) return false;
    return !targets || (index_tensor(*targets) && targets->numel() == offsets.numel() - 1);
}

bool attention_operands(const Tensor& q, const Tensor& k, const Tensor& v, const Tensor& offsets, const OptTensor& targets) {
    if (q.dim() != 3 || k.dim() != 3 || v.dim() != 3 || !q.is_cuda() || !k.is_cuda() || !v.is_cuda() || !index_operands(offsets, targets)) return false;
    if (attention_dtype(q.scalar_type()) < 0 || k.scalar_type() != q.scalar_type() || v.scalar_type() != q.scalar_type()) return false;
    if (k.size(1) != q.size(1) || k.size(2) != q.size(2) || v.size(0) != k.size(0) || v.size(1) != q.size(1)) return false;
    if (q.numel() == 0 || k.numel() == 0 || v.numel() == 0) return false;
    return kernel_layout(q) && kernel_layout(k) && kernel_layout(v) && !contract_checks();
}

at::ScalarType result_type(const Tensor& q) { return q.scalar_type() == at::kFloat8_e4m3fn ? at::kBFloat16 : q.scalar_type(); }

Tensor attention_result(const Tensor& q, const Tensor& k, const Tensor& v, const Tensor& offsets, const OptTensor& targets, const AttentionCall& call) {
    Tensor out = at::empty({v.size(0), v.size(1), v.size(2)}, v.options().dtype(result_type(q)));
    if (attention_forward(q, k, v, out, offsets, targets, call) != HSTU_OK) throw Declined();
    return out;
}

// dq, dk, dv (any rows the kernels can write) from dout.  `workspace`: the caller's dS scratch, else scores are recomputed.
void attention_backward(const Tensor& dout, const Tensor& q, const Tensor& k, const Tensor& v, const Tensor& dq, const Tensor& dk, const Tensor& dv,
                        const Tensor& offsets, const OptTensor& targets, AttentionCall call, const OptTensor& workspace) {
    HstuFwdArgs a{};
    call.tile_config = call.kv_splits = 0;
    call.sort = false;
    fill_attention(a, q, k, v, offsets, targets, call);
    Tensor scratch;
    if (workspace) {
        a.workspace = workspace->data_ptr(), a.workspace_bytes = workspace->numel(), a.sort_by_length = 1;
    } else if (a.batch >= 2) {
        scratch = at::empty({4 * (int64_t)a.batch}, q.options().dtype(at::kByte));
        a.workspace = scratch.data_ptr(), a.workspace_bytes = 4 * (int64_t)a.batch, a.sort_by_length = 1;
    }
    HstuBwdGrads g{};
    g.dout = dout.const_data_ptr(), g.dq = dq.data_ptr(), g.dk = dk.data_ptr(), g.dv = dv.data_ptr();
    g.do_row_stride = dout.stride(0), g.do_head_stride = dout.stride(1);
    g.dq_row_stride = dq.stride(0), g.dq_head_stride = dq.stride(1);
    g.dk_row_stride = dk.stride(0), g.dk_head_stride = dk.stride(1);
    g.dv_row_stride = dv.stride(0), g.dv_head_stride = dv.stride(1);
    const c10::DeviceGuard guard(q.device());
    int rc;
    if (q.scalar_type() == at::kFloat) {
        const int64_t bytes = (int64_t)hstu_hip_mha_bwd_f32_copies_bytes(&a);
        Tensor copies = at::empty({bytes}, q.options().dtype(at::kByte));
        rc = hstu_hip_mha_bwd_f32(&a, &g, copies.data_ptr(), bytes, stream_of(q));
    } else {
        rc = hstu_hip_mha_bwd(&a, &g, stream_of(q));
    }
    if (rc == HSTU_OK) return;
    // (the classes that the Python operators raise for a status)
    const std::string what = c10::str("hstu_hip: ", hstu_hip_status_string(rc), " (", hstu_hip_last_error(), ") [status ", rc, "]");
    TORCH_CHECK_VALUE(rc != HSTU_ERR_NULL_POINTER && rc != HSTU_ERR_BAD_SHAPE, what);
    TORCH_CHECK_NOT_IMPLEMENTED(rc != HSTU_ERR_UNSUPPORTED, what);
    TORCH_CHECK(false, what);
}

Tensor kernel_rows(const Tensor& t) { return kernel_layout(t) ? t : t.clone(at::MemoryFormat::Contiguous); }

std::vector<int64_t> pack(const AttentionCall& c) { return {c.max_seq_len, c.w, c.c, c.f}; }
AttentionCall unpack(const std::vector<int64_t>& i, double alpha) { return {i[0], 0, i[1], i[2], i[3], alpha, 1.0, 1.0, 1.0, 0, 0, false}; }

struct MhaFunction : torch::autograd::Function<MhaFunction> {
    static Tensor forward(AutogradContext* ctx, const Tensor& q, const Tensor& k, const Tensor& v, const Tensor& offsets, const OptTensor& targets,
                          const AttentionCall& call, const OptTensor& workspace) {
        Tensor out = attention_result(q, k, v, offsets, targets, call);
        ctx->save_for_backward({q, k, v, offsets, targets ? *targets : Tensor()});
        ctx->saved_data["call"] = pack(call);
        ctx->saved_data["alpha"] = call.alpha;
        if (workspace) ctx->saved_data["workspace"] = *workspace;
        return out;
    }
    static variable_list backward(AutogradContext* ctx, const variable_list& grads) {
        const BackwardScope scope;
        const auto saved = ctx->get_saved_variables();
        const Tensor q = kernel_rows(saved[0]), k = kernel_rows(saved[1]), v = kernel_rows(saved[2]);
        const OptTensor targets = saved[4].defined() ? OptTensor(saved[4].contiguous()) : OptTensor();
        const auto ws = ctx->saved_data.find("workspace");
        const OptTensor workspace = ws == ctx->saved_data.end() ? OptTensor() : OptTensor(ws->second.toTensor());
        const Tensor dout = kernel_rows(grads[0].to(q.scalar_type()));
        Tensor dq = at::empty_like(q, at::MemoryFormat::Contiguous), dk = at::empty_like(k, at::MemoryFormat::Contiguous),
               dv = at::empty_like(v, at::MemoryFormat::Contiguous);
        attention_backward(dout, q, k, v, dq, dk, dv, saved[3].contiguous(), targets,
                           unpack(ctx->saved_data["call"].toIntVector(), ctx->saved_data["alpha"].toDouble()), workspace);
        return {dq, dk, dv, Tensor(), Tensor(), Tensor(), Tensor()};
    }
};

OptTensor hstu_mha(int64_t max_seq_len, double alpha, const Tensor& q, const Tensor& k, const Tensor& v, const Tensor& offsets,
                   const OptTensor& targets, int64_t w, int64_t c, int64_t f, bool sort, double q_scale, double k_scale, double v_scale,
                   int64_t tile_config, int64_t kv_splits, const OptTensor& bwd_workspace) {
    if (max_seq_len <= 0 || !attention_operands(q, k, v, offsets, targets) || q.size(0) != k.size(0)) return {};
    const AttentionCall call{max_seq_len, 0, w, c, f, alpha, q_scale, k_scale, v_scale, tile_config, kv_splits, sort};
    const bool grad = wants_grad({&q, &k, &v});
    if (grad && q.scalar_type() == at::kFloat8_e4m3fn) return {};
    // (a workspace of the wrong kind is refused by the Python operator's backward)
    if (grad && bwd_workspace && (bwd_workspace->scalar_type() != at::kByte || !bwd_workspace->is_contiguous() || bwd_workspace->device() != q.device())) return {};
    RECORD_USER_SCOPE("hstu_mha");
    try {
        return grad ? MhaFunction::apply(q, k, v, offsets, targets, call, bwd_workspace) : attention_result(q, k, v, offsets, targets, call);
    } catch (const Declined&) {
        return {};
    }
}

OptTensor delta_hstu_mha(int64_t max_seq_len, double alpha, const Tensor& q, const Tensor& k, const Tensor& v, const Tensor& offsets,
                         const OptTensor& targets, int64_t w, int64_t c, double q_scale, double k_scale, double v_scale, int64_t tile_config,
                         int64_t kv_splits) {
    if (max_seq_len <= 0 || !attention_operands(q, k, v, offsets, targets) || wants_grad({&q, &k, &v})) return {};
    const int64_t batch = offsets.numel() - 1;
    if (q.size(0) % batch != 0) return {};
    RECORD_USER_SCOPE("delta_hstu_mha");
    Tensor out = at::empty({q.size(0), v.size(1), v.size(2)}, q.options().dtype(result_type(q)));
    const AttentionCall call{max_seq_len, q.size(0) / batch, w, c, 0, alpha, q_scale, k_scale, v_scale, tile_config, kv_splits, false};
    if (attention_forward(q, k, v, out, offsets, targets, call) != HSTU_OK) return {};
    return out;
}

// ---- row copies ---------------------------------------------------------------------------------------------------------

void fill_side(const OptTensor& offsets, const void*& ptr, int32_t& i64) {
    if (offsets) ptr = offsets->const_data_ptr(), i64 = offsets->scalar_type() == at::kLong;
}

int jagged_copy(bool split, const Tensor& left, const Tensor& right, const Tensor& joined, const OptTensor& offsets_left,
                const OptTensor& offsets_right, int64_t batch, int64_t max_left, int64_t max_right) {
    HstuJaggedCopyArgs a{};
    const int64_t es = joined.element_size();
    auto pitch = [es](const Tensor& t) { return (t.size(0) > 1 ? t.stride(0) : t.size(1)) * es; };
    a.left = left.data_ptr(), a.right = right.data_ptr(), a.joined = joined.data_ptr();
    a.left_row_stride = pitch(left), a.right_row_stride = pitch(right), a.joined_row_stride = pitch(joined);
    a.row_bytes = joined.size(1) * es;
    fill_side(offsets_left, a.offsets_left, a.offsets_left_i64);
    fill_side(offsets_right, a.offsets_right, a.offsets_right_i64);
    a.batch = (int32_t)batch, a.max_len_left = (int32_t)max_left, a.max_len_right = (int32_t)max_right;
    a.total_left = left.size(0), a.total_right = right.size(0);
    const c10::DeviceGuard guard(joined.device());
    return split ? hstu_hip_split_2d_jagged(&a, stream_of(joined)) : hstu_hip_concat_2d_jagged(&a, stream_of(joined));
}

bool rows_2d(const Tensor& t) { return t.dim() == 2 && t.is_cuda() && t.stride(1) == 1 && t.numel() > 0; }
bool optional_index(const OptTensor& t) { return !t || (index_tensor(*t) && t->dim() == 1 && t->numel() > 1); }

OptTensor concat_2d_jagged(const Tensor& left, const Tensor& right, std::optional<int64_t> max_left, std::optional<int64_t> max_right,
                           const OptTensor& offsets_left, const OptTensor& offsets_right) {
    if (!rows_2d(left) || !rows_2d(right) || left.size(1) != right.size(1) || left.scalar_type() != right.scalar_type()) return {};
    if (!max_left || !max_right || *max_left <= 0 || *max_right <= 0 || !optional_index(offsets_left) || !optional_index(offsets_right)) return {};
    if (wants_grad({&left, &right})) return {};
    const int64_t batch = offsets_right ? offsets_right->numel() - 1 : right.size(0) / *max_right;
    if (offsets_left ? batch != offsets_left->numel() - 1 : batch != left.size(0) / *max_left) return {};
    Tensor out = at::empty({left.size(0) + right.size(0), left.size(1)}, left.options());
    if (jagged_copy(false, left, right, out, offsets_left, offsets_right, batch, *max_left, *max_right) != HSTU_OK) return {};
    return out;
}

std::optional<std::tuple<Tensor, Tensor>> split_2d_jagged(const Tensor& values, std::optional<int64_t> total_left,
                                                          std::optional<int64_t> total_right, std::optional<int64_t> max_left,
                                                          std::optional<int64_t> max_right, const OptTensor& offsets_left,
                                                          const OptTensor& offsets_right) {
    if (!rows_2d(values) || wants_grad({&values}) || !max_left || !max_right || *max_left < 0 || *max_right < 0) return {};
    if (!optional_index(offsets_left) || !optional_index(offsets_right) || (!offsets_left && !offsets_right)) return {};
    const int64_t batch = (offsets_left ? offsets_left->numel() : offsets_right->numel()) - 1, total = values.size(0);
    int64_t left_rows, right_rows;
    if (!offsets_left) {
        left_rows = *max_left * batch, right_rows = total - left_rows;
    } else if (!offsets_right) {
        right_rows = *max_right * batch, left_rows = total - right_rows;
    } else {
        if (!total_left || !total_right || *total_left + *total_right != total || offsets_right->numel() != offsets_left->numel()) return {};
        left_rows = *total_left, right_rows = *total_right;
    }
    if (left_rows < 0 || right_rows < 0) return {};
    Tensor left = at::empty({left_rows, values.size(1)}, values.options()), right = at::empty({right_rows, values.size(1)}, values.options());
    if (jagged_copy(true, left, right, values, offsets_left, offsets_right, batch, *max_left, *max_right) != HSTU_OK) return {};
    return std::make_tuple(left, right);
}

bool write_kv_tail(const Tensor& full, const Tensor& offsets, const Tensor& tail) {
    if (!rows_2d(full) || !rows_2d(tail) || full.size(1) != tail.size(1) || full.scalar_type() != tail.scalar_type()) return false;
    if (!index_tensor(offsets) || offsets.dim() != 1 || offsets.numel() < 2 || tail.size(0) % (offsets.numel() - 1) != 0) return false;
    const int64_t es = full.element_size(), batch = offsets.numel() - 1;
    const c10::DeviceGuard guard(full.device());
    return hstu_hip_jagged_write_tail(full.data_ptr(), full.stride(0) * es, offsets.const_data_ptr(), offsets.scalar_type() == at::kLong,
                                      tail.const_data_ptr(), tail.stride(0) * es, full.size(1) * es, (int32_t)batch,
                                      (int32_t)(tail.size(0) / batch), stream_of(full)) == HSTU_OK;
}

// ---- dense steps --------------------------------------------------------------------------------------------------------

int dense_dtype(const Tensor& t) { return t.scalar_type() == at::kBFloat16 ? 0 : t.scalar_type() == at::kHalf ? 1 : -1; }
bool aligned16(const Tensor& t) { return (reinterpret_cast<uintptr_t>(t.const_data_ptr()) & 15) == 0; }
// a parameter as the kernels read it: dense, 16-byte aligned, of x's type
bool parameter(const Tensor& t, const Tensor& x) { return t.is_cuda() && t.scalar_type() == x.scalar_type() && t.is_contiguous() && aligned16(t); }
// rows of a matrix: dense innermost, every row on a 16-byte boundary
bool matrix_rows(const Tensor& t) {
    return t.dim() == 2 && t.is_cuda() && t.size(0) > 0 && t.stride(1) == 1 && t.stride(0) >= t.size(1) && t.stride(0) % 8 == 0 && aligned16(t);
}

// An incoming gradient as the kernels read it.  (contiguous() is no help: a view of a flat gradient at an odd offset and a single
// row of any row stride are contiguous.)
Tensor gradient_rows(const Tensor& t) { return matrix_rows(t) ? t : t.clone(at::MemoryFormat::Contiguous); }
Tensor dense_gradient(const Tensor& t) {
    return t.stride(1) == 1 && t.stride(0) == t.size(1) && aligned16(t) ? t : t.clone(at::MemoryFormat::Contiguous);
}

// Saved tensors as the kernels read them: what saved-tensor hooks give back has the values of what was saved, in any layout.
Tensor saved_rows(const Tensor& t) { return gradient_rows(t); }
Tensor saved_dense(const Tensor& t) { return t.is_contiguous() && aligned16(t) ? t : t.clone(at::MemoryFormat::Contiguous); }

Tensor aligned_scratch(size_t bytes, const Tensor& like, void** ptr) {
    Tensor t = at::empty({(int64_t)bytes + 256}, like.options().dtype(at::kByte));
    *ptr = reinterpret_cast<void*>((reinterpret_cast<uintptr_t>(t.data_ptr()) + 255) & ~(uintptr_t)255);
    return t;
}

// u [L, hidden * H], q, k [L, H, attn], v [L, H, hidden] as views of the buffer u | v | q | k
std::tuple<Tensor, Tensor, Tensor, Tensor> uqvk_views(const Tensor& buf, int64_t heads, int64_t attn, int64_t hidden) {
    const int64_t rows = buf.size(0), pitch = buf.size(1), nu = hidden * heads, na = attn * heads;
    const at::AutoDispatchBelowADInplaceOrView below;
    auto view = [&](at::IntArrayRef sizes, at::IntArrayRef strides, int64_t offset) {
        Tensor t = buf.as_strided(sizes, strides, offset);
        // a change through one of them is a change of the buffer that a backward node has saved
        if (!buf.is_inference()) t.unsafeGetTensorImpl()->set_version_counter(buf.unsafeGetTensorImpl()->version_counter());
        return t;
    };
    return {view({rows, nu}, {pitch, 1}, 0), view({rows, heads, attn}, {pitch, attn, 1}, 2 * nu),
            view({rows, heads, attn}, {pitch, attn, 1}, 2 * nu + na), view({rows, heads, hidden}, {pitch, hidden, 1}, nu)};
}

struct UqvkShape {
    int64_t heads, attn, hidden;
    int64_t n_u() const { return hidden * heads; }
    int64_t n_out() const { return (2 * hidden + 2 * attn) * heads; }
};

bool uqvk_operands(const Tensor& x, const Tensor& norm_weight, const Tensor& norm_bias, const Tensor& weight, const Tensor& bias, const UqvkShape& s) {
    if (!matrix_rows(x) || dense_dtype(x) < 0 || s.heads <= 0 || s.attn <= 0 || s.hidden <= 0) return false;
    if (weight.dim() != 2 || weight.size(0) != x.size(1) || weight.size(1) != s.n_out() || bias.dim() != 1 || bias.size(0) != s.n_out()) return false;
    if (norm_weight.dim() != 1 || norm_weight.size(0) != x.size(1) || norm_bias.dim() != 1 || norm_bias.size(0) != x.size(1)) return false;
    return parameter(norm_weight, x) && parameter(norm_bias, x) && parameter(weight, x) && parameter(bias, x);
}

// The buffer u | v | q | k, u through SiLU.
Tensor uqvk_buffer(const Tensor& x, const Tensor& norm_weight, const Tensor& norm_bias, const Tensor& weight, const Tensor& bias, double eps,
                   const UqvkShape& s, int64_t path) {
    Tensor buf = at::empty({x.size(0), s.n_out()}, x.options());
    HstuUqvkArgs a{};
    a.x = x.const_data_ptr(), a.x_row_stride = x.stride(0);
    a.norm_weight = norm_weight.const_data_ptr(), a.norm_bias = norm_bias.const_data_ptr(), a.norm_eps = (float)eps;
    a.uvqk_weight = weight.const_data_ptr(), a.uvqk_bias = bias.const_data_ptr(), a.uvqk = buf.data_ptr();
    a.rows = x.size(0), a.d_model = (int32_t)x.size(1);
    a.heads = (int32_t)s.heads, a.attn_dim = (int32_t)s.attn, a.hidden_dim = (int32_t)s.hidden;
    a.dtype = dense_dtype(x), a.path = (int32_t)path;
    const size_t need = hstu_uqvk_workspace_bytes(&a);
    Tensor scratch;
    if (need > 0) scratch = aligned_scratch(need, x, &a.workspace), a.workspace_bytes = (int64_t)need;
    const c10::DeviceGuard guard(x.device());
    if (hstu_uqvk_forward(&a, stream_of(x)) != 0) throw Declined();
    return buf;
}

// what the weight gradient takes: result columns (wider ones get their gradients from the Python operator)
constexpr int64_t kWeightGradColumns = 65536;

void check_linear(int rc) { TORCH_CHECK(rc == 0, "hstu_linear: status ", rc, " (", hstu_linear_last_error(), ")"); }

// a @ weight^T.  The shapes that are not the kernels' are the framework's product, which chooses for these rows: the library's plans are made for a size class
// by the first rows that it sees, so that a gradient would depend on the batches before it, and asking for every batch costs the host 64 us.
Tensor product_t(const Tensor& a, const Tensor& weight) {
    const int64_t rows = a.size(0), n = weight.size(0);
    const int32_t k = (int32_t)a.size(1);
    if (hstu_linear_product_t_workspace_bytes(rows, k, (int32_t)n) > 0) return at::mm(a, weight.t());
    Tensor out = at::empty({rows, n}, a.options());
    check_linear(hstu_linear_product_t(a.const_data_ptr(), a.stride(0), weight.const_data_ptr(), weight.stride(0), rows, k, (int32_t)n, dense_dtype(a),
                                       out.data_ptr(), n, nullptr, 0, stream_of(a)));
    return out;
}

// a^T @ b, and the column sums of b where `b_sums` is defined.
Tensor weight_grad(const Tensor& a, const Tensor& b, const Tensor& b_sums) {
    Tensor out = at::empty({a.size(1), b.size(1)}, a.options());
    const int32_t m = (int32_t)a.size(1), n = (int32_t)b.size(1);
    const int64_t need = (int64_t)hstu_linear_weight_grad_workspace_bytes(m, n, a.size(0), a.stride(0), b.stride(0));
    Tensor scratch = at::empty({need}, a.options().dtype(at::kByte));
    check_linear(hstu_linear_weight_grad(a.const_data_ptr(), a.stride(0), m, b.const_data_ptr(), b.stride(0), n, a.size(0), dense_dtype(a),
                                         out.data_ptr(), b_sums.defined() ? b_sums.data_ptr() : nullptr, scratch.data_ptr(), need, stream_of(a)));
    return out;
}

// Gradients of x, norm_weight, norm_bias, weight, bias (those of `ctx`'s first five inputs that are wanted) from `d`, the gradient of
// the producer's buffer u | v | q | k: its v, q and k columns are filled in, the u columns are formed here from `du` (the gradient
// behind SiLU; undefined: zero).
variable_list uqvk_backward(const AutogradContext* ctx, const Tensor& x, const Tensor& norm_weight, const Tensor& norm_bias, const Tensor& weight,
                            const Tensor& bias, double eps, int64_t n_u, Tensor d, Tensor du) {
    const bool rows_wanted = ctx->needs_input_grad(0) || ctx->needs_input_grad(1) || ctx->needs_input_grad(2);
    const bool weight_wanted = ctx->needs_input_grad(3) || ctx->needs_input_grad(4);
    const int64_t rows = x.size(0), dm = x.size(1);
    const c10::DeviceGuard guard(x.device());
    void* stream = stream_of(x);
    variable_list got(5);
    Tensor d_u = d.narrow(1, 0, n_u);
    Tensor normed;
    if (weight_wanted) normed = at::empty({rows, dm}, x.options());
    bool u_done = !du.defined(), normed_done = false;
    if (u_done) {
        d_u.zero_();
    } else {
        du = gradient_rows(du);
        const int rc = hstu_uqvk_u_grad(x.const_data_ptr(), x.stride(0), norm_weight.const_data_ptr(), norm_bias.const_data_ptr(), (float)eps,
                                        weight.const_data_ptr(), weight.stride(0), bias.const_data_ptr(), du.const_data_ptr(), du.stride(0), d_u.data_ptr(),
                                        d_u.stride(0), weight_wanted ? normed.data_ptr() : nullptr, rows, (int32_t)dm, (int32_t)n_u, dense_dtype(x), stream);
        if (rc != -6 && rc != -5) check_linear(rc);  // (another shape: the product and what follows it below)
        u_done = normed_done = rc == 0;
    }
    if (!normed_done && (!u_done || weight_wanted)) {
        if (!normed.defined()) normed = at::empty({rows, dm}, x.options());
        check_linear(hstu_uqvk_layer_norm(x.const_data_ptr(), x.stride(0), norm_weight.const_data_ptr(), norm_bias.const_data_ptr(), (float)eps,
                                          normed.data_ptr(), dm, rows, (int32_t)dm, dense_dtype(x), stream));
    }
    if (!u_done) {
        at::mm_out(d_u, normed, weight.narrow(1, 0, n_u));
        check_linear(hstu_uqvk_silu_bwd(d_u.data_ptr(), d_u.stride(0), bias.const_data_ptr(), du.const_data_ptr(), du.stride(0), rows, n_u,
                                        dense_dtype(x), stream));
    }
    if (rows_wanted) {
        Tensor dy = product_t(d, weight);
        got[0] = at::empty({rows, dm}, x.options()), got[1] = at::empty_like(norm_weight), got[2] = at::empty_like(norm_bias);
        const int64_t need = (int64_t)hstu_uqvk_layer_norm_bwd_workspace_bytes(rows, (int32_t)dm);
        Tensor scratch = at::empty({need}, x.options().dtype(at::kByte));
        check_linear(hstu_uqvk_layer_norm_bwd(x.const_data_ptr(), x.stride(0), norm_weight.const_data_ptr(), (float)eps, dy.const_data_ptr(), dm,
                                              got[0].data_ptr(), dm, got[1].data_ptr(), got[2].data_ptr(), rows, (int32_t)dm, dense_dtype(x),
                                              scratch.data_ptr(), need, stream));
    }
    if (weight_wanted) {
        got[4] = at::empty_like(bias);
        got[3] = weight_grad(normed, d, got[4]);
    }
    return got;
}

struct UqvkFunction : torch::autograd::Function<UqvkFunction> {
    static variable_list forward(AutogradContext* ctx, const Tensor& x, const Tensor& norm_weight, const Tensor& norm_bias, const Tensor& weight,
                                 const Tensor& bias, double eps, const UqvkShape& s, int64_t path) {
        Tensor buf = uqvk_buffer(x, norm_weight, norm_bias, weight, bias, eps, s, path);
        ctx->save_for_backward({x, norm_weight, norm_bias, weight, bias});
        ctx->saved_data["shape"] = std::vector<int64_t>{s.heads, s.attn, s.hidden};
        ctx->saved_data["eps"] = eps;
        ctx->set_materialize_grads(false);
        auto [u, q, k, v] = uqvk_views(buf, s.heads, s.attn, s.hidden);
        return {u, q, k, v};
    }
    static variable_list backward(AutogradContext* ctx, const variable_list& grads) {
        const BackwardScope scope;
        const auto saved = ctx->get_saved_variables();
        const auto i = ctx->saved_data["shape"].toIntVector();
        const UqvkShape s{i[0], i[1], i[2]};
        Tensor d = at::empty({saved[0].size(0), s.n_out()}, saved[0].options());
        auto views = uqvk_views(d, s.heads, s.attn, s.hidden);
        auto put = [](Tensor to, const Tensor& from) { from.defined() ? to.copy_(from) : to.zero_(); };
        put(std::get<1>(views), grads[1]);
        put(std::get<2>(views), grads[2]);
        put(std::get<3>(views), grads[3]);
        variable_list got = uqvk_backward(ctx, saved_rows(saved[0]), saved_dense(saved[1]), saved_dense(saved[2]), saved_dense(saved[3]),
                                          saved_dense(saved[4]), ctx->saved_data["eps"].toDouble(), s.n_u(), d, grads[0]);
        got.resize(8);
        return got;
    }
};

// Producer and attention as one node: the attention's gradients are written straight into the producer's gradient buffer.
struct PreprocessFunction : torch::autograd::Function<PreprocessFunction> {
    static variable_list forward(AutogradContext* ctx, const Tensor& x, const Tensor& norm_weight, const Tensor& norm_bias, const Tensor& weight,
                                 const Tensor& bias, const Tensor& offsets, const OptTensor& targets, double eps, const UqvkShape& s,
                                 const AttentionCall& call) {
        Tensor buf = uqvk_buffer(x, norm_weight, norm_bias, weight, bias, eps, s, 0);
        auto [u, q, k, v] = uqvk_views(buf, s.heads, s.attn, s.hidden);
        Tensor out = attention_result(q, k, v, offsets, targets, call).view({x.size(0), s.n_u()});
        ctx->save_for_backward({x, norm_weight, norm_bias, weight, bias, offsets, targets ? *targets : Tensor(), buf});
        ctx->saved_data["shape"] = std::vector<int64_t>{s.heads, s.attn, s.hidden};
        ctx->saved_data["call"] = pack(call);
        ctx->saved_data["alpha"] = call.alpha;
        ctx->saved_data["eps"] = eps;
        ctx->set_materialize_grads(false);
        return {u, out, k, v};
    }
    static variable_list backward(AutogradContext* ctx, const variable_list& grads) {
        const BackwardScope scope;
        const auto saved = ctx->get_saved_variables();
        const auto i = ctx->saved_data["shape"].toIntVector();
        const UqvkShape s{i[0], i[1], i[2]};
        const Tensor x = saved_rows(saved[0]), offsets = saved[5].contiguous(), buf = saved_dense(saved[7]);
        const OptTensor targets = saved[6].defined() ? OptTensor(saved[6].contiguous()) : OptTensor();
        Tensor d = at::empty({x.size(0), s.n_out()}, x.options());
        const auto grad = uqvk_views(d, s.heads, s.attn, s.hidden), value = uqvk_views(buf, s.heads, s.attn, s.hidden);
        const Tensor &dq = std::get<1>(grad), &dk = std::get<2>(grad), &dv = std::get<3>(grad);
        if (grads[1].defined()) {
            const Tensor dout = kernel_rows(grads[1].reshape({x.size(0), s.heads, s.hidden}));
            attention_backward(dout, std::get<1>(value), std::get<2>(value), std::get<3>(value), dq, dk, dv, offsets, targets,
                               unpack(ctx->saved_data["call"].toIntVector(), ctx->saved_data["alpha"].toDouble()), {});
            if (grads[2].defined()) dk.add_(grads[2]);
            if (grads[3].defined()) dv.add_(grads[3]);
        } else {
            dq.zero_();
            grads[2].defined() ? dk.copy_(grads[2]) : dk.zero_();
            grads[3].defined() ? dv.copy_(grads[3]) : dv.zero_();
        }
        variable_list got = uqvk_backward(ctx, x, saved_dense(saved[1]), saved_dense(saved[2]), saved_dense(saved[3]), saved_dense(saved[4]),
                                          ctx->saved_data["eps"].toDouble(), s.n_u(), d, grads[0]);
        got.resize(10);
        return got;
    }
};

typedef std::tuple<Tensor, Tensor, Tensor, Tensor> FourTensors;

std::optional<FourTensors> compute_uqvk(const Tensor& x, const Tensor& norm_weight, const Tensor& norm_bias, double eps, int64_t heads, int64_t attn,
                                        int64_t hidden, const Tensor& weight, const Tensor& bias, int64_t path) {
    const UqvkShape s{heads, attn, hidden};
    if (!uqvk_operands(x, norm_weight, norm_bias, weight, bias, s)) return {};
    try {
        if (wants_grad({&x, &norm_weight, &norm_bias, &weight, &bias})) {
            if (s.n_out() > kWeightGradColumns) return {};
            const variable_list o = UqvkFunction::apply(x, norm_weight, norm_bias, weight, bias, eps, s, path);
            return FourTensors(o[0], o[1], o[2], o[3]);
        }
        return uqvk_views(uqvk_buffer(x, norm_weight, norm_bias, weight, bias, eps, s, path), heads, attn, hidden);
    } catch (const Declined&) {
        return {};
    }
}

// Whether the attention will take the views of a producer's buffer: asked before the producer runs, which the Python operators
// would otherwise repeat.  The library looks at sizes, strides and alignment alone; the buffer is allocated, so it is aligned
// as x is here.
bool attention_takes(const Tensor& x, const UqvkShape& s, const Tensor& offsets, const OptTensor& targets, const AttentionCall& call) {
    if (!index_operands(offsets, targets) || contract_checks()) return false;
    HstuFwdArgs a{};
    a.q = a.k = a.v = x.const_data_ptr(), a.out = const_cast<void*>(x.const_data_ptr());
    a.q_row_stride = a.k_row_stride = a.v_row_stride = s.n_out(), a.o_row_stride = s.n_u();
    a.q_head_stride = a.k_head_stride = s.attn, a.v_head_stride = a.o_head_stride = s.hidden;
    a.seq_offsets = offsets.const_data_ptr();
    a.batch = (int32_t)(offsets.numel() - 1), a.heads = (int32_t)s.heads, a.dqk = (int32_t)s.attn, a.dv = (int32_t)s.hidden;
    a.total_q = a.total_kv = x.size(0);
    a.max_seq_len = (int32_t)call.max_seq_len, a.max_attn_len = (int32_t)call.w, a.contextual_seq_len = (int32_t)call.c;
    a.dtype = attention_dtype(x.scalar_type());
    return hstu_hip_check_args(&a) == HSTU_OK;
}

// Producer and attention with gradients: (u, attention output [L, hidden * H], k, v).  Without gradients the two operators do.
std::optional<FourTensors> preprocess_and_attention(const Tensor& x, const Tensor& norm_weight, const Tensor& norm_bias, double eps, int64_t heads,
                                                    int64_t attn, int64_t hidden, const Tensor& weight, const Tensor& bias, int64_t max_seq_len,
                                                    const Tensor& offsets, double alpha, const OptTensor& targets, int64_t w, int64_t c, bool sort) {
    const UqvkShape s{heads, attn, hidden};
    if (max_seq_len <= 0 || !wants_grad({&x, &norm_weight, &norm_bias, &weight, &bias})) return {};
    if (!uqvk_operands(x, norm_weight, norm_bias, weight, bias, s) || s.n_out() > kWeightGradColumns) return {};
    const AttentionCall call{max_seq_len, 0, w, c, 0, alpha, 1.0, 1.0, 1.0, 0, 0, sort};
    if (!attention_takes(x, s, offsets, targets, call)) return {};
    RECORD_USER_SCOPE("hstu_preprocess_and_attention");
    try {
        const variable_list o = PreprocessFunction::apply(x, norm_weight, norm_bias, weight, bias, offsets, targets, eps, s, call);
        return FourTensors(o[0], o[1], o[2], o[3]);
    } catch (const Declined&) {
        return {};
    }
}

struct OutputCall {
    int64_t heads, linear_dim, activation, path;
    bool concat_u, concat_x, group_norm;
    double eps, dropout;
    uint64_t seed, offset;
    int64_t blocks() const { return group_norm ? (concat_u && concat_x ? 3 : 1) : 1 + concat_u + concat_x; }
};

void fill_output(HstuOutputArgs& a, const Tensor& attn, const Tensor& u, const Tensor& norm_weight, const Tensor& norm_bias, const OutputCall& c) {
    a.attn = attn.const_data_ptr(), a.attn_row_stride = attn.stride(0), a.u = u.const_data_ptr(), a.u_row_stride = u.stride(0);
    a.norm_weight = norm_weight.const_data_ptr(), a.norm_bias = norm_bias.const_data_ptr(), a.norm_eps = (float)c.eps;
    a.rows = attn.size(0), a.heads = (int32_t)c.heads, a.linear_dim = (int32_t)c.linear_dim;
    a.concat_u = c.concat_u, a.concat_x = c.concat_x, a.group_norm = c.group_norm, a.mul_u_activation = (int32_t)c.activation;
    a.dtype = dense_dtype(attn), a.path = (int32_t)c.path;
    a.dropout_ratio = (float)c.dropout, a.dropout_seed = c.seed, a.dropout_offset = c.offset;
}

Tensor output_result(const Tensor& attn, const Tensor& u, const Tensor& x, const Tensor& norm_weight, const Tensor& norm_bias, const Tensor& weight,
                     const OutputCall& c) {
    Tensor out = at::empty({x.size(0), x.size(1)}, x.options());
    HstuOutputArgs a{};
    fill_output(a, attn, u, norm_weight, norm_bias, c);
    a.x = x.const_data_ptr(), a.x_row_stride = x.stride(0), a.output_weight = weight.const_data_ptr(), a.out = out.data_ptr();
    a.d_out = (int32_t)x.size(1);
    const size_t need = hstu_output_workspace_bytes(&a);
    Tensor scratch;
    if (need > 0) scratch = aligned_scratch(need, x, &a.workspace), a.workspace_bytes = (int64_t)need;
    const c10::DeviceGuard guard(x.device());
    if (hstu_output_forward(&a, stream_of(x)) != 0) throw Declined();
    return out;
}

struct OutputFunction : torch::autograd::Function<OutputFunction> {
    static Tensor forward(AutogradContext* ctx, const Tensor& attn, const Tensor& u, const Tensor& x, const Tensor& norm_weight, const Tensor& norm_bias,
                          const Tensor& weight, const OutputCall& c) {
        Tensor out = output_result(attn, u, x, norm_weight, norm_bias, weight, c);
        ctx->save_for_backward({attn, u, norm_weight, norm_bias, weight});
        ctx->saved_data["sizes"] = std::vector<int64_t>{c.heads, c.linear_dim, c.activation, c.concat_u, c.concat_x, c.group_norm, (int64_t)c.seed,
                                                        (int64_t)c.offset};
        ctx->saved_data["floats"] = std::vector<double>{c.eps, c.dropout};
        return out;
    }
    static variable_list backward(AutogradContext* ctx, const variable_list& grads) {
        const BackwardScope scope;
        const auto saved = ctx->get_saved_variables();
        const Tensor attn = saved_rows(saved[0]), u = saved_rows(saved[1]), norm_weight = saved_dense(saved[2]), norm_bias = saved_dense(saved[3]),
                     weight = saved_dense(saved[4]);
        const auto i = ctx->saved_data["sizes"].toIntVector();
        const auto f = ctx->saved_data["floats"].toDoubleVector();
        const OutputCall c{i[0], i[1], i[2], 0, i[3] != 0, i[4] != 0, i[5] != 0, f[0], f[1], (uint64_t)i[6], (uint64_t)i[7]};
        const Tensor dout = dense_gradient(grads[0]);
        const int64_t rows = attn.size(0), width = attn.size(1);
        variable_list got(7);
        // The residual: the tensor that came in, for a leaf's accumulation to see that others hold it too and copy it.  (Another
        // tensor on the same memory would be taken over, and the next gradient added into the caller's.)
        got[2] = grads[0].requires_grad() ? grads[0].clone() : grads[0];
        const bool weight_too = ctx->needs_input_grad(5);
        if (ctx->needs_input_grad(0) || ctx->needs_input_grad(1) || ctx->needs_input_grad(3) || ctx->needs_input_grad(4)) {
            const c10::DeviceGuard guard(attn.device());
            const Tensor dj = product_t(dout, weight);
            Tensor joined = weight_too ? at::empty_like(dj) : Tensor();
            got[0] = at::empty({rows, width}, attn.options()), got[1] = at::empty({rows, width}, attn.options());
            got[3] = at::empty_like(norm_weight), got[4] = at::empty_like(norm_bias);
            HstuOutputArgs a{};
            fill_output(a, attn, u, norm_weight, norm_bias, c);
            HstuNormMulGrads g{};
            g.d_joined = dj.const_data_ptr(), g.d_joined_row_stride = dj.size(1);
            if (weight_too) g.joined = joined.data_ptr(), g.joined_row_stride = joined.size(1);
            g.d_attn = got[0].data_ptr(), g.d_u = got[1].data_ptr(), g.d_attn_row_stride = g.d_u_row_stride = width;
            g.d_norm_weight = got[3].data_ptr(), g.d_norm_bias = got[4].data_ptr();
            g.workspace_bytes = (int64_t)hstu_output_norm_mul_bwd_workspace_bytes(&a);
            Tensor scratch = at::empty({g.workspace_bytes}, attn.options().dtype(at::kByte));
            g.workspace = scratch.data_ptr();
            check_linear(hstu_output_norm_mul_bwd(&a, &g, stream_of(attn)));
            if (weight_too) got[5] = weight_grad(joined, dout, Tensor());
        } else if (weight_too) {
            const c10::DeviceGuard guard(attn.device());
            Tensor joined = at::empty({rows, c.blocks() * width}, attn.options());
            HstuOutputArgs a{};
            fill_output(a, attn, u, norm_weight, norm_bias, c);
            check_linear(hstu_output_norm_mul(&a, joined.data_ptr(), joined.size(1), stream_of(attn)));
            got[5] = weight_grad(joined, dout, Tensor());
        }
        return got;
    }
};

OptTensor compute_output(const Tensor& attn, const Tensor& u, const Tensor& x, const Tensor& norm_weight, const Tensor& norm_bias, double eps,
                         const Tensor& weight, int64_t heads, int64_t linear_dim, bool concat_u, bool concat_x, int64_t activation,
                         bool group_norm, int64_t path, double dropout, uint64_t seed, uint64_t offset) {
    const OutputCall c{heads, linear_dim, activation, path, concat_u, concat_x, group_norm, eps, dropout, seed, offset};
    if (!matrix_rows(attn) || !matrix_rows(u) || !matrix_rows(x) || dense_dtype(x) < 0) return {};
    if (attn.scalar_type() != x.scalar_type() || u.scalar_type() != x.scalar_type()) return {};
    const int64_t rows = attn.size(0), width = attn.size(1), norm = group_norm ? heads : width;
    if (u.size(0) != rows || u.size(1) != width || x.size(0) != rows || width != heads * linear_dim || heads <= 0 || activation < 0) return {};
    if (norm_weight.dim() != 1 || norm_weight.size(0) != norm || norm_bias.dim() != 1 || norm_bias.size(0) != norm) return {};
    if (weight.dim() != 2 || weight.size(0) != c.blocks() * width || weight.size(1) != x.size(1)) return {};
    if (!parameter(norm_weight, x) || !parameter(norm_bias, x) || !parameter(weight, x)) return {};
    const bool grad = wants_grad({&attn, &u, &x, &norm_weight, &norm_bias, &weight});
    if (grad && x.size(1) > kWeightGradColumns) return {};
    try {
        return grad ? OutputFunction::apply(attn, u, x, norm_weight, norm_bias, weight, c)
                   : output_result(attn, u, x, norm_weight, norm_bias, weight, c);
    } catch (const Declined&) {
        return {};
    }
}

}  // namespace

PYBIND11_MODULE(TORCH_EXTENSION_NAME, m) {
    m.doc() = "native front of the HSTU operators; every function returns None for a call it leaves to the Python operator";
    const auto nogil = py::call_guard<py::gil_scoped_release>();
    m.def("hstu_mha", &hstu_mha, nogil);
    m.def("delta_hstu_mha", &delta_hstu_mha, nogil);
    m.def("concat_2d_jagged", &concat_2d_jagged, nogil);
    m.def("split_2d_jagged", &split_2d_jagged, nogil);
    m.def("write_kv_tail", &write_kv_tail, nogil);
    m.def("compute_uqvk", &compute_uqvk, nogil);
    m.def("preprocess_and_attention", &preprocess_and_attention, nogil);
    m.def("compute_output", &compute_output, nogil);
}
