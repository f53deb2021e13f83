// Native front of the operators: a Python module (`hstu_native`) that takes torch tensors, checks them, allocates the
// result and the scratch memory and calls the C ABI (hstu_hip.h, hstu_linear.h) -- the work that ops/*.py does through
// ctypes for every argument it has to look at, in a few microseconds instead of ten to thirty.
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

bool attention_operands(const Tensor& q, const Tensor& k, const Tensor& v, const Tensor& offsets, const OptTensor& targets) {
    if (q.dim() != 3 || k.dim() != 3 || v.dim() != 3 || !q.is_cuda() || !k.is_cuda() || !v.is_cuda() || !index_tensor(offsets)) return false;
    if (attention_dtype(q.scalar_type()) < 0 || k.scalar_type() != q.scalar_type() || v.scalar_type() != q.scalar_type()) return false;
    if (k.size(1) != q.size(1) || k.size(2) != q.size(2) || v.size(0) != k.size(0) || v.size(1) != q.size(1)) return false;
    if (offsets.dim() != 1 || offsets.numel() < 2 || q.numel() == 0 || k.numel() == 0 || v.numel() == 0) return false;
    if (targets && (!index_tensor(*targets) || targets->numel() != offsets.numel() - 1)) return false;
    return kernel_layout(q) && kernel_layout(k) && kernel_layout(v) && !contract_checks();
}

at::ScalarType result_type(const Tensor& q) { return q.scalar_type() == at::kFloat8_e4m3fn ? at::kBFloat16 : q.scalar_type(); }

OptTensor hstu_mha(int64_t max_seq_len, double alpha, const Tensor& q, const Tensor& k, const Tensor& v, const Tensor& offsets,
                   const OptTensor& targets, int64_t w, int64_t c, int64_t f, bool sort, double q_scale, double k_scale, double v_scale,
                   int64_t tile_config, int64_t kv_splits) {
    if (max_seq_len <= 0 || !attention_operands(q, k, v, offsets, targets) || q.size(0) != k.size(0) || wants_grad({&q, &k, &v})) return {};
    RECORD_USER_SCOPE("hstu_mha");
    Tensor out = at::empty({v.size(0), v.size(1), v.size(2)}, v.options().dtype(result_type(q)));
    const AttentionCall call{max_seq_len, 0, w, c, f, alpha, q_scale, k_scale, v_scale, tile_config, kv_splits, sort};
    if (attention_forward(q, k, v, out, offsets, targets, call) != HSTU_OK) return {};
    return out;
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

Tensor aligned_scratch(size_t bytes, const Tensor& like, void** ptr) {
    Tensor t = at::empty({(int64_t)bytes + 256}, like.options().dtype(at::kByte));
    *ptr = reinterpret_cast<void*>((reinterpret_cast<uintptr_t>(t.data_ptr()) + 255) & ~(uintptr_t)255);
    return t;
}

// u [L, hidden * H], q, k [L, H, attn], v [L, H, hidden] as views of the buffer u | v | q | k
std::tuple<Tensor, Tensor, Tensor, Tensor> uqvk_views(const Tensor& buf, int64_t heads, int64_t attn, int64_t hidden) {
    const int64_t rows = buf.size(0), pitch = buf.size(1), nu = hidden * heads, na = attn * heads;
    const at::AutoDispatchBelowADInplaceOrView below;
    return {buf.as_strided({rows, nu}, {pitch, 1}, 0), buf.as_strided({rows, heads, attn}, {pitch, attn, 1}, 2 * nu),
            buf.as_strided({rows, heads, attn}, {pitch, attn, 1}, 2 * nu + na), buf.as_strided({rows, heads, hidden}, {pitch, hidden, 1}, nu)};
}

std::optional<std::tuple<Tensor, Tensor, Tensor, Tensor>> compute_uqvk(const Tensor& x, const Tensor& norm_weight, const Tensor& norm_bias,
                                                                       double eps, int64_t heads, int64_t attn, int64_t hidden,
                                                                       const Tensor& weight, const Tensor& bias, int64_t path) {
    const int64_t n_out = (2 * hidden + 2 * attn) * heads;
    if (!matrix_rows(x) || dense_dtype(x) < 0 || heads <= 0 || attn <= 0 || hidden <= 0) return {};
    if (weight.dim() != 2 || weight.size(0) != x.size(1) || weight.size(1) != n_out || bias.dim() != 1 || bias.size(0) != n_out) return {};
    if (!parameter(norm_weight, x) || !parameter(norm_bias, x) || !parameter(weight, x) || !parameter(bias, x)) return {};
    if (wants_grad({&x, &norm_weight, &norm_bias, &weight, &bias})) return {};
    Tensor buf = at::empty({x.size(0), n_out}, x.options());
    HstuUqvkArgs a{};
    a.x = x.const_data_ptr(), a.x_row_stride = x.stride(0);
    a.norm_weight = norm_weight.const_data_ptr(), a.norm_bias = norm_bias.const_data_ptr(), a.norm_eps = (float)eps;
    a.uvqk_weight = weight.const_data_ptr(), a.uvqk_bias = bias.const_data_ptr(), a.uvqk = buf.data_ptr();
    a.rows = x.size(0), a.d_model = (int32_t)x.size(1), a.heads = (int32_t)heads, a.attn_dim = (int32_t)attn, a.hidden_dim = (int32_t)hidden;
    a.dtype = dense_dtype(x), a.path = (int32_t)path;
    const size_t need = hstu_uqvk_workspace_bytes(&a);
    Tensor scratch;
    if (need > 0) scratch = aligned_scratch(need, x, &a.workspace), a.workspace_bytes = (int64_t)need;
    const c10::DeviceGuard guard(x.device());
    if (hstu_uqvk_forward(&a, stream_of(x)) != 0) return {};
    return uqvk_views(buf, heads, attn, hidden);
}

// The output step without dropout.
OptTensor compute_output(const Tensor& attn, const Tensor& u, const Tensor& x, const Tensor& norm_weight, const Tensor& norm_bias, double eps,
                         const Tensor& weight, int64_t heads, int64_t linear_dim, bool concat_u, bool concat_x, int64_t activation,
                         bool group_norm, int64_t path) {
    if (!matrix_rows(attn) || !matrix_rows(u) || !matrix_rows(x) || dense_dtype(x) < 0) return {};
    if (attn.scalar_type() != x.scalar_type() || u.scalar_type() != x.scalar_type()) return {};
    const int64_t rows = attn.size(0), width = attn.size(1);
    if (u.size(0) != rows || u.size(1) != width || x.size(0) != rows || width != heads * linear_dim || heads <= 0 || activation < 0) return {};
    const int64_t norm = group_norm ? heads : width, blocks = group_norm ? (concat_u && concat_x ? 3 : 1) : 1 + concat_u + concat_x;
    if (norm_weight.dim() != 1 || norm_weight.size(0) != norm || norm_bias.dim() != 1 || norm_bias.size(0) != norm) return {};
    if (weight.dim() != 2 || weight.size(0) != blocks * width || weight.size(1) != x.size(1)) return {};
    if (!parameter(norm_weight, x) || !parameter(norm_bias, x) || !parameter(weight, x)) return {};
    if (wants_grad({&attn, &u, &x, &norm_weight, &norm_bias, &weight})) return {};
    Tensor out = at::empty({rows, x.size(1)}, x.options());
    HstuOutputArgs a{};
    a.attn = attn.const_data_ptr(), a.attn_row_stride = attn.stride(0), a.u = u.const_data_ptr(), a.u_row_stride = u.stride(0);
    a.x = x.const_data_ptr(), a.x_row_stride = x.stride(0);
    a.norm_weight = norm_weight.const_data_ptr(), a.norm_bias = norm_bias.const_data_ptr(), a.norm_eps = (float)eps;
    a.output_weight = weight.const_data_ptr(), a.out = out.data_ptr();
    a.rows = rows, a.d_out = (int32_t)x.size(1), a.heads = (int32_t)heads, a.linear_dim = (int32_t)linear_dim;
    a.concat_u = concat_u, a.concat_x = concat_x, a.group_norm = group_norm, a.mul_u_activation = (int32_t)activation;
    a.dtype = dense_dtype(x), a.path = (int32_t)path;
    const size_t need = hstu_output_workspace_bytes(&a);
    Tensor scratch;
    if (need > 0) scratch = aligned_scratch(need, x, &a.workspace), a.workspace_bytes = (int64_t)need;
    const c10::DeviceGuard guard(x.device());
    if (hstu_output_forward(&a, stream_of(x)) != 0) return {};
    return out;
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
    m.def("compute_output", &compute_output, nogil);
}
