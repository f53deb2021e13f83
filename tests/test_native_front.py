"""The operators' native front: it serves the usual call with the same bits as the Python path, and leaves (returns None
for) every call that path has to copy for or refuse; gradients of the dense steps against the recomputation in Python."""

import pytest
import torch

from util import make_case

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def front():
    from generative_recommenders_amd.ops import native

    return native.front


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32, torch.float8_e4m3fn])
@pytest.mark.parametrize("delta", [0, 5])
def test_attention_through_the_front_and_through_python(pkg, dev, front, dtype, delta):
    from generative_recommenders_amd.ops import hstu_attention as A

    print(f"[case] native front attention {dtype} delta={delta}", flush=True)
    q, k, v, offs, t = make_case(1, [70, 9, 5, 130], 2, 64, targets=[5, 3, 2, 9], delta_size=delta, dtype=torch.float32)
    q, k, v = (x.to(dtype).to(dev) for x in (q, k, v))
    offs, t = offs.to(dev), t.to(dev)
    if delta:
        args = (150, 0.1, q, k, v, offs, t, 20, 3, 0.5, 2.0, 1.5, 0, 0)
        got, want = front.delta_hstu_mha(*args), A._delta_hstu_mha(*args)
        wide = front.delta_hstu_mha(150, 0.1, q.transpose(1, 2).contiguous().transpose(1, 2), *args[3:])
        wrong = front.delta_hstu_mha(150, 0.1, q[:-1], *args[3:])
    else:
        args = (150, 0.1, q, k, v, offs, t, 20, 3, 0, True, 0.5, 2.0, 1.5, 0, 0, None)
        got = front.hstu_mha(*args)
        want = A._hstu_mha(150, 0.1, q, k, v, offs, True, 0.0, t, None, 20, 3, 0, True, 0.5, 2.0, 1.5, 0, 0, None)
        wide = front.hstu_mha(150, 0.1, q.transpose(1, 2).contiguous().transpose(1, 2), *args[3:])
        wrong = front.hstu_mha(150, 0.1, q[:-1], *args[3:])
    torch.cuda.synchronize()
    assert got is not None and torch.equal(got, want) and got.dtype == want.dtype
    assert wide is None and wrong is None  # not dense in the innermost dimension; a row short


def test_dense_steps_and_row_copies_leave_what_they_cannot_serve(pkg, dev, front):
    x, nw, w, b = (torch.randn(*s, device=dev).bfloat16() for s in ((20, 128), (128,), (128, 256), (256,)))
    args = (x, nw, nw, 1e-6, 1, 64, 64, w, b, 0)
    print("[case] native front, calls it leaves", flush=True)
    assert front.compute_uqvk(*args) is not None
    assert front.compute_uqvk(x.float(), *args[1:]) is None and front.compute_uqvk(x[:, 1:], *args[1:]) is None
    assert all(t.requires_grad for t in front.compute_uqvk(x.clone().requires_grad_(), *args[1:]))
    attn, wo, ow = x[:, :64], torch.randn(192, 128, device=dev).bfloat16(), nw[:64]
    out = (attn, attn, x, ow, ow, 1e-6, wo, 1, 64, True, True, 0, False, 0, 0.0, 0, 0)
    assert front.compute_output(*out) is not None and front.compute_output(*out[:11], -1, *out[12:]) is None
    offs = torch.tensor([0, 12, 20], device=dev)
    assert front.concat_2d_jagged(x, x, 12, 12, offs, offs) is not None and front.concat_2d_jagged(x, x, None, 12, offs, offs) is None
    assert front.split_2d_jagged(torch.cat([x, x]), 20, 20, 12, 12, offs, offs) is not None and front.split_2d_jagged(x, 12, 9, 12, 8, offs, offs) is None
    assert front.write_kv_tail(x, offs, x[:4].clone()) and not front.write_kv_tail(x, offs, x[:3].clone())
    torch.cuda.synchronize()


def _grads(fn, tensors, d_out):
    leaves = [t.detach().clone().requires_grad_() for t in tensors]
    return torch.autograd.grad(fn(*leaves), leaves, d_out)


def _close(got, want, what):
    """Both are sums of the same terms with the same roundings of the operands, accumulated in fp32 in another order and rounded
    once: a matrix of results in bf16 differs by its last bit here and there (2^-9 relative, half of it on average), a vector
    that is summed over the rows by the cancellation on top, so four times that."""
    assert got.shape == want.shape and torch.isfinite(got).all(), what
    rel = float((got.float() - want.float()).norm() / want.float().norm())
    assert rel <= (4e-3 if got.dim() > 1 else 1.6e-2), f"{what}: {rel:.2e}"


@pytest.mark.parametrize("rows,heads,dim,cu,cx,act,group,drop", [
    (1, 1, 8, True, True, "none", False, 0.0), (5, 2, 64, True, True, "silu", False, 0.3), (300, 3, 168, False, True, "sigmoid", False, 0.0),
    (4100, 4, 128, True, False, "none", False, 0.2), (77, 8, 128, True, True, "none", True, 0.1), (9, 8, 512, True, True, "none", False, 0.0),
    (513, 2, 8, False, False, "none", True, 0.0), (260, 1, 512, True, True, "none", True, 0.5),
])
def test_output_step_gradients_against_the_recomputation(dev, rows, heads, dim, cu, cx, act, group, drop):
    """The norm-multiply backward kernel and the products around it, at widths of one lane to the widest row, one row to more
    rows than waves, against the package's own restatement with torch operators (same operands, same mask)."""
    from generative_recommenders_amd.ops import hstu_compute as hc

    print(f"[case] output gradients {rows} {heads} {dim} {cu} {cx} {act} group={group} drop={drop}", flush=True)
    g = torch.Generator(device=dev).manual_seed(rows)
    width, d = heads * dim, 64
    blocks = hc._blocks(cu, cx, group)
    norm = heads if group else width
    shapes = ((rows, width), (rows, width), (rows, d), (norm,), (norm,), (blocks * width, d))
    ins = [torch.randn(s, generator=g, device=dev).bfloat16() for s in shapes]
    d_out = torch.randn((rows, d), generator=g, device=dev).bfloat16()
    state = hc._dropout_state(drop, True, 0, dev, (3, 8))
    mask = hc._keep_scaled(state, rows, blocks * width, dev)
    got = _grads(lambda a, u, x, nw, nb, w: hc.hstu_compute_output(a, u, x, nw, nb, 1e-6, w, heads, dim, drop, True, cu, cx, act, group, True, seed=(3, 8)),
                 ins, d_out)
    want = _grads(lambda a, u, x, nw, nb, w: torch.addmm(x, hc._norm_mul_math(a, u, nw, nb, 1e-6, False, cu, cx, act, group, heads, dim, keep_scaled=mask), w),
                  ins, d_out)
    torch.cuda.synchronize()
    for name, a, b in zip(("attn", "u", "x", "norm_weight", "norm_bias", "weight"), got, want):
        _close(a, b, f"d/d{name}")


@pytest.mark.parametrize("rows,heads,dim,cx,act,group,drop", [
    (5, 2, 64, True, "none", False, 0.0), (300, 4, 128, False, "sigmoid", False, 0.2), (77, 8, 128, True, "none", True, 0.0), (260, 1, 512, True, "none", True, 0.3),
])
def test_norm_multiply_backward_with_silu_on_the_copied_u(dev, rows, heads, dim, cx, act, group, drop):
    """``silu_u``, which only the C entry passes on to its kernel (the Python operator that has the flag differentiates the restatement):
    d attn, d u, the norm's gradients and the recomputed operand."""
    import ctypes

    from generative_recommenders_amd.ops import hstu_compute as hc

    print(f"[case] norm-multiply backward, silu_u {rows} {heads} {dim} {cx} {act} group={group} drop={drop}", flush=True)
    g = torch.Generator(device=dev).manual_seed(rows)
    width, norm = heads * dim, heads if group else heads * dim
    ins = [torch.randn(s, generator=g, device=dev).bfloat16() for s in ((rows, width), (rows, width), (norm,), (norm,))]
    a, keep, blocks = hc._output_args(*ins, 1e-6, heads, dim, True, cx, act, group, True)
    d_joined = torch.randn((rows, blocks * width), generator=g, device=dev).bfloat16()
    state = hc._dropout_state(drop, True, 0, dev, (3, 8))
    hc._set_dropout(a, state)
    mask = hc._keep_scaled(state, rows, blocks * width, dev)

    got = [torch.full_like(t, float("nan")) for t in ins]
    joined = torch.full_like(d_joined, float("nan"))
    L, P, Q = hc.lib(), ctypes.c_void_p, ctypes.c_int64
    L.hstu_output_norm_mul_bwd_workspace_bytes.restype = ctypes.c_size_t
    need = L.hstu_output_norm_mul_bwd_workspace_bytes(ctypes.byref(a))
    ws = torch.full((need // 4,), float("nan"), device=dev)

    class Grads(ctypes.Structure):  # HstuNormMulGrads
        _fields_ = [(f"f{i}", P if i not in (1, 3, 5, 7, 11) else Q) for i in range(12)]

    grads = Grads(d_joined.data_ptr(), d_joined.stride(0), joined.data_ptr(), joined.stride(0), got[0].data_ptr(), width, got[1].data_ptr(), width,
                  got[2].data_ptr(), got[3].data_ptr(), ws.data_ptr(), need)
    rc = L.hstu_output_norm_mul_bwd(ctypes.byref(a), ctypes.byref(grads), P(torch.cuda.current_stream(dev).cuda_stream))
    torch.cuda.synchronize()
    assert rc == 0, L.hstu_linear_last_error()

    def restated(attn, u, nw, nb):
        return hc._norm_mul_math(attn, u, nw, nb, 1e-6, True, True, cx, act, group, heads, dim, keep_scaled=mask)

    _close(joined, restated(*ins), "joined")
    for name, x, y in zip(("attn", "u", "norm_weight", "norm_bias"), got, _grads(restated, ins, d_joined)):
        _close(x, y, f"d/d{name}")


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("rows,d,heads,attn,hidden", [(1, 64, 1, 16, 16), (4101, 128, 2, 32, 64), (63, 1024, 1, 64, 64), (20, 4096, 1, 8, 8), (300, 520, 3, 16, 8), (3, 64, 1, 32768, 16)])
def test_producer_gradients_against_the_recomputation(dev, dtype, rows, d, heads, attn, hidden):
    """Layer-norm and SiLU backward kernels, at widths up to the widest row, with rows past the waves of the grid, and at more columns
    than the weight gradient takes."""
    from generative_recommenders_amd.ops import hstu_compute as hc

    print(f"[case] producer gradients {rows} {d} {heads} {attn} {hidden} {dtype}", flush=True)
    g = torch.Generator(device=dev).manual_seed(rows)
    n = (2 * attn + 2 * hidden) * heads
    ins = [torch.randn(s, generator=g, device=dev).to(dtype) for s in ((rows, d), (d,), (d,), (d, n), (n,))]
    ins[3] = (ins[3] / d**0.5).contiguous()
    d_out = torch.randn((rows, n), generator=g, device=dev).to(dtype)

    def through_kernels(x, nw, nb, w, b):
        u, q, k, v = hc.hstu_compute_uqvk(x, nw, nb, 1e-6, heads, attn, hidden, w, b)
        return torch.cat([u, v.flatten(1), q.flatten(1), k.flatten(1)], dim=1)

    got = _grads(through_kernels, ins, d_out)
    want = _grads(lambda x, nw, nb, w, b: hc._uqvk_math(x, nw, nb, 1e-6, hidden * heads, w, b), ins, d_out)
    torch.cuda.synchronize()
    for name, a, b in zip(("x", "norm_weight", "norm_bias", "weight", "bias"), got, want):
        _close(a, b, f"d/d{name}")


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("rows,m,n,sliced", [(1, 8, 8, False), (33, 264, 248, False), (64, 256, 512, True), (1000, 72, 776, False), (40000, 520, 256, True)])
def test_weight_gradient_kernel(dev, dtype, rows, m, n, sliced):
    """out = a^T b and the column sums of b, against fp64: one row, part tiles in both directions, rows that fill no tile, more
    splits than one, operands that are column slices.  The bound: rounding the result to nearest moves a value by at
    most half a unit of its last place, 2^-8 of it in bf16 (8 bits of significand) and 2^-11 in fp16 (11 bits), so the 2-norm of
    the result by no more than that; a tenth of it more for the fp32 sums of at most 40000 products (each rounding 2^-24, random
    in sign)."""
    import ctypes

    from generative_recommenders_amd.ops import hstu_compute as hc

    print(f"[case] weight gradient {rows} {m} {n} {sliced} {dtype}", flush=True)
    g = torch.Generator(device=dev).manual_seed(rows + m)
    pad = 40 if sliced else 0
    a = torch.randn((rows, m + pad), generator=g, device=dev).to(dtype)[:, pad:]
    b = torch.randn((rows, n + pad), generator=g, device=dev).to(dtype)[:, :n]
    out, sums = torch.full((m, n), float("nan"), dtype=dtype, device=dev), torch.full((n,), float("nan"), dtype=dtype, device=dev)
    L = hc.lib()
    L.hstu_linear_weight_grad_workspace_bytes.restype = ctypes.c_size_t
    L.hstu_linear_weight_grad_workspace_bytes.argtypes = [ctypes.c_int32, ctypes.c_int32] + [ctypes.c_int64] * 3
    need = L.hstu_linear_weight_grad_workspace_bytes(m, n, rows, a.stride(0), b.stride(0))
    ws = torch.full((need // 4,), float("nan"), device=dev)
    P, I, Q = ctypes.c_void_p, ctypes.c_int32, ctypes.c_int64
    rc = L.hstu_linear_weight_grad(P(a.data_ptr()), Q(a.stride(0)), I(m), P(b.data_ptr()), Q(b.stride(0)), I(n), Q(rows), I(0 if dtype == torch.bfloat16 else 1),
                                   P(out.data_ptr()), P(sums.data_ptr()), P(ws.data_ptr()), Q(need), P(torch.cuda.current_stream(dev).cuda_stream))
    torch.cuda.synchronize()
    assert rc == 0, hc.lib().hstu_linear_last_error()
    unit = 2.0**-8 if dtype == torch.bfloat16 else 2.0**-11
    for got, want in ((out, a.double().t() @ b.double()), (sums, b.double().sum(0))):
        assert torch.isfinite(got).all()
        assert float((got.double() - want).norm() / want.norm()) <= 1.1 * unit


def test_gradients_under_create_graph_are_the_plain_ones_without_a_graph(pkg, dev):
    """The backward kernels are not differentiable: with ``create_graph`` the gradients are those of the plain call and carry no
    graph, not part of one."""
    print("[case] gradients with create_graph", flush=True)
    g = torch.Generator(device=dev).manual_seed(5)
    H, D, d, L = 2, 64, 128, 90
    shapes = ((L, d), (d,), (d,), (d, 4 * H * D), (4 * H * D,), (H * D,), (H * D,), (3 * H * D, d))
    ins = [(0.1 * torch.randn(s, generator=g, device=dev)).bfloat16().requires_grad_() for s in shapes]
    offsets = torch.tensor([0, 30, 90], device=dev)
    d_out = torch.randn((L, d), generator=g, device=dev).bfloat16().requires_grad_()

    def layer(x, nw, nb, w, b, onw, onb, ow):
        u, attn, _, _ = pkg.hstu_preprocess_and_attention(x, nw, nb, 1e-6, H, D, D, w, b, 60, offsets, D**-0.5, True, None, 0, 0, True, True, False)
        return pkg.hstu_compute_output(attn, u, x, onw, onb, 1e-6, ow, H, D, 0.0, True, True, True, "none", False, True)

    plain = torch.autograd.grad(layer(*ins), ins, d_out.detach())
    graph = torch.autograd.grad(layer(*ins), ins, d_out, create_graph=True)
    torch.cuda.synchronize()
    for a, b in zip(plain, graph):
        assert torch.equal(a, b) and not b.requires_grad
