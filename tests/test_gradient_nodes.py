"""The autograd nodes of the operators' native front: what they hand back to autograd and what they take from it."""

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def hc():
    from generative_recommenders_amd.ops import hstu_compute

    return hstu_compute


H, D, D_MODEL = 2, 64, 128
N_OUT = 4 * H * D


def _rand(dev, seed, shapes, dtype=torch.bfloat16):
    g = torch.Generator(device=dev).manual_seed(seed)
    return [torch.randn(s, generator=g, device=dev).to(dtype) for s in shapes]


def _output_inputs(dev, rows, dtype=torch.bfloat16):
    """attn, u, x, norm weight, norm bias, weight"""
    return _rand(dev, rows, ((rows, H * D), (rows, H * D), (rows, D_MODEL), (H * D,), (H * D,), (3 * H * D, D_MODEL)), dtype)


def _output(hc, attn, u, x, nw, nb, w):
    return hc.hstu_compute_output(attn, u, x, nw, nb, 1e-6, w, H, D, 0.0, True, True, True, "none", False, True)


def _producer_inputs(dev, rows, dtype=torch.bfloat16):
    """x, norm weight, norm bias, weight, bias"""
    ins = _rand(dev, rows + 1, ((rows, D_MODEL), (D_MODEL,), (D_MODEL,), (D_MODEL, N_OUT), (N_OUT,)), dtype)
    ins[3] = ins[3] / D_MODEL**0.5
    return ins


def _producer(hc, x, nw, nb, w, b):
    return hc.hstu_compute_uqvk(x, nw, nb, 1e-6, H, D, D, w, b)


def _first_half(hc, dev, x, nw, nb, w, b):
    """(u, attention output, k, v) of one sequence"""
    offsets = torch.tensor([0, x.shape[0]], device=dev)
    return hc.hstu_preprocess_and_attention(x, nw, nb, 1e-6, H, D, D, w, b, x.shape[0], offsets, D**-0.5, True, None, 0, 0, True, True, False)


def _leaves(tensors):
    return [t.detach().clone().requires_grad_() for t in tensors]


def test_the_residuals_gradient_is_not_the_callers_tensor(dev, hc):
    """Autograd adds later gradients to a leaf's first one in place: it must not share the memory of the gradient that came in."""
    print("[case] residual gradient of a leaf", flush=True)
    attn, u, x, nw, nb, w = _output_inputs(dev, 40)
    x.requires_grad_()
    d_out = torch.ones_like(x)
    for _ in range(3):
        _output(hc, attn, u, x, nw, nb, w).backward(d_out)
    torch.cuda.synchronize()
    assert (d_out == 1).all() and (x.grad == 3).all()


@pytest.mark.parametrize("dtype,other", [(torch.bfloat16, torch.float16), (torch.float16, torch.bfloat16)])
def test_backward_inside_autocast_of_the_other_type(dev, hc, dtype, other):
    """The nodes' products are of the inputs' type whatever autocast would make of them: the kernels read that type."""
    print(f"[case] backward of {dtype} under autocast to {other}", flush=True)
    ins = _leaves([0.1 * t for t in _producer_inputs(dev, 50, dtype) + _output_inputs(dev, 50, dtype)[3:]])

    def layer():
        u, attn, _, _ = _first_half(hc, dev, *ins[:5])
        return _output(hc, attn, u, ins[0], *ins[5:])

    (d_out,) = _rand(dev, 9, ((50, D_MODEL),), dtype)
    want = torch.autograd.grad(layer(), ins, d_out) + torch.autograd.grad(_producer(hc, *ins[:5])[0], ins[:5], d_out)
    first, second = layer(), _producer(hc, *ins[:5])[0]
    with torch.autocast("cuda", dtype=other):
        got = torch.autograd.grad(first, ins, d_out) + torch.autograd.grad(second, ins[:5], d_out)
    torch.cuda.synchronize()
    for a, b in zip(got, want):
        assert a.dtype == b.dtype and torch.equal(a, b)


def _odd_offset(t):
    """The same values, contiguous, two bytes past a 16-byte boundary."""
    return torch.cat([t.new_zeros(1), t.flatten()])[1:].view(t.shape)


def _one_row_of_a_wider_buffer(t):
    """The same values; strides that count as contiguous although the row stride is odd, and for the last form below the row's width."""
    return t.as_strided(t.shape, (t.shape[1] + 5, 1))


def _one_row_overlapping(t):
    return t.as_strided(t.shape, (1, 1))


@pytest.mark.parametrize("rows,layout", [(40, _odd_offset), (1, _odd_offset), (1, _one_row_of_a_wider_buffer), (1, _one_row_overlapping)])
def test_gradients_that_are_not_as_the_kernels_read_rows(dev, hc, rows, layout):
    """Slices of a flat gradient and single rows of wider ones, for the output step and for u: the result of a dense copy."""
    print(f"[case] gradient layout {rows} {layout.__name__}", flush=True)
    out_ins, ins = _leaves(_output_inputs(dev, rows)), _leaves(_producer_inputs(dev, rows))
    d_out, du = _rand(dev, 4, ((rows, D_MODEL), (rows, H * D)))
    calls = (
        (lambda: _output(hc, *out_ins), out_ins, d_out),
        (lambda: _producer(hc, *ins)[0], ins, du),
        (lambda: _first_half(hc, dev, *ins)[0], ins, du),
        (lambda: _first_half(hc, dev, *ins)[1], ins, du),
    )
    for fn, tensors, d in calls:
        want = torch.autograd.grad(fn(), tensors, d)
        got = torch.autograd.grad(fn(), tensors, layout(d))
        torch.cuda.synchronize()
        for a, b in zip(got, want):
            assert torch.equal(a, b)


def test_saved_tensors_that_come_back_in_another_layout(dev, hc):
    """What saved-tensor hooks give back (from a flat store, say) has the values, not the alignment, of what was saved."""
    print("[case] saved tensors at odd offsets", flush=True)
    out_ins, ins = _leaves(_output_inputs(dev, 40)), _leaves(_producer_inputs(dev, 40))
    d_out, du = _rand(dev, 4, ((40, D_MODEL), (40, H * D)))
    calls = (
        (lambda: _output(hc, *out_ins), out_ins, d_out),
        (lambda: _producer(hc, *ins)[0], ins, du),
        (lambda: _first_half(hc, dev, *ins)[1], ins, du),
    )
    for fn, tensors, d in calls:
        want = torch.autograd.grad(fn(), tensors, d)
        with torch.autograd.graph.saved_tensors_hooks(lambda t: t.detach(), lambda t: _odd_offset(t) if t.is_floating_point() else t):
            out = fn()
        got = torch.autograd.grad(out, tensors, d)
        torch.cuda.synchronize()
        for a, b in zip(got, want):
            assert torch.equal(a, b)


@pytest.mark.parametrize("wanted,d_model,heads,dim,limit_mb", [((0,), 128, 2, 64, 16), ((3,), 2048, 1, 16, 96), ((1, 2), 128, 2, 64, 16)])
def test_gradients_that_nobody_asked_for_are_not_formed(dev, hc, wanted, d_model, heads, dim, limit_mb):
    """Seen by the memory that the backward takes at its peak, 4096 rows.  d_model 128, 512 columns: 10 MB without the weight's
    gradient, whose partial sums take 32 MB.  d_model 2048, 64 columns, the weight alone: LN(x) and the partial sums, 16 + 64 MB; the
    layer norm's backward would add 16 MB for its operand and 32 for its results."""
    print(f"[case] gradients wanted {wanted} of d_model {d_model}", flush=True)
    n = 4 * heads * dim
    ins = _rand(dev, 3, ((4096, d_model), (d_model,), (d_model,), (d_model, n), (n,)))
    (du,) = _rand(dev, 4, ((4096, heads * dim),))
    everything = _leaves(ins)
    want = torch.autograd.grad(hc.hstu_compute_uqvk(*everything[:3], 1e-6, heads, dim, dim, *everything[3:])[0], everything, du)
    want = [want[i].clone() for i in wanted]
    some = [t.detach().clone().requires_grad_(i in wanted) for i, t in enumerate(ins)]
    u = hc.hstu_compute_uqvk(*some[:3], 1e-6, heads, dim, dim, *some[3:])[0]
    torch.cuda.synchronize()
    torch.cuda.reset_peak_memory_stats(dev)
    before = torch.cuda.memory_allocated(dev)
    got = torch.autograd.grad(u, [some[i] for i in wanted], du)
    torch.cuda.synchronize()
    peak = torch.cuda.max_memory_allocated(dev) - before
    for a, b in zip(got, want):
        assert torch.equal(a, b)
    assert peak <= limit_mb << 20, f"{peak / 2**20:.0f} MB"


@pytest.mark.parametrize("wanted,drop", [((2,), 0.0), ((5,), 0.0), ((5,), 0.3), ((0, 1), 0.0)])
def test_output_step_with_part_of_its_gradients_wanted(dev, hc, wanted, drop):
    """The weight's gradient alone comes from the forward's kernel (the joined operand) without the product that the others need."""
    print(f"[case] output gradients wanted {wanted} dropout {drop}", flush=True)
    ins = _output_inputs(dev, 300)
    (d_out,) = _rand(dev, 4, ((300, D_MODEL),))

    def step(t):
        return hc.hstu_compute_output(*t[:5], 1e-6, t[5], H, D, drop, True, True, True, "silu", False, True, seed=(3, 8))

    everything = _leaves(ins)
    want = torch.autograd.grad(step(everything), everything, d_out)
    some = [t.detach().clone().requires_grad_(i in wanted) for i, t in enumerate(ins)]
    got = torch.autograd.grad(step(some), [some[i] for i in wanted], d_out)
    torch.cuda.synchronize()
    for i, a in zip(wanted, got):
        assert torch.equal(a, want[i])


def test_producer_does_not_run_for_an_attention_that_is_left_to_python(dev, hc):
    """Head dims without a kernel, offsets that need a copy, too few target counts, a negative window: known before the producer's buffer is
    allocated."""
    from generative_recommenders_amd.ops import native

    print("[case] attention declined ahead of the producer", flush=True)
    rows = 512

    def declined(heads, dim, offsets, targets=None, window=0):
        n = 4 * heads * dim
        x, nw, nb, w, b = _rand(dev, 2, ((rows, D_MODEL), (D_MODEL,), (D_MODEL,), (D_MODEL, n), (n,)))
        x.requires_grad_()
        torch.cuda.reset_peak_memory_stats(dev)
        before = torch.cuda.memory_allocated(dev)
        got = native.front.preprocess_and_attention(x, nw, nb, 1e-6, heads, dim, dim, w, b, rows, offsets, 0.1, targets, window, 0, False)
        torch.cuda.synchronize()
        return got is None and torch.cuda.max_memory_allocated(dev) == before

    offsets = torch.tensor([0, rows], device=dev)
    assert declined(2, 24, offsets)
    assert declined(2, 64, torch.tensor([0, 1, rows, 1], device=dev)[::2])
    assert declined(2, 64, offsets, targets=offsets)
    assert declined(2, 64, offsets, window=-1)
    assert not declined(2, 64, offsets)


def test_a_workspace_that_is_none_is_refused_as_before(pkg, dev):
    print("[case] dS workspace of another type", flush=True)
    q, k, v = _leaves(_rand(dev, 1, ((20, 2, 64),) * 3))
    offsets = torch.tensor([0, 20], device=dev)
    for bad in (torch.empty(1 << 20, dtype=torch.int8, device=dev), torch.empty((1 << 10, 1 << 10), dtype=torch.uint8, device=dev).t(),
                torch.empty(1 << 20, dtype=torch.uint8)):
        out = pkg.hstu_mha(20, 0.1, q, k, v, offsets, bwd_workspace=bad)
        with pytest.raises(AssertionError, match="workspace must be"):
            torch.autograd.grad(out, [q, k, v], torch.ones_like(out))


def test_a_refused_dropout_leaves_the_generator_where_it_was(dev, hc):
    print("[case] refused calls and the dropout generator", flush=True)
    attn, u, x, nw, nb, w = _output_inputs(dev, 8)
    gen = torch.cuda.default_generators[0]
    gen.set_offset(8)
    for wrong in (dict(act="tanh"), dict(x=x[:-1]), dict(nw=nw.half()), dict(attn=attn.cpu())):
        a = dict(attn=attn, x=x, nw=nw, act="none")
        a.update(wrong)
        with pytest.raises(AssertionError):
            hc.hstu_compute_output(a["attn"], u, a["x"], a["nw"], nb, 1e-6, w, H, D, 0.1, True, True, True, a["act"], False, True)
        assert gen.get_offset() == 8


@pytest.mark.parametrize("arrive", ["u", "out", "k", "v", "kv", "out k", "out v", "u out k v"])
def test_gradients_that_arrive_through_any_of_the_outputs(dev, hc, arrive):
    """The one node for producer and attention against the two operators one after the other: the same kernels, but with the attention's
    and the callers' gradients of k and v added in bf16 by autograd there, as here."""
    print(f"[case] gradients through {arrive}", flush=True)
    rows = 70
    one, two = _leaves(_producer_inputs(dev, rows)), _leaves(_producer_inputs(dev, rows))
    offsets = torch.tensor([0, rows], device=dev)
    from generative_recommenders_amd.ops import hstu_attention

    u, q, k, v = _producer(hc, *two)
    attn = hstu_attention.hstu_mha(rows, D**-0.5, q, k, v, offsets).view(rows, H * D)
    first, second = _first_half(hc, dev, *one), (u, attn, k, v)
    picked = [i for i, name in enumerate(("u", "out", "k", "v")) if name in arrive.split() or (arrive == "kv" and name in "kv")]
    assert picked
    d = _rand(dev, 5, [first[i].shape for i in picked])
    got = torch.autograd.grad([first[i] for i in picked], one, d)
    want = torch.autograd.grad([second[i] for i in picked], two, d)
    torch.cuda.synchronize()
    for a, b in zip(got, want):
        assert torch.equal(a, b)
