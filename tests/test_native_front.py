"""The operators' native front: it serves the usual call with the same bits as the Python path, and leaves (returns None
for) every call that path has to copy for, refuse or differentiate."""

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
        args = (150, 0.1, q, k, v, offs, t, 20, 3, 0, True, 0.5, 2.0, 1.5, 0, 0)
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
    assert front.compute_uqvk(x.clone().requires_grad_(), *args[1:]) is None  # gradients: the Python operator
    attn, wo, ow = x[:, :64], torch.randn(192, 128, device=dev).bfloat16(), nw[:64]
    out = (attn, attn, x, ow, ow, 1e-6, wo, 1, 64, True, True, 0, False, 0)
    assert front.compute_output(*out) is not None and front.compute_output(*out[:11], -1, False, 0) is None
    offs = torch.tensor([0, 12, 20], device=dev)
    assert front.concat_2d_jagged(x, x, 12, 12, offs, offs) is not None and front.concat_2d_jagged(x, x, None, 12, offs, offs) is None
    assert front.split_2d_jagged(torch.cat([x, x]), 20, 20, 12, 12, offs, offs) is not None and front.split_2d_jagged(x, 12, 9, 12, 8, offs, offs) is None
    assert front.write_kv_tail(x, offs, x[:4].clone()) and not front.write_kv_tail(x, offs, x[:3].clone())
    torch.cuda.synchronize()
