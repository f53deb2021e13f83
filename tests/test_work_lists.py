"""Work lists built with and without the ranking by length in the same kernel: every row block is listed once either way."""

import pytest
import torch

from oracle import hstu_oracle as O
from util import assert_parity, make_case

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("i64", [True, False])
# around the number of sequences that the list's kernel ranks itself, and the fewest that can be ranked
@pytest.mark.parametrize("batch,heads,longest", [(2, 64, 1024), (65, 8, 300), (255, 2, 512), (256, 2, 512), (257, 2, 512)])
def test_ranked_lists(pkg, dev, batch, heads, longest, i64):
    print(f"[case] ranked work lists {batch} x {heads} heads up to {longest}", flush=True)
    gen = torch.Generator().manual_seed(batch)
    lengths = torch.randint(0, longest + 1, (batch,), generator=gen).tolist()
    lengths[0], lengths[-1] = longest, longest  # a tie
    if batch > 4:
        lengths[2] = lengths[3] = 0
    q, k, v, offs, t = make_case(batch, lengths, heads, 64, targets=[min(3, n) for n in lengths])
    if not i64:
        offs, t = offs.int(), t.int()
    args = [longest, 0.125] + [x.to(dev) for x in (q, k, v, offs)]
    ranked = pkg.hstu_mha(*args, num_targets=t.to(dev), sort_by_length=True)
    plain = pkg.hstu_mha(*args, num_targets=t.to(dev))
    torch.cuda.synchronize()
    assert torch.equal(ranked, plain)
    assert_parity(ranked, O.hstu_mha_per_sequence(longest, 0.125, q.float(), k.float(), v.float(), offs.long(), num_targets=t.long()), "ranked lists")


# (batch, heads, longest, columns): a workgroup for every item there could be, with one row block per sequence, up to four (unranked) and more (ranked); on the other
# side of each line the lists, around the number of sequences that their kernel ranks itself and the 1024 candidates of an XCD that it looks up one to a thread;
# 32 columns have a line of their own
@pytest.mark.parametrize("batch,heads,longest,d", [
    (512, 8, 128, 64), (513, 8, 128, 64), (64, 8, 512, 128), (65, 8, 512, 64), (28, 8, 1000, 64), (29, 8, 1000, 64), (64, 8, 1000, 32), (65, 8, 1000, 32),
    (255, 4, 384, 64), (256, 4, 384, 64), (257, 4, 384, 64), (256, 8, 512, 64), (257, 8, 512, 64), (205, 8, 640, 32)])
def test_items_with_and_without_lists(pkg, dev, batch, heads, longest, d):
    print(f"[case] items {batch} x {heads} heads up to {longest}, {d} columns", flush=True)
    gen = torch.Generator().manual_seed(batch + longest)
    lengths = torch.randint(0, longest + 1, (batch,), generator=gen).tolist()
    lengths[0], lengths[1], lengths[-1] = longest, 0, longest
    q, k, v, offs, t = make_case(batch, lengths, heads, d, targets=[min(3, n) for n in lengths])
    args = [longest, 0.125] + [x.to(dev) for x in (q, k, v, offs)]
    ranked = pkg.hstu_mha(*args, num_targets=t.to(dev), sort_by_length=True)
    plain = pkg.hstu_mha(*args, num_targets=t.to(dev))
    torch.cuda.synchronize()
    assert torch.equal(ranked, plain)
    some = [0, 1, 2, batch // 2, batch - 2, batch - 1]  # (the reference on the host takes the time)
    for b in some:
        lo, hi = int(offs[b]), int(offs[b + 1])
        if hi == lo:
            continue
        one = O.hstu_mha_per_sequence(longest, 0.125, q[lo:hi].float(), k[lo:hi].float(), v[lo:hi].float(), torch.tensor([0, hi - lo]), num_targets=t[b : b + 1].long())
        assert_parity(plain[lo:hi], one, f"items of sequence {b}")


@pytest.mark.parametrize("batch,heads,longest,window,contextual", [(520, 8, 128, 0, 10), (70, 8, 512, 100, 6), (300, 4, 640, 0, 130), (33, 8, 1000, 200, 3)])
def test_lists_with_contextual_rows(pkg, dev, batch, heads, longest, window, contextual):
    """The one-group kernel through lists where a sequence's first row block is its longest: against the same call without scratch memory, which deals the row blocks
    arithmetically, and some sequences against the oracle."""
    from generative_recommenders_amd.ops import hip_backend as hb

    print(f"[case] lists with {contextual} contextual rows {batch} x {heads} heads up to {longest}, window {window}", flush=True)
    gen = torch.Generator().manual_seed(batch + contextual)
    lengths = torch.randint(contextual + 3, longest + 1, (batch,), generator=gen).tolist()
    lengths[0], lengths[1], lengths[-1] = longest, 0, contextual + 3
    q, k, v, offs, t = make_case(batch, lengths, heads, 64, targets=[min(3, n) for n in lengths])
    form, items, wgs = hb.plan_grid_for(batch, heads, 64, 64, q.shape[0], q.shape[0], longest, tile_config=3)
    assert form == "whole" and items > wgs  # (counters and lists, not a workgroup for every item there could be)
    dq, dk, dv, do, dt = (x.to(dev) for x in (q, k, v, offs, t))
    got, plain = (torch.full_like(dv, float("nan")) for _ in range(2))
    for out, limit in ((got, None), (plain, 0)):
        hb.mha_fwd(dq, dk, dv, out, do, dt, longest, 0.125, 0, window, contextual, 0, tile_config=3, workspace_bytes=limit)
    torch.cuda.synchronize()
    assert torch.equal(got, plain) and bool(torch.isfinite(got).all())
    for b in (0, 2, batch // 2, batch - 1):
        lo, hi = int(offs[b]), int(offs[b + 1])
        one = O.hstu_mha_per_sequence(longest, 0.125, q[lo:hi].float(), k[lo:hi].float(), v[lo:hi].float(), torch.tensor([0, hi - lo]), num_targets=t[b : b + 1].long(),
                                      max_attn_len=window, contextual_seq_len=contextual)
        assert_parity(got[lo:hi], one, f"contextual items of sequence {b}")
