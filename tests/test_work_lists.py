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
