"""The delta form with few row blocks: kv runs fitted to the lengths (decode_fitted), against the oracle and the unsplit kernel."""

import pytest
import torch

from oracle import hstu_oracle as O
from util import assert_parity, make_case

pytestmark = pytest.mark.gpu

CASES = [
    # lengths (history + delta), delta, heads, dim
    ([900], 1, 1, 32),                                   # one sequence, one row
    ([450], 50, 4, 128),                                 # a run per tile
    ([129, 2500], 129, 2, 64),                           # two row blocks, the second of one row; a sequence without history
    ([2000, 100, 64, 1037, 700], 64, 3, 128),            # tile multiples, heads that do not divide the XCDs
    ([5000, 300], 300, 1, 128),                          # row blocks of 128 and of 256 with a part over
    ([6000, 40, 3513] + [65] * 61, 33, 1, 64),           # 64 sequences (every lane), most of them one or two tiles
    # one tile among long histories, whose longest runs are 41 tiles (41 * (1 / 41) is below 1 in fp32): not a run more than workgroups
    ([204 * 64 - 5, 164 * 64 - 3] * 3 + [204 * 64, 40], 16, 8, 32),
    # fewer than four workgroups per sequence: the tiles as one line (decode_line)
    ([2000 + 37 * i for i in range(18)], 3, 8, 128),     # parts that end inside sequences
    ([133] * 32 + [4000] * 32, 33, 4, 64),               # 64 sequences; parts that hold many of them, sequences in several parts
    ([300, 8000] + [3640] * 30 + [4096, 301], 300, 2, 32),  # row blocks with a part over, sequences without history, whole tiles
    ([500 + 331 * i for i in range(20)], 129, 8, 128),   # more sequences than workgroups per plane, two row blocks
]


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float8_e4m3fn])
@pytest.mark.parametrize("lengths,delta,heads,dim", CASES)
@pytest.mark.parametrize("cfg", [0, 2])
def test_fitted_runs(pkg, dev, lengths, delta, heads, dim, dtype, cfg):
    print(f"[case] fitted runs {len(lengths)} sequences up to {max(lengths)}, delta {delta}, {heads} x {dim} {dtype} cfg {cfg}", flush=True)
    from generative_recommenders_amd.ops import hip_backend as hb

    B, N, alpha = len(lengths), max(lengths) + 7, dim**-0.5
    q, k, v, offs, t = make_case(11, lengths, heads, dim, targets=[min(delta, 5)] * B, delta_size=delta)
    form = hb.plan_grid_for(B, heads, dim, dim, B * delta, int(offs[-1]), N, delta_size=delta, tile_config=cfg)[0]
    q, k, v = (x.to(dtype) for x in (q, k, v))
    args = [N, alpha] + [x.to(dev) for x in (q, k, v, offs)]
    got = pkg.delta_hstu_mha(*args, num_targets=t.to(dev), tile_config=cfg)
    again = pkg.delta_hstu_mha(*args, num_targets=t.to(dev), tile_config=cfg)
    one = pkg.delta_hstu_mha(*args, num_targets=t.to(dev), tile_config=cfg, kv_splits=1)
    torch.cuda.synchronize()
    assert form == ("line" if (lengths, delta, heads, dim) in CASES[-4:] else "fitted")
    assert torch.equal(got, again)
    # the same products, summed in fp32 run by run: what is left is the rounding of the result (at most 2^-8 of it, in bf16)
    assert float((got.float() - one.float()).norm() / one.float().norm()) <= 2.0**-8
    if dtype == torch.bfloat16:
        assert_parity(got, O.cached_hstu_mha_per_sequence(N, alpha, q.float(), k.float(), v.float(), offs, t), "fitted runs")


def test_runs_at_scratch_limits(pkg, dev):
    """Workspaces that hold the fitted runs, fewer equal ones, none: the same products in another order."""
    from generative_recommenders_amd.ops import hip_backend as hb

    lengths, delta, heads, dim = [2000, 100, 64, 1037, 7000], 64, 3, 128
    B, N, alpha = len(lengths), max(lengths) + 7, dim**-0.5
    q, k, v, offs, _ = make_case(12, lengths, heads, dim, delta_size=delta)
    want = O.cached_hstu_mha_per_sequence(N, alpha, q.float(), k.float(), v.float(), offs, None)
    q, k, v, offs = (x.to(dev) for x in (q, k, v, offs))
    run = B * delta * heads * dim * 4
    for limit in (None, 8 * run + 4096, 3 * run + 4096, 2 * run + 4096, run, 600, 0):
        print(f"[case] runs with {limit} bytes of scratch memory", flush=True)
        out = torch.full((B * delta, heads, dim), float("nan"), dtype=q.dtype, device=dev)
        hb.mha_fwd(q, k, v, out, offs, None, N, alpha, delta, 0, 0, 0, workspace_bytes=limit)
        torch.cuda.synchronize()
        assert_parity(out, want, f"{limit} bytes")


def test_a_line_at_scratch_limits(pkg, dev):
    """Workspaces that hold a line's partial sums, one byte less, none: the plan falls back and the result stays."""
    from generative_recommenders_amd.ops import hip_backend as hb

    lengths, delta, heads, dim = [500 + 331 * i for i in range(20)], 129, 4, 64
    B, N, alpha = len(lengths), max(lengths) + 7, dim**-0.5
    q, k, v, offs, _ = make_case(13, lengths, heads, dim, delta_size=delta)
    want = O.cached_hstu_mha_per_sequence(N, alpha, q.float(), k.float(), v.float(), offs, None)
    sizes = (B, heads, dim, dim, B * delta, int(offs[-1]), N)
    need = hb._plan_args(*sizes, delta, 0, 0, False, hb.HSTU_BF16, None).workspace_bytes
    q, k, v, offs = (x.to(dev) for x in (q, k, v, offs))
    forms = []
    for limit in (need, need - 1, need // 4, 600, 0):
        forms.append(hb.plan_grid_for(*sizes, delta_size=delta, workspace_bytes=limit)[0])
        print(f"[case] a line with {limit} bytes of scratch memory: {forms[-1]}", flush=True)
        out = torch.full((B * delta, heads, dim), float("nan"), dtype=q.dtype, device=dev)
        hb.mha_fwd(q, k, v, out, offs, None, N, alpha, delta, 0, 0, 0, workspace_bytes=limit)
        torch.cuda.synchronize()
        assert_parity(out, want, f"{limit} bytes")
    assert forms[0] == "line" and "line" not in forms[1:]


def test_a_line_past_sequences_shorter_than_the_candidates(pkg, dev):
    """They have no result (the caller's contract is broken for them): their rows stay as they were, the others' are what they are without the line."""
    from generative_recommenders_amd.ops import hip_backend as hb

    lengths, delta, heads, dim = [2000, 30, 2600, 0] + [2000 + 37 * i for i in range(14)] + [1], 64, 8, 128
    B, N, alpha = len(lengths), 2700, dim**-0.5
    assert hb.plan_grid_for(B, heads, dim, dim, B * delta, sum(lengths), N, delta_size=delta)[0] == "line"
    print("[case] a line past short sequences", flush=True)
    q, k, v, offs = (x.to(dev) for x in make_case(14, lengths, heads, dim, delta_size=delta)[:4])
    got, whole = (torch.full((B, delta, heads, dim), 7.0, dtype=q.dtype, device=dev) for _ in range(2))
    hb.mha_fwd(q, k, v, got.view(B * delta, heads, dim), offs, None, N, alpha, delta, 0, 0, 0)
    hb.mha_fwd(q, k, v, whole.view(B * delta, heads, dim), offs, None, N, alpha, delta, 0, 0, 0, kv_splits=1)
    torch.cuda.synchronize()
    short = torch.tensor([n < delta for n in lengths], device=dev)
    assert bool((got[short] == 7.0).all()) and bool((whole[short] == 7.0).all())
    assert float((got[~short].float() - whole[~short].float()).norm() / whole[~short].float().norm()) <= 2.0**-8
