"""What this framework is used for, as cases that can be timed: listed ones, and more drawn from the same ranges.

A case is a dict of plain values; ``op`` says which of the user's programs it is:

* ``layer``        one layer of a ranker: producer of u, q, k, v -> jagged attention -> output step; with ``prefill``, also
                   the K and V rows of the histories split from those of the targets, for the cache
* ``cached``       the same layer for a micro-batch of candidates against a K/V cache (all sequences get ``delta`` new rows)
* ``layer_fp8``    producer with 8-bit copies of v, q, k -> 8-bit attention
* ``train_layer``  the layer forward and backward: its output, the gradients of its input and of every weight
* ``attention``    the attention alone on column slices of one buffer
* ``train_attention``  the attention forward and backward

The shape of a case (lengths, targets) depends on the case alone, through ``shape_seed``; values, and which sequence has
which length, on the seed that ``prepare`` gets.
"""

import math

import numpy as np
import torch

import __graft_entry__

pkg = __graft_entry__.load_package()
from generative_recommenders_amd import workloads  # noqa: E402
from generative_recommenders_amd.ops import hip_backend  # noqa: E402
from generative_recommenders_amd.ops.hstu_compute import hstu_compute_uqvk_fp8  # noqa: E402

EPS = 1e-6
DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16, "fp32": torch.float32}
# Every field that not all cases name, with the value that stands for "not used".
DEFAULTS = {
    "op": "layer", "dtype": "bf16", "batch": 1, "lengths": "uniform", "lo": 1, "hi": 1, "heads": 4, "dqk": 128, "dv": 128, "d_model": 512,
    "targets": 0, "delta": 0, "window": 0, "contextual": 0, "group_norm": False, "dropout": 0.0, "cache": "tail", "sort": False,
    "prefill": False, "keep_ds": False, "shape_seed": 0,
}


def listed():
    return [
        # One user's request: a handful of candidates scored against a short history, the cache put together row by row as
        # the reference's layer does.  Nothing but latency, launches and the host's work.
        dict(name="cached_one_user", op="cached", batch=1, lo=400, hi=400, delta=50, cache="concat", shape_seed=1),
        # A serving micro-batch: 32 users, 256 candidates each, new rows written into the cache's spare rows.
        dict(name="cached_micro_batch", op="cached", batch=32, lo=1024, hi=4096, delta=256, shape_seed=1004),
        # A few heavy users with very long histories and an odd number of candidates: little to do in parallel but the history.
        dict(name="cached_long_history", op="cached", batch=5, lo=8000, hi=16000, delta=100, shape_seed=3),
        # Ranking many short histories, targets at the end, fp16 and group norm: a layer of the smaller width.
        dict(name="layer_short_fp16", op="layer", dtype="fp16", batch=96, lo=20, hi=276, targets=20, heads=4, dqk=64, dv=64, d_model=256,
             contextual=10, group_norm=True, shape_seed=4),
        # The second baseline batch (256 sequences of 64..1024 rows) through the whole layer, as a prefill that fills the cache.
        dict(name="layer_prefill", op="layer", batch=256, lo=64, hi=1024, targets=20, prefill=True, shape_seed=1002),
        # The headline: every sequence 8192 rows, nothing but matrix work.
        dict(name="attention_full", op="attention", batch=64, lengths="equal", lo=8192, hi=8192, shape_seed=1000),
        # The third baseline batch: lengths of a power law, a window, a contextual prefix, targets.
        dict(name="attention_window", op="attention", batch=64, lengths="zipf", lo=256, hi=8192, targets=512, window=2048, contextual=6,
             sort=True, shape_seed=1003),
        # The fifth: long sequences in 8 bits from the producer on, eight heads.
        dict(name="layer_fp8", op="layer_fp8", batch=16, lo=4096, hi=16384, targets=256, heads=8, shape_seed=1005),
        # A training step of the layer at the sizes of the operator tests: few short sequences, unequal head dims.
        dict(name="train_layer_small", op="train_layer", dtype="fp16", batch=8, lo=20, hi=150, targets=20, heads=2, dqk=64, dv=128,
             d_model=256, group_norm=True, shape_seed=5),
        # A training step on a ragged batch of ordinary histories, with the output step's dropout.
        dict(name="train_layer", op="train_layer", batch=48, lo=200, hi=2048, targets=20, dropout=0.2, sort=True, shape_seed=6),
        # The attention's forward and backward on long ragged histories.
        dict(name="train_attention", op="train_attention", batch=32, lo=1024, hi=8192, targets=20, sort=True, shape_seed=1006),
        # ... and in the second data type of the operator tests, at their head dims.
        dict(name="train_attention_fp32", op="train_attention", dtype="fp32", batch=16, lo=100, hi=768, targets=20, heads=4, dqk=64, dv=32,
             contextual=10, shape_seed=7),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _cost(c):
    """Rough microseconds of one pass, to keep drawn cases below the listed ones."""
    w = work(c)
    slow = {"train_layer": 2.0, "train_attention": 2.0, "cached": 2.0}.get(c["op"], 1.0)
    return slow * max(w["flops"] / 5e8, w["bytes"] / 2e6)


def draw(rng):
    """One more case of the listed ones' ranges."""
    while True:
        op = rng.choice(["layer", "cached", "cached", "layer_fp8", "train_layer", "train_layer", "attention", "train_attention"])
        c = dict(op=op, shape_seed=rng.randrange(1 << 20), heads=rng.choice([1, 2, 4, 4, 8]))
        hi = _log_int(rng, 40, 16000 if op in ("cached", "layer_fp8") else 8192)
        c.update(hi=hi, lo=max(24, int(hi * rng.choice([0.06, 0.25, 0.5, 0.95]))), batch=_log_int(rng, 1, 256))
        if c["lo"] > hi:
            c["lo"] = hi
        c["dtype"] = rng.choice(["bf16", "bf16", "fp16"])
        c["dqk"] = c["dv"] = rng.choice([128, 128, 64, 32])
        if op != "cached":
            c["targets"] = rng.choice([0, 1, 20, min(512, c["lo"] // 2)])
            c["sort"] = rng.random() < 0.5
        if op in ("layer", "train_layer", "cached"):
            c["d_model"] = rng.choice([512, 512, 256, 384, 640])
            c["group_norm"] = rng.random() < 0.3
        if op in ("attention", "layer", "train_layer", "train_attention"):
            c["contextual"] = rng.choice([0, 0, 6, 10])
        if op in ("attention", "train_attention"):
            c["window"] = rng.choice([0, 0, max(1, hi // 4)])
            if rng.random() < 0.3:
                c["dv"] = rng.choice([32, 64, 128])
            if rng.random() < 0.25:
                c["dtype"] = "fp32"
            if op == "attention" and rng.random() < 0.2:
                c["lengths"] = "equal"
                c["lo"] = hi
            if op == "train_attention":
                c["keep_ds"] = c["dtype"] != "fp32" and rng.random() < 0.3
        if op == "layer_fp8":
            c["dtype"], c["dqk"], c["dv"], c["heads"] = "bf16", 128, 128, rng.choice([2, 4, 8])
            c["d_model"] = rng.choice([256, 512])
        if op == "layer":
            c["prefill"] = c["targets"] > 0 and rng.random() < 0.5
        if op == "cached":
            c["delta"] = _log_int(rng, 1, 512)
            c["cache"] = rng.choice(["tail", "concat"])
            c["batch"] = _log_int(rng, 1, 64)
        if op == "train_layer":
            c["dropout"] = rng.choice([0.0, 0.1, 0.2])
        if _cost(_full(c)) <= 8000 and _rows(_full(c)) * c["heads"] * c["dqk"] <= 6 << 26:
            return c


def _full(case):
    return {**DEFAULTS, **case}


def _lengths(c):
    """Lengths of the histories (of the whole sequences where nothing is cached) and numbers of targets."""
    rng = np.random.default_rng(c["shape_seed"])
    if c["lengths"] == "equal":
        n = np.full(c["batch"], c["hi"], dtype=np.int64)
    elif c["lengths"] == "zipf":
        n = np.clip(rng.zipf(1.2, size=c["batch"]), c["lo"], c["hi"]).astype(np.int64)
    else:
        n = rng.integers(c["lo"], c["hi"] + 1, size=c["batch"]).astype(np.int64)
    if c["targets"] <= 0:
        return n, None
    return n, np.minimum(rng.integers(1, c["targets"] + 1, size=c["batch"]), np.maximum(n - c["contextual"] - 1, 0)).astype(np.int64)


def _rows(c):
    return int(_lengths(c)[0].sum()) + c["batch"] * c["delta"]


def _max_seq_len(c):
    return c["hi"] + c["delta"]


def _params(c, draw, dtype):
    """A layer's weights: as they are after the usual initialisation, norms near the identity."""
    H, dqk, dv, d = c["heads"], c["dqk"], c["dv"], c["d_model"]
    n_out, width = (2 * dv + 2 * dqk) * H, H * dv
    norm = H if c["group_norm"] else width
    return {
        "norm_weight": (1 + 0.1 * draw(d)).to(dtype), "norm_bias": (0.1 * draw(d)).to(dtype),
        "uvqk_weight": (draw(d, n_out) / d**0.5).to(dtype), "uvqk_bias": (0.1 * draw(n_out)).to(dtype),
        "out_norm_weight": (1 + 0.1 * draw(norm)).to(dtype), "out_norm_bias": (0.1 * draw(norm)).to(dtype),
        "out_weight": (draw(3 * width, d) / (3 * width) ** 0.5).to(dtype),
    }


def prepare(case, seed):
    c = _full(case)
    dev = torch.device("cuda")
    gen = torch.Generator(device=dev).manual_seed(int(seed))
    dtype = DTYPES[c["dtype"]]
    H, dqk, dv, d = c["heads"], c["dqk"], c["dv"], c["d_model"]

    def draw(*shape):
        return torch.randn(shape, generator=gen, device=dev)

    n, t = _lengths(c)
    place = np.random.default_rng(int(seed)).permutation(c["batch"])
    n, t = n[place], (None if t is None else t[place])

    def offsets_of(lengths):
        return torch.from_numpy(np.concatenate([[0], np.cumsum(lengths)]).astype(np.int64)).to(dev)

    s = {
        "case": c, "alpha": 1.0 / dqk**0.5, "max_seq_len": _max_seq_len(c), "offsets": offsets_of(n + c["delta"]),
        "targets": None if t is None else torch.from_numpy(t).to(dev),
    }
    L = int(n.sum())
    op = c["op"]
    if op in ("layer", "layer_fp8", "train_layer"):
        s["x"] = draw(L, d).to(dtype)
        s.update(_params(c, draw, dtype))
        if c["prefill"]:
            s["history"], s["target_offsets"] = offsets_of(n - t), offsets_of(t)
            s["totals"] = int((n - t).sum()), int(t.sum())
        if op == "layer_fp8":
            # the scales a serving loop carries over from the batches before: largest magnitude / 448
            s["scales"] = tuple((1.3 * 5.5) / 448.0 for _ in range(3))
        if op == "train_layer":
            s["dout"] = draw(L, d).to(dtype)
            for k in ("x",) + PARAMS:
                s[k].requires_grad_(True)
    elif op == "cached":
        s["x"] = draw(c["batch"] * c["delta"], d).to(dtype)
        s.update(_params(c, draw, dtype))
        s["targets"] = torch.full((c["batch"],), c["delta"], dtype=torch.int64, device=dev)
        s["history"] = offsets_of(n)
        rows = L + (c["batch"] * c["delta"] if c["cache"] == "tail" else 0)
        s["k_cache"], s["v_cache"] = draw(rows, H * dqk).to(dtype), draw(rows, H * dv).to(dtype)
    else:
        # v | q | k side by side, as the producer leaves them
        buffer = draw(L, H * (dv + 2 * dqk)).to(dtype)
        v, q, k = torch.split(buffer, [H * dv, H * dqk, H * dqk], dim=1)
        s["q"], s["k"], s["v"] = q.view(L, H, dqk), k.view(L, H, dqk), v.view(L, H, dv)
        if op == "train_attention":
            s["dout"] = draw(L, H, dv).to(dtype)
            for name in "qkv":
                s[name] = s[name].detach().requires_grad_(True)
            if c["keep_ds"]:
                need = hip_backend.mha_bwd_workspace_bytes(L, c["batch"], H, s["max_seq_len"])
                s["workspace"] = torch.empty(need, dtype=torch.uint8, device=dev)
    return s


PARAMS = ("norm_weight", "norm_bias", "uvqk_weight", "uvqk_bias", "out_norm_weight", "out_norm_bias", "out_weight")


def _output_step(s, attn, u, training):
    c = s["case"]
    return pkg.hstu_compute_output(
        attn, u, s["x"], s["out_norm_weight"], s["out_norm_bias"], EPS, s["out_weight"], c["heads"], c["dv"], c["dropout"] if training else 0.0,
        training, True, True, "none", c["group_norm"], True, seed=(1234, 0) if training else None,
    )


def _layer(s, training):
    c = s["case"]
    u, attn, k, v = pkg.hstu_preprocess_and_attention(
        s["x"], s["norm_weight"], s["norm_bias"], EPS, c["heads"], c["dqk"], c["dv"], s["uvqk_weight"], s["uvqk_bias"], s["max_seq_len"],
        s["offsets"], s["alpha"], True, s["targets"], c["window"], c["contextual"], True, True, c["sort"],
    )
    return _output_step(s, attn, u, training), k, v


def _attention(s, q, k, v, **more):
    c = s["case"]
    return pkg.hstu_mha(
        s["max_seq_len"], s["alpha"], q, k, v, s["offsets"], num_targets=s["targets"], max_attn_len=c["window"],
        contextual_seq_len=c["contextual"], sort_by_length=c["sort"], **more,
    )


def _history_rows(s, rows):
    """(rows of the histories, rows of the targets)"""
    c = s["case"]
    return pkg.split_2D_jagged(
        s["max_seq_len"], rows, total_len_left=s["totals"][0], total_len_right=s["totals"][1], max_len_left=c["hi"], max_len_right=c["targets"],
        offsets_left=s["history"], offsets_right=s["target_offsets"],
    )


def _cached(s):
    c = s["case"]
    B, H, dqk, dv = c["batch"], c["heads"], c["dqk"], c["dv"]
    u, q, k, v = pkg.hstu_compute_uqvk(s["x"], s["norm_weight"], s["norm_bias"], EPS, H, dqk, dv, s["uvqk_weight"], s["uvqk_bias"])
    rows = []
    for cache, new in ((s["k_cache"], k.flatten(1, 2)), (s["v_cache"], v.flatten(1, 2))):
        if c["cache"] == "tail":
            rows.append(pkg.write_kv_tail(cache, s["offsets"], new))
        else:
            rows.append(pkg.concat_2D_jagged(s["max_seq_len"], cache, new, c["hi"], c["delta"], s["history"], None))
    attn = pkg.delta_hstu_mha(
        s["max_seq_len"], s["alpha"], q, rows[0].view(-1, H, dqk), rows[1].view(-1, H, dv), s["offsets"], num_targets=s["targets"],
    )
    return _output_step(s, attn.view(B * c["delta"], H * dv), u, False), rows[0], rows[1]


def run(s):
    c = s["case"]
    op = c["op"]
    if op == "train_layer":
        out, _, _ = _layer(s, True)
        return [out] + list(torch.autograd.grad(out, [s[k] for k in ("x",) + PARAMS], s["dout"]))
    if op == "train_attention":
        out = _attention(s, s["q"], s["k"], s["v"], bwd_workspace=s.get("workspace"))
        return [out] + list(torch.autograd.grad(out, [s["q"], s["k"], s["v"]], s["dout"]))
    with torch.no_grad():
        if op == "layer":
            out, k, v = _layer(s, False)
            if not c["prefill"]:
                return [out, k, v]
            return [out] + [_history_rows(s, rows.flatten(1, 2)) for rows in (k, v)]
        if op == "cached":
            return list(_cached(s))
        if op == "layer_fp8":
            q_scale, k_scale, v_scale = s["scales"]
            u, q8, k8, v8, absmax = hstu_compute_uqvk_fp8(
                s["x"], s["norm_weight"], s["norm_bias"], EPS, c["heads"], c["dqk"], c["dv"], s["uvqk_weight"], s["uvqk_bias"], q_scale, k_scale,
                v_scale,
            )
            return [_attention(s, q8, k8, v8, q_scale=q_scale, k_scale=k_scale, v_scale=v_scale), u, absmax]
        return [_attention(s, s["q"], s["k"], s["v"])]


def work(case):
    c = _full(case)
    n, t = _lengths(c)
    B, H, dqk, dv, d = c["batch"], c["heads"], c["dqk"], c["dv"], c["d_model"]
    op = c["op"]
    es = 4 if c["dtype"] == "fp32" else 2
    new = B * c["delta"] if op == "cached" else int(n.sum())
    total = int(n.sum()) + (new if op == "cached" else 0)
    row = H * (2 * dqk + 2 * dv)  # u, v, q, k of a row
    wl = workloads.Workload(
        "", B, H, dqk, dv, _max_seq_len(c), n + c["delta"], num_targets=np.full(B, c["delta"]) if op == "cached" else t, max_attn_len=c["window"],
        contextual_seq_len=c["contextual"], delta_size=c["delta"] if op == "cached" else 0,
    )
    pairs = float(workloads.count_valid_pairs(wl)) * H
    attention = 2.0 * (dqk + dv) * pairs
    backward = 2.0 * (3 * dqk + 2 * dv) * pairs
    dense = 2.0 * new * d * row + (2.0 * new * 3 * H * dv * d if op != "layer_fp8" else 0.0)
    weights = es * (d * row + (3 * H * dv * d if op != "layer_fp8" else 0))
    if op == "attention":
        return {"bytes": es * new * H * (2 * dqk + 2 * dv), "flops": attention}
    if op == "train_attention":
        return {"bytes": es * new * H * (4 * dqk + 4 * dv), "flops": attention + backward}
    if op == "layer":  # x in; the layer's output and the k and v to cache out
        return {"bytes": es * new * (2 * d + H * (dqk + dv)) + weights, "flops": dense + attention}
    if op == "layer_fp8":  # x in; u and the attention's output out
        return {"bytes": 2 * new * (d + 2 * H * dv) + weights, "flops": dense + attention}
    if op == "cached":  # x and the history in (and out again where the cache is put together anew), the new rows and the output out
        kept = es * (total - new) * H * (dqk + dv) * (2 if c["cache"] == "concat" else 1)
        return {"bytes": kept + es * new * (2 * d + H * (dqk + dv)) + weights, "flops": dense + attention}
    return {"bytes": 4 * es * new * d + 2 * weights, "flops": 3 * dense + attention + backward}


# About four times the distance from the same path in 64 bits (relative 2-norm; largest difference over the larger of value
# and root mean square), as measured on the listed cases (fewer sequences of the long ones) and on drawn ones:
# forward bf16 2.9e-3 / 0.022, fp16 3.1e-4 / 0.0023, fp32 (fp16 products) 4.7e-4 / 0.0031; attention with gradients bf16
# 2.9e-3 / 0.017, fp32 (bf16 products in the backward) 4.1e-3 / 0.029; layer with gradients bf16 6.1e-3 / 0.049, fp16 8.2e-4 /
# 0.0079; 8 bits 2.2e-2 / 0.17 on long sequences, more on short ones.
TOLERANCES = {
    ("forward", "bf16"): {"rel": 0.012, "max": 0.09}, ("forward", "fp16"): {"rel": 0.0013, "max": 0.01},
    ("forward", "fp32"): {"rel": 0.002, "max": 0.013},
    ("train_attention", "bf16"): {"rel": 0.012, "max": 0.09}, ("train_attention", "fp16"): {"rel": 0.0033, "max": 0.032},
    ("train_attention", "fp32"): {"rel": 0.016, "max": 0.12},
    ("train_layer", "bf16"): {"rel": 0.024, "max": 0.2}, ("train_layer", "fp16"): {"rel": 0.0033, "max": 0.032},
}


def tolerance(case):
    c = _full(case)
    if c["op"] == "layer_fp8":
        return {"rel": 0.03, "max": 0.7}
    return dict(TOLERANCES[c["op"] if c["op"].startswith("train_") else "forward", c["dtype"]])
