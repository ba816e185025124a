"""The decode-step token-selection calls whose time matters, as data.

Each case is one call (or one decode step) of the public entry points of
``nvjsel`` on device tensors: the fused LM-head projection with greedy top-1 or
Gumbel-max sampling, the dense-logits + top-k verifier route, the logits
sampler, and the sampled step from the hidden state (key derivation, logits,
filters).  Inputs follow a real decode step: LM-head weights N(0, 0.02), hidden
states whose logits have the spread of a served model's row (standard deviation
about 2, a few tokens well above the bulk), and sampler logits with a Zipf tail.
"""
from __future__ import annotations

import math
import os
import sys

import torch

_PKG = os.path.abspath("nano-vllm-jax_amd")  # the package's folder is not importable by its own name
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

import nvjsel  # noqa: E402

VOCAB, HIDDEN = 248320, 1024  # the served model's LM head (tied table [VOCAB, HIDDEN])
_DT = {"f32": torch.float32, "bf16": torch.bfloat16, "f16": torch.float16}
_SIZE = {"f32": 4, "bf16": 2, "f16": 2}


def _lm(name, kind, rows, *, vocab=VOCAB, hidden=HIDDEN, layout="vh", weight="bf16", act="bf16", norm=False, k=0):
    return {"name": name, "kind": kind, "rows": rows, "vocab": vocab, "hidden": hidden, "layout": layout,
            "weight": weight, "act": act, "norm": norm, "k": k}


def _sampler(name, rows, *, vocab=VOCAB, dtype="f32", filters=False):
    return {"name": name, "kind": "sampler", "rows": rows, "vocab": vocab, "dtype": dtype, "filters": filters}


def listed():
    return [
        # one interactive sequence, greedy, the promoted config: pre-norm hidden, bf16 activations
        _lm("greedy_one", "greedy", 1, norm=True),
        # a verifier or a full server's greedy step: 64 sequences x width 4 in one call
        _lm("greedy_rows256", "greedy", 256),
        # a busy server's sampled step on the tied table
        _lm("sample_rows64", "sample", 64),
        # the same at the largest batch with the default fp32 activations and the final norm in the call
        _lm("sample_f32_rows256", "sample", 256, act="f32", norm=True),
        # the materialised [H, V] head of the promoted server config, a moderate batch
        _lm("sample_hv_rows24", "sample", 24, layout="hv"),
        # speculative verification that wants top-k values too: 16 sequences x width 5
        _lm("verify_topk_rows80", "verify", 80, k=20),
        # a larger model of the usual shape: wider hidden, another vocabulary
        _lm("greedy_wide_rows16", "greedy", 16, vocab=151936, hidden=2560),
        # a half-precision checkpoint
        _lm("greedy_f16_rows12", "greedy", 12, vocab=128256, hidden=2048, weight="f16", act="f16"),
        # a materialised head of an unpadded, odd vocabulary
        _lm("sample_hv_odd_rows4", "sample", 4, vocab=50257, hidden=768, layout="hv"),
        # per-row temperature, top-k and top-p over a full server's bf16 logits
        _sampler("sampler_mixed_rows256", 256, dtype="bf16", filters=True),
        # the smallest call: temperature sampling of a few rows of f32 logits
        _sampler("sampler_temps_rows8", 8),
        # the sampled step with filters: keys, logits from the hidden state, filtered sampling
        _lm("step_filtered_rows32", "step", 32),
    ]


def _log_uniform(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["greedy", "greedy", "sample", "sample", "verify", "step", "sampler"])
    vocab = _log_uniform(rng, 32000, VOCAB)  # any size, odd ones too
    if rng.random() < 0.5:
        vocab -= vocab % 64  # a padded vocabulary
    rows = _log_uniform(rng, 1, 256)
    if kind == "sampler":
        c = _sampler("", rows, vocab=vocab, dtype=rng.choice(["f32", "bf16", "f16"]), filters=rng.random() < 0.6)
    else:
        hidden = rng.choice([512, 768, 1024, 1024, 1536, 2048, 2560, 4096])
        while vocab * hidden > VOCAB * HIDDEN:
            hidden //= 2
        hidden -= hidden % 64
        weight = rng.choice(["bf16", "bf16", "bf16", "bf16", "f16"])
        act = "f16" if weight == "f16" else rng.choice(["bf16", "f32"])
        layout = rng.choice(["vh", "vh", "hv"])
        if layout == "hv":
            rows = _log_uniform(rng, 1, 64)
        c = _lm("", kind, rows, vocab=vocab, hidden=hidden, layout=layout, weight=weight, act=act,
                norm=kind in ("greedy", "sample") and rng.random() < 0.5, k=rng.randint(1, 64) if kind == "verify" else 0)
    del c["name"]
    return c


def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed))
    return g


def _pick(g, values, n, dtype):
    return torch.tensor(values, device="cuda", dtype=dtype)[torch.randint(0, len(values), (n,), device="cuda", generator=g)]


def _row_parameters(g, rows, filters):
    """Temperatures (greedy rows among them), and the served mix of top-k / top-p."""
    p = {"temperatures": _pick(g, [0.0, 0.6, 0.7, 1.0] if filters else [0.6, 0.7, 0.8, 1.0], rows, torch.float32)}
    if filters:
        p["top_k"] = _pick(g, [0, 20, 100], rows, torch.int32)
        p["top_p"] = _pick(g, [1.0, 0.95, 0.8], rows, torch.float32)
    return p


def _head(c, g):
    """LM-head weight in its layout and the hidden rows: noise that spreads the
    logits by about 2, plus a few weight rows, so that some tokens stand out."""
    v, h, n = c["vocab"], c["hidden"], c["rows"]
    shape = (v, h) if c["layout"] == "vh" else (h, v)
    w = torch.empty(shape, dtype=_DT[c["weight"]], device="cuda").normal_(0.0, 0.02, generator=g)
    scale = 2.0 / (0.02 * math.sqrt(h))
    x = torch.randn(n, h, device="cuda", generator=g) * scale
    for top in (20.0, 12.0, 10.0):
        t = torch.randint(0, v, (n,), device="cuda", generator=g)
        peak = top * (0.75 + 0.25 * torch.rand(n, 1, device="cuda", generator=g))
        x += peak / (h * 4e-4) * (w[t] if c["layout"] == "vh" else w[:, t].T).float()
    norm_weight = None
    if c["norm"]:  # the state before the final norm: (1 + w) carries the scale
        norm_weight = scale * (1.0 + 0.1 * torch.randn(h, device="cuda", generator=g)) - 1.0
        x = 3.0 * x / (1.0 + norm_weight)
    return w, x.to(_DT[c["act"]]), norm_weight


def prepare(case, seed):
    g, n = _gen(seed), case["rows"]
    s = {"kind": case["kind"], "slots": torch.randperm(n, device="cuda", generator=g).to(torch.int32),
         "counters": torch.randint(0, 4096, (n,), device="cuda", generator=g, dtype=torch.int32)}
    if case["kind"] == "sampler":
        x = torch.empty(n, case["vocab"], device="cuda").exponential_(1.0, generator=g)
        x = x * (1.05 + 0.25 * torch.rand(n, 1, device="cuda", generator=g))
        x = x + torch.randn(n, case["vocab"], device="cuda", generator=g)
        s["logits"] = x.to(_DT[case["dtype"]])
        s["args"] = _row_parameters(g, n, case["filters"])
        s["keys"] = nvjsel.derive_rng_keys(s["slots"], s["counters"])[0]
        return s
    w, x, norm_weight = _head(case, g)
    s["weight"], s["k"] = w, case["k"]
    # the tied table is handed over as its [H, V] view, as an engine does
    s["operand"] = w.T if case["layout"] == "vh" else w
    s["hidden"] = x.reshape(n, 1, case["hidden"])
    s["norm"] = {} if norm_weight is None else {
        "norm_weight": norm_weight, "rms_norm_eps": 1e-6, "act_dtype": _DT[case["act"]]}
    if case["kind"] in ("sample", "step"):
        s["args"] = _row_parameters(g, n, case["kind"] == "step")
        s["keys"] = nvjsel.derive_rng_keys(s["slots"], s["counters"])[0]
    return s


def run(state):
    kind = state["kind"]
    if kind == "sampler":
        return nvjsel.sample_token_ids(state["logits"], rng_keys=state["keys"], **state["args"])
    if kind == "greedy":
        return nvjsel.lm_head_greedy_top1_hip(state["hidden"], state["operand"], return_best=True, **state["norm"])
    if kind == "sample":
        return nvjsel.lm_head_sample_token_ids(state["hidden"], state["operand"], rng_keys=state["keys"],
                                               **state["args"], **state["norm"])
    if kind == "verify":
        return nvjsel.lm_head_token_ids_and_topk(state["hidden"], state["operand"], top_k=state["k"])
    keys, counters = nvjsel.derive_rng_keys(state["slots"], state["counters"])
    ids = nvjsel.lm_head_sample_token_ids(state["hidden"], state["operand"], rng_keys=keys, **state["args"])
    return ids, keys, counters


def work(case):
    n, v = case["rows"], case["vocab"]
    if case["kind"] == "sampler":
        # one read of the logits; a comparison per value
        return {"bytes": n * v * _SIZE[case["dtype"]] + n * 24, "flops": n * v}
    h = case["hidden"]
    out = n * (4 + 8 * case["k"])
    return {"bytes": v * h * _SIZE[case["weight"]] + n * h * _SIZE[case["act"]] + n * 24 + out, "flops": 2 * n * v * h}


def tolerance(case):
    # The best logit of a 16-bit dot is rounded to 16 bits: two sums in another
    # order may round apart by one unit in the last place (2^-7, 2^-10 of the
    # value at most).  fp32 activations keep the fp32 sum: 4e-8 to 5e-7 off 64
    # bits measured over these sizes.  Tokens agree (the inputs' best scores are
    # apart by far more than a rounding; none of 80 x 20 indices differed between
    # one pass and passes of 2 rows); of the verifier's indices, two values that
    # round together or apart may swap.
    if case["kind"] in ("sampler", "sample", "step"):
        return {"rel": 0.0, "differ": 0.004}
    rel = {"bf16": 8e-3, "f16": 1e-3, "f32": 2e-6}[case["act"]]
    return {"rel": rel, "max": 2 * rel, "differ": 0.005}


def exact(case, seed):
    """The winning logits (greedy) and the sorted top values (verify) in 64
    bits; tokens, indices and keys have no such value."""
    if case["kind"] not in ("greedy", "verify"):
        return None
    s = prepare(case, seed)
    x = s["hidden"].reshape(case["rows"], case["hidden"]).double()
    if s["norm"]:
        x = x / torch.sqrt((x * x).mean(dim=1, keepdim=True) + 1e-6) * (1.0 + s["norm"]["norm_weight"].double())
    w, v = s["weight"], case["vocab"]
    best = []
    for v0 in range(0, v, 65536):
        part = w[v0:v0 + 65536].double().T if case["layout"] == "vh" else w[:, v0:v0 + 65536].double()
        best.append(torch.topk(x @ part.contiguous(), min(max(1, case["k"]), part.shape[1]), dim=1).values)
    top = torch.topk(torch.cat(best, dim=1), max(1, case["k"]), dim=1).values
    if case["kind"] == "greedy":
        return [None, top[:, 0]]
    return [None, top[:, None, :], None]
