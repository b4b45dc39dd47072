"""The work that a user of this package has it do, as cases that can be timed and checked.

A case is one call of a public entry point of ``moe_fp8`` on one expert-parallel rank of a
256-expert DeepSeek-V3 MoE layer: 32 local experts, H = 7168, I = 2048, the operator's own sizes.

* ``run``       the operator: one layer's routed experts for the T tokens of a step;
* ``quantize``  the 1x128 activation quantizer in front of it;
* ``route``     the routing alone (a dispatcher that has to know where tokens go before they move).

T is what varies in use: 1 to 64 tokens in a decode step, a few hundred in a chunked or mixed
step, thousands in a prefill; odd values are the rule, since a scheduler packs whatever is there.
"""
from __future__ import annotations

import math
import sys
from pathlib import Path

import torch

sys.path.insert(0, str(Path(__file__).resolve().parent.parent / "rocm-flashinfer-contest_amd"))

import moe_fp8  # noqa: E402
from moe_fp8 import workloads  # noqa: E402

H, I, E_LOCAL, E_GLOBAL, TOP_K, BLOCK = 7168, 2048, 32, 256, 8, 128
N_GROUP, TOPK_GROUP = 8, 4
RSF = 2.5                      # DeepSeek-V3's routed scaling factor
RANKS = E_GLOBAL // E_LOCAL
LARGEST_T = 14107              # the longest sequence of the contest's own workloads

_DT = {"f32": torch.float32, "bf16": torch.bfloat16}


def _run_case(T, rank=0, hidden="normal", routing="even", logits="f32", out="bf16", shared="none", local_pairs=0):
    """``hidden``: "normal" rows, or "lognormal" ones (per-token amplitude exp(z), z ~ N(0, 1)), which
    make use of the precision classes.  ``routing``: "even" (a trained no-aux bias keeps the experts'
    load level) or "zipf" (a few hot experts).  ``local_pairs``: every token has exactly that many
    experts on this rank, as after a dispatch that only moves tokens to ranks with work for them; 0
    takes the tokens as they come."""
    return {"op": "run", "T": T, "rank": rank, "hidden": hidden, "routing": routing, "logits": logits,
            "out": out, "shared": shared, "local_pairs": local_pairs}


def listed():
    return [
        # the quantizer in front of a decode step (launch latency) and of a prefill (bandwidth)
        {"name": "quantize_t16", "op": "quantize", "T": 16, "x": "bf16"},
        {"name": "quantize_t8192", "op": "quantize", "T": 8192, "x": "bf16"},
        # the routing alone, for a dispatcher
        {"name": "route_t2048", "op": "route", "T": 2048, "logits": "f32"},
        # one token's decode step, two of its experts here: nothing but latency
        {"name": "run_t1", **_run_case(1, local_pairs=2)},
        # a decode batch, the package's headline size
        {"name": "run_t16", **_run_case(16, rank=1)},
        # the contest's own middle workload; bf16 logits, as a bf16 gate gives them
        {"name": "run_t55", **_run_case(55, rank=2, logits="bf16")},
        # past a decode batch: decode tokens mixed with a short prompt
        {"name": "run_t100", **_run_case(100, rank=3)},
        # a chunked-prefill step of odd size on a rank that returns its fp32 partial sum
        {"name": "run_t333", **_run_case(333, rank=4, out="f32")},
        # a prefill chunk with the shared expert's rows added in the combine
        {"name": "run_t1024", **_run_case(1024, rank=5, shared="bf16")},
        # a prefill with a few hot experts
        {"name": "run_t5000", **_run_case(5000, rank=6, routing="zipf")},
        # a large prefill whose tokens differ much in size
        {"name": "run_t8192", **_run_case(8192, rank=7, hidden="lognormal")},
        # the longest sequence of the contest's workloads
        {"name": "run_t14107", **_run_case(LARGEST_T)},
    ]


def draw(rng):
    def size(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    kind = rng.random()
    if kind < 0.15:
        return {"op": "quantize", "T": size(1, 16384), "x": rng.choice(["bf16", "bf16", "f32"])}
    if kind < 0.25:
        return {"op": "route", "T": size(1, 16384), "logits": rng.choice(["f32", "bf16"])}
    routing = rng.choice(["even", "even", "even", "zipf"])
    T = size(1, 5000 if routing == "zipf" else 13000)
    return _run_case(T, rank=rng.randrange(RANKS), hidden=rng.choice(["normal", "normal", "lognormal"]), routing=routing,
                     logits=rng.choice(["f32", "bf16"]), out=rng.choice(["bf16", "bf16", "bf16", "f32"]),
                     shared=rng.choice(["none", "none", "bf16", "f32"]), local_pairs=2 if T <= 8 else 0)


# ------------------------------------------------------------------------------------------ inputs
def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    return g


def _select(logits, bias):
    """The operator's choice of experts: ids [T, 8] ascending, by fp32 ranking of the sigmoid (taken in
    64 bits, rounded once) plus the bias; and the unbiased sigmoid in 64 bits."""
    s64 = torch.sigmoid(logits.double())
    sb = s64.float() + bias.float()
    T = sb.shape[0]
    group = sb.view(T, N_GROUP, -1).topk(2, dim=2).values.sum(2).topk(TOPK_GROUP, dim=1).indices
    kept = torch.zeros(T, N_GROUP, dtype=torch.bool, device=sb.device).scatter_(1, group, True)
    sb = sb.masked_fill(~kept.repeat_interleave(E_GLOBAL // N_GROUP, dim=1), -math.inf)
    return sb.topk(TOP_K, dim=1).indices.sort(dim=1).values, s64


def _logits_and_bias(case, g):
    T = case["T"]
    # a no-aux bias as training leaves it: small corrections between the experts
    bias = (torch.randn(E_GLOBAL, generator=g, device="cuda") * 0.02).to(torch.bfloat16)
    extra = None
    if case.get("routing") == "zipf":
        extra = workloads.zipf_logit_bias(E_GLOBAL, 1.2, torch.randperm(E_GLOBAL, generator=g, device="cuda").cpu()).cuda()

    def rows(n):
        x = torch.randn(n, E_GLOBAL, generator=g, device="cuda")
        return (x if extra is None else x + extra).to(_DT[case["logits"]])

    want = case.get("local_pairs", 0)
    if not want:
        return rows(T), bias
    got, have = [], 0
    while have < T:
        x = rows(256)
        ids, _ = _select(x, bias)
        here = ((ids // E_LOCAL) == case["rank"]).sum(1)
        got.append(x[here == want])
        have += got[-1].shape[0]
    return torch.cat(got)[:T].contiguous(), bias


def prepare(case, seed):
    g = _gen(seed)
    T = case["T"]
    if case["op"] == "quantize":
        return {"op": "quantize", "x": torch.randn(T, H, generator=g, device="cuda").to(_DT[case["x"]])}
    logits, bias = _logits_and_bias(case, g)
    if case["op"] == "route":
        return {"op": "route", "args": (logits, bias, RSF)}
    x = torch.randn(T, H, generator=g, device="cuda")
    if case["hidden"] == "lognormal":
        x *= torch.exp(torch.randn(T, 1, generator=g, device="cuda"))
    hidden, hidden_scale = workloads.quantize_rows_1x128(x)
    del x
    w13, s13, w2, s2 = workloads.make_weights(E_LOCAL, H, I, device="cuda", seed=seed + 1)
    kw = {"output_dtype": _DT[case["out"]]}
    if case["shared"] != "none":
        # a shared expert's output, of the size of the routed sum of normal rows
        kw["shared_output"] = torch.randn(T, H, generator=g, device="cuda").to(_DT[case["shared"]])
    return {"op": "run", "kw": kw,
            "args": (logits, bias, hidden, hidden_scale, w13, s13, w2, s2, E_LOCAL * case["rank"], RSF)}


def run(state):
    if state["op"] == "quantize":
        return moe_fp8.quantize_hidden(state["x"])
    if state["op"] == "route":
        return moe_fp8.route(*state["args"])
    return moe_fp8.run(*state["args"], **state["kw"])


# ------------------------------------------------------------------------------------------ figures
def work(case):
    """Bytes and operations that the call cannot do without: inputs read once (of the weights, the
    experts that the tokens are expected to pick), outputs written once."""
    T = case["T"]
    if case["op"] == "quantize":
        return {"bytes": T * H * ((2 if case["x"] == "bf16" else 4) + 1) + T * H // BLOCK * 4, "flops": 3 * T * H}
    logits = T * E_GLOBAL * (2 if case["logits"] == "bf16" else 4) + 2 * E_GLOBAL
    if case["op"] == "route":
        return {"bytes": logits + T * TOP_K * 8, "flops": 8 * T * E_GLOBAL}
    per_token = case["local_pairs"] or E_LOCAL * TOP_K / E_GLOBAL      # pairs of a token on this rank
    active = E_LOCAL * (1.0 - (1.0 - per_token / E_LOCAL) ** T)
    weights = 3 * H * I + 3 * (H // BLOCK) * (I // BLOCK) * 4
    rows = T * (H + H // BLOCK * 4 + H * (4 if case["out"] == "f32" else 2))
    rows += T * H * {"none": 0, "bf16": 2, "f32": 4}[case["shared"]]
    return {"bytes": int(active * weights) + rows + logits, "flops": int(T * per_token * 6 * H * I)}


def tolerance(case):
    """Routing ids, codes and scales are whole values of fp32 arithmetic: equal.  The operator's sums are
    fp32 sums of exact fp8 products, with C held in 11 bits where its rows are small, rounded once."""
    if case["op"] == "quantize":
        return "exact"
    if case["op"] == "route":
        return {"rel": 1e-6, "max": 1e-5}
    if case["out"] == "f32":
        return {"rel": 1e-3, "max": 1e-2}
    return {"rel": 7e-3, "max": 2e-2}


# ------------------------------------------------------------------------------------------ oracle
def _dequant(w, s):
    return w.double() * s.double().repeat_interleave(BLOCK, 0).repeat_interleave(BLOCK, 1)


def exact(case, seed):
    state = prepare(case, seed)
    if case["op"] == "quantize":
        x = state["x"].double().view(case["T"], H // BLOCK, BLOCK)
        amax = x.abs().amax(2)
        return None, torch.where(amax > 0, amax / 448.0, torch.ones_like(amax)).t().contiguous()
    logits, bias = state["args"][:2]
    ids, s64 = _select(logits, bias)
    w = s64.gather(1, ids)
    w = w / w.sum(1, keepdim=True) * RSF
    if case["op"] == "route":
        return None, w
    hidden, hidden_scale, w13, s13, w2, s2, offset = state["args"][2:9]
    T = case["T"]
    out = torch.zeros(T, H, dtype=torch.float64, device="cuda")
    for e in range(E_LOCAL):
        t, k = torch.nonzero(ids == offset + e, as_tuple=True)
        if t.numel() == 0:
            continue
        a = hidden[t].double() * hidden_scale.t()[t].double().repeat_interleave(BLOCK, 1)
        g = a @ _dequant(w13[e], s13[e]).t().contiguous()
        c = torch.nn.functional.silu(g[:, I:]) * g[:, :I]
        out.index_add_(0, t, (c @ _dequant(w2[e], s2[e]).t().contiguous()) * w[t, k].unsqueeze(1))
    shared = state["kw"].get("shared_output")
    return out if shared is None else out + shared.double()
