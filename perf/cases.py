"""The work whose speed counts: what a user of this framework has it do, over the range they do it in.

A case is one forward pass of an MoE layer (`MoeLayer.run`) or of a stack of pre-norm residual blocks
(`MoeChain.step`) on resident weights: decode steps of one and a few tokens, small batches, prefill.
Shapes are those of deepstrix_amd/workloads.py and those the library's path thresholds were set on
(deepstrix_amd/csrc/dsx_layer.inc); weights, activations and router logits follow their distributions.

Keys of a case
  shape    a name of SHAPES
  tokens   tokens of one pass
  planar   the MXFP4 tensors in the library's planar form instead of the engine's rows
  shared   the shared expert's format: "same" (as the routed experts) or "q8_0" (the engine's own mix)
  routing  "normal": N(0, 1) logits; "zipf": logits skewed so that a tenth of the experts gets about
           half of the picks; "uniform": the caller pins uniform random picks; "same": it pins the same
           experts for every token
  blocks   0: one layer on given logits; n: n chained blocks (RMSNorm, router, layer, residual)
"""
import math
from dataclasses import replace

import torch

from deepstrix_amd import synth, workloads
from deepstrix_amd.capi import FMT_MXFP4, FMT_Q8_0
from deepstrix_amd.executor import MoeChain, MoeLayer

SHAPES = {
    # DeepSeek-V3: 256 experts, top-8 of 4 of 8 groups, sigmoid gating with bias; MXFP4
    "v3": workloads.CFG2,
    # the same widths, gate/up in MXFP4 and down in Q8_0
    "v3-mixed": workloads.CFG5,
    # middle-sized and small all-MXFP4 layers; the reference's own router (sqrt-softplus) and clamp
    "mid": workloads.Shape(4096, 1024, 128, 8, router_mode=0, route_scale=1.5, clamp=10.0, bias_sigma=0.01, seed=0xD5EE0011),
    "small": workloads.Shape(2048, 1536, 64, 6, router_mode=0, route_scale=1.5, clamp=10.0, bias_sigma=0.01, seed=0xD5EE0012),
    # all-Q8_0: hidden 2048, 64 experts of 1408, top-6 softmax
    "q8_0": workloads.CFG1,
}
ZIPF_ALPHA = 0.416   # factor on the -1.1 ln(rank) shift: the top tenth of 256 experts then has half of the picks


def _case(shape, tokens, planar=False, shared="same", routing="normal", blocks=0, name=None):
    c = {"shape": shape, "tokens": tokens, "planar": planar, "shared": shared, "routing": routing, "blocks": blocks}
    return dict(c, name=name) if name else c


def listed():
    return [
        _case("v3", 1, name="decode 1"),                                   # one user's next token
        _case("v3", 3, shared="q8_0", name="decode 3, q8_0 shared"),       # speculative verify on the engine's own mix of formats
        _case("v3", 2, blocks=4, name="4 blocks, decode 2"),               # the same through a stack, router included
        _case("v3", 16, name="batch 16"),                                  # a few users' tokens
        _case("v3", 64, name="batch 64"),                                  # continuous batching
        _case("mid", 37, name="middle layer, batch 37"),                   # ragged batch on a smaller layer
        _case("v3", 200, planar=True, name="planar, batch 200"),           # a large decode batch or a short prompt
        _case("v3", 777, planar=True, routing="zipf", name="planar, prefill 777"),   # a prompt, skewed experts
        _case("v3", 4096, routing="zipf", name="prefill 4096"),            # a full prefill chunk on the engine's rows
        _case("v3-mixed", 512, routing="uniform", name="mixed, prefill 512"),        # MXFP4 gate/up with Q8_0 down
        _case("q8_0", 4, name="q8_0, decode 4"),                           # the small Q8_0 layer: launches and latency count
        _case("q8_0", 512, name="q8_0, prefill 512"),
    ]


def draw(rng):
    """One more case of the same ranges: token counts spread over their logarithm, odd ones included."""
    def tokens(lo, hi):
        return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi + 0.5)))))))

    kind = rng.choice(["v3", "v3", "v3", "v3", "shared", "chain", "mid", "small", "mixed", "q8_0", "q8_0"])
    planar = rng.random() < 0.35
    if kind == "v3":
        return _case("v3", tokens(1, 3000), planar, routing=rng.choice(["normal", "normal", "zipf"]))
    if kind == "shared":
        return _case("v3", tokens(1, 1000), planar, shared="q8_0")
    if kind == "chain":
        return _case(rng.choice(["v3", "mid", "small"]), tokens(1, 24), planar, blocks=rng.randint(2, 4))
    if kind == "mixed":
        return _case("v3-mixed", tokens(1, 1000), planar, routing=rng.choice(["normal", "uniform", "same"]))
    if kind == "q8_0":
        return _case("q8_0", tokens(1, 2048))
    return _case(kind, tokens(1, 2048), planar, routing=rng.choice(["normal", "zipf"]))


def _shape(case):
    s = SHAPES[case["shape"]]
    return replace(s, sh_gate_fmt=FMT_Q8_0, sh_down_fmt=FMT_Q8_0) if case["shared"] == "q8_0" else s


def prepare(case, seed):
    """Weights, layer handle and workspace, and the pass's inputs, all on the GPU."""
    s, T = replace(_shape(case), seed=0xD5EE0000 + seed * 64), case["tokens"]
    x = synth.normal_dev(s.seed, synth.T_X, T * s.hidden).view(T, s.hidden)
    x = x.bfloat16().float()   # bf16 activations, handed over as f32
    if case["blocks"]:
        weights = [workloads.device_weights(replace(s, seed=s.seed + 1 + i), block=True, planar=case["planar"])
                   for i in range(case["blocks"])]
        for w in weights:
            w.router_w = w.router_w.view(s.n_expert, s.hidden)
        return {"chain": MoeChain(weights, T), "x": x, "h": torch.empty_like(x)}
    state = {"layer": MoeLayer(workloads.device_weights(s, planar=case["planar"]), T), "x": x, "out": torch.empty_like(x),
             "logits": None, "picks": None, "pick_weights": None}
    if case["routing"] in ("normal", "zipf"):
        lg = synth.normal_dev(s.seed, synth.T_LOGITS, T * s.n_expert).view(T, s.n_expert)
        if case["routing"] == "zipf":
            lg = lg + ZIPF_ALPHA * torch.from_numpy(workloads.zipf_logit_shift(s.n_expert, seed)).cuda()
        state["logits"] = lg
    else:
        g = torch.Generator(device="cuda").manual_seed(seed)
        rank = torch.rand((T, s.n_expert), generator=g, device="cuda")
        if case["routing"] == "same":
            rank = rank[:1].expand(T, -1)
        state["picks"] = rank.argsort(dim=1)[:, :s.n_used].to(torch.int32).contiguous()
        state["pick_weights"] = torch.rand((T, s.n_used), generator=g, device="cuda") * 0.55 + 0.05
    return state


def run(state):
    if "chain" in state:
        state["h"].copy_(state["x"])
        return state["chain"].step(state["h"])
    return state["layer"].run(state["x"], state["logits"], out=state["out"], selected_in=state["picks"],
                              weights_in=state["pick_weights"])


def work(case):
    """Every expert that some token names read once (their expected number where the routing is random),
    the shared expert, the router matrix of a block, activations and logits in, results out; the
    products' multiplications and additions."""
    s, T, n = _shape(case), case["tokens"], max(1, case["blocks"])

    def expert(gate_fmt, down_fmt, inter):
        per = {FMT_MXFP4: 17.0 / 32.0, FMT_Q8_0: 34.0 / 32.0}
        return s.hidden * inter * (2 * per[gate_fmt] + per[down_fmt])

    distinct = s.n_used if case["routing"] == "same" else s.n_expert * (1.0 - (1.0 - s.n_used / s.n_expert) ** T)
    weights = distinct * expert(s.gate_fmt, s.down_fmt, s.inter) + expert(s.shg, s.shd, s.shi)
    if case["blocks"]:
        weights += 4.0 * s.n_expert * s.hidden
        flops = 2.0 * T * s.n_expert * s.hidden
    else:
        flops = 0.0
    flops += 6.0 * T * s.hidden * (s.n_used * s.inter + s.shi)
    routing = 0 if case["blocks"] else 8 * s.n_used if case["routing"] in ("uniform", "same") else 4 * s.n_expert
    return {"bytes": n * weights + 8.0 * T * s.hidden + T * routing, "flops": n * flops}


def tolerance(case):
    """About four times what the library's own paths differ by (one-launch decode, one launch per stage,
    by-expert kernels, grouped GEMMs of either tile: other orders of the same f32 sums).  The sums differ
    by about 1e-7; through them a few intermediate values round to the neighbouring int8 step before the
    down product: 1.1e-4 in the 2-norm and 5e-3 in a single value for one layer.  In a stack the next
    block's activations are rounded to int8 again, and such steps multiply: 7.3e-3 and 0.041 were seen
    over four blocks."""
    return {"rel": 0.028, "max": 0.17} if case["blocks"] else {"rel": 4e-4, "max": 0.02}
