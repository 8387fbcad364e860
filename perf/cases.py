"""The work a user of this framework has it do, as measurable cases: MXFP4 fused-MoE layer calls through ``fused_moe`` and
``fused_moe_routed`` over the layer shapes of ``pyhip_amd.workloads`` and over generic shapes of the same kind, from a
single decoded token to an 8192-token prefill, with even and skewed routers, biases, the clamped SwiGLU, padded
shapes, expert parallelism and both output types.

``listed()`` names the fixed cases, ``draw(rng)`` gives more of the same ranges, ``prepare`` / ``run`` / ``work`` /
``tolerance`` say what a case holds, does, needs and may differ by.
"""
import math

import torch

from pyhip_amd import fused_moe, fused_moe_routed
from pyhip_amd import workloads
from pyhip_amd.enums import ActivationType

MAX_TOKENS = 8192
# the largest listed call (256 experts, top-8, hidden 7168, intermediate 2048, 8192 tokens); a drawn case stays below it
MAX_FLOPS = 6.0 * 8192 * 8 * 7168 * 2048
MAX_WEIGHTS = 256 * 3 * 7168 * 2048


def _case(name, shape, tokens, **more):
    s = workloads.SHAPES[shape]
    c = dict(name=name, E=s["E"], k=s["k"], H=s["H"], I=s["I"], router=s["router"], bias=bool(s.get("bias")), swiglu=False,
             ranks=1, routed=False, f32=False, tokens=tokens)
    c.update(more)
    return c


def listed():
    return [
        # a small layer, a small batch: what a unit test, a toy model or a draft model calls; launches and host time
        _case("tiny_t64", "tiny", 64),
        # one user's next token in a layer of few, wide experts: the smallest decode call
        _case("mixtral_t1", "mixtral", 1),
        # a small decode batch of an odd size in the same layer: every expert is read
        _case("mixtral_t29", "mixtral", 29),
        # a decode batch of a biased layer with clamped SwiGLU whose sizes are no multiple of the tiles
        _case("gptoss_t16", "gptoss", 16, swiglu=True),
        # a decode batch under a router that loads its experts unevenly
        _case("qwen3_t64_skewed", "qwen3", 64),
        # a decode batch of a layer of many experts, router scores in: grouped sigmoid routing inside the call
        _case("dsv3_t16_routed", "dsv3", 16, routed=True),
        # a large decode batch (or a short prompt): nearly every expert is read for a few rows
        _case("dsv3_t128", "dsv3", 128),
        # one rank of an expert-parallel group of eight: 32 of 256 experts here, an odd number of gathered tokens
        _case("dsv3_ep8_t4001", "dsv3", 4001, ranks=8),
        # prefill in a layer of few experts: many rows for each
        _case("mixtral_t4096", "mixtral", 4096),
        # prefill of the biased, padded layer
        _case("gptoss_t4096", "gptoss", 4096, swiglu=True),
        # prefill under the skewed router: some experts get ten times the mean, some a handful
        _case("qwen3_t2048_skewed", "qwen3", 2048),
        # the largest prefill
        _case("dsv3_t8192", "dsv3", 8192),
    ]


def draw(rng):
    """One more case: a shape of ``workloads`` (two times in three) or a generic one, tokens spread over 1..8192 by their
    logarithm, the options mixed."""
    for _ in range(1000):
        if rng.random() < 2 / 3:
            c = _case("", rng.choice(sorted(workloads.SHAPES)), 1)
        else:
            experts = rng.choice([8, 16, 32, 60, 64, 96, 128, 160, 256])
            c = dict(E=experts, k=rng.choice([k for k in (1, 2, 4, 6, 8) if k <= experts // 4]), H=rng.randrange(32, 225) * 32,
                     I=rng.randrange(16, 113) * 32, router=rng.choice(["softmax", "softmax", "zipf"]), bias=rng.random() < 0.25,
                     ranks=1, routed=False)
        c.pop("name", None)
        c["tokens"] = int(round(math.exp(rng.uniform(0.0, math.log(MAX_TOKENS)))))
        c["swiglu"] = c["bias"] and rng.random() < 0.5
        c["f32"] = rng.random() < 0.15
        c["routed"] = c["E"] in (64, 128, 256) and c["router"] != "zipf" and c["H"] % 512 == 0 and rng.random() < 0.4
        c["ranks"] = rng.choice([2, 4, 8]) if c["E"] >= 64 and c["E"] % 8 == 0 and rng.random() < 0.2 else 1
        if c["E"] * 3 * c["H"] * c["I"] <= MAX_WEIGHTS and 6.0 * c["tokens"] * c["k"] * c["H"] * c["I"] <= MAX_FLOPS:
            return c
    raise RuntimeError("no case drawn")


def _layer(case, experts=None):
    return dict(E=experts or case["E"], k=case["k"], H=case["H"], I=case["I"], router=case["router"], bias=case["bias"])


def _logits(case, tokens, generator, device):
    return torch.randn(tokens, case["E"], generator=generator, device=device)


def prepare(case, seed):
    """The layer's weights (quantised once, as a model is when it is loaded), the hidden states N(0, 1), and the routing:
    logits N(0, 1) through the shape's router, or the logits themselves where the call routes."""
    dev = torch.device("cuda")
    local = case["E"] // case["ranks"]
    W = workloads.make_weights(_layer(case, local), dev, seed=seed)
    g = torch.Generator(device=dev).manual_seed(seed + 7919)
    hidden = torch.randn(case["tokens"], case["H"], generator=g, device=dev).to(torch.bfloat16)
    logits = _logits(case, case["tokens"], g, dev)
    opts = dict(w1_scale=W["w1_scale"], w2_scale=W["w2_scale"], bias1=W.get("bias1"), bias2=W.get("bias2"),
                activation=ActivationType.Swiglu if case["swiglu"] else ActivationType.Silu,
                dtype=torch.float32 if case["f32"] else None,
                hidden_pad=W["hidden_pad"], intermediate_pad=W["intermediate_pad"])
    if case["ranks"] > 1:
        # this rank (drawn from the seed) holds `local` consecutive experts
        mask = torch.zeros(case["E"], dtype=torch.int32, device=dev)
        r = seed % case["ranks"]
        mask[r * local:(r + 1) * local] = 1
        opts["expert_mask"] = mask
    state = dict(case=case, hidden=hidden, w1=W["w1"], w2=W["w2"], opts=opts)
    if case["routed"]:
        state["logits"] = logits
        if case["router"] == "grouped":
            opts.update(num_expert_group=8, topk_group=4)
    else:
        state["topk_w"], state["topk_ids"] = workloads.route(_layer(case), logits)
    return state


def run(state):
    if "logits" in state:
        return fused_moe_routed(state["hidden"], state["w1"], state["w2"], state["logits"], state["case"]["k"],
                                return_routing=True, **state["opts"])
    return fused_moe(state["hidden"], state["w1"], state["w2"], state["topk_w"], state["topk_ids"], **state["opts"])


def _experts_read(case):
    """Experts of this rank that at least one token picks, by routing up to 1024 tokens once (more tokens: the same share
    of never-picked experts, squared for every doubling)."""
    n = min(case["tokens"], 1024)
    g = torch.Generator().manual_seed(1)
    _, ids = workloads.route(_layer(case), _logits(case, n, g, "cpu"))
    p = torch.bincount(ids.flatten().long(), minlength=case["E"]).double() / n
    hit = (1.0 - (1.0 - p.clamp(max=1.0)) ** case["tokens"]).sum().item() if case["tokens"] > n else float((p > 0).sum())
    return hit / case["ranks"]


def work(case):
    """Every picked expert's weights and scales once (4.25 bits a value), the hidden states in, the output out, the routing;
    2 operations for each of the 3 * H * I weights of a (token, expert) pair that this rank owns."""
    T, k, H, I = case["tokens"], case["k"], case["H"], case["I"]
    pairs = T * k / case["ranks"]
    route_bytes = 4.0 * T * case["E"] + 8.0 * T * k if case["routed"] else 8.0 * T * k
    return dict(bytes=_experts_read(case) * 3.0 * H * I * (0.5 + 1.0 / 32) + 2.0 * T * H + (4.0 if case["f32"] else 2.0) * T * H + route_bytes,
                flops=6.0 * pairs * H * I)


def tolerance(case):
    """Measured against the same path with its products summed in 64 bits (the same quantisation steps, the intermediate and
    the per-slot results rounded to bf16) on 48 tokens of each listed and 14 drawn cases.  With MXFP4 activations the
    products are multiples of powers of two that 32-bit sums hold exactly: no difference.  With bf16 activations (the
    smallest calls) a few of the bf16 roundings on the way go the other way: up to 2e-4 in the 2-norm, and 7e-3 of the
    larger of the value and the root mean square (one bf16 step of a slot's value).  Four times that."""
    return {"rel": 8e-4, "max": 3e-2}


_VALUES = [0.0, 0.5, 1.0, 1.5, 2.0, 3.0, 4.0, 6.0, -0.0, -0.5, -1.0, -1.5, -2.0, -3.0, -4.0, -6.0]


def _weights64(w, scales, e):
    """Expert e's matrix [N, K] in 64 bits from the packed layout: 1 KB blocks of 16 rows x 128 values in the order
    (32-value group, row), and scale tiles of 32 rows x 8 groups in the order (group % 4, row % 16, group / 4, row / 16)."""
    N, kb = w.shape[1:]
    codes = w[e].view(N // 16, kb // 64, 4, 16, 16).permute(0, 3, 1, 2, 4).reshape(N, kb)
    codes = torch.stack([codes & 15, codes >> 4], dim=-1).reshape(N, kb // 16, 32)
    s = scales[e * N:(e + 1) * N].reshape(N // 32, -1, 4, 16, 2, 2).permute(0, 5, 3, 1, 4, 2).reshape(N, -1)[:, :kb // 16]
    table = torch.tensor(_VALUES, dtype=torch.float64, device=w.device)
    return torch.ldexp(table[codes.long()], (s.int() - 127)[..., None]).reshape(N, 2 * kb)


def _mxfp4(x):
    """x rounded to MXFP4: blocks of 32 share a power of two, 2 ** (floor(log2(largest)) - 2); ties go to even codes."""
    b = x.reshape(x.shape[0], -1, 32)
    exponent = torch.frexp(b.abs().amax(-1, keepdim=True))[1] - 3
    a = torch.ldexp(b.abs(), -exponent)
    step = torch.where(a < 2, 0.5, torch.where(a < 4, 1.0, 2.0)).double()
    return torch.ldexp((torch.round(a / step) * step).clamp(max=6.0) * torch.sign(b), exponent).reshape(x.shape)


def _bf16_activations(case):
    """The smallest calls keep the activations in bf16, all others round them to MXFP4: part of what the call computes."""
    pairs = case["tokens"] * case["k"]
    hidden = (case["H"] + 511) // 512 * 512
    few = min(pairs, case["E"]) * (hidden // 256) < 512 and pairs <= 8 * case["E"]
    return 8 * pairs <= case["E"] or few


def _routing64(case, logits):
    if case["router"] == "grouped":
        p = torch.sigmoid(logits.double())
        groups = p.view(p.shape[0], 8, -1)
        best = groups.topk(2, dim=-1).values.sum(-1).topk(4, dim=-1).indices
        keep = torch.zeros(groups.shape[:2], dtype=torch.bool, device=p.device).scatter_(1, best, True)
        p = groups.masked_fill(~keep[..., None], -1.0).view(p.shape)
    else:
        p = torch.softmax(logits.double(), dim=-1)
    w, ids = p.topk(case["k"], dim=-1)
    return w / w.sum(-1, keepdim=True), ids


def exact(case, seed):
    """The layer in 64 bits, expert by expert, with the roundings that define it: activations and intermediate to MXFP4
    (the intermediate to bf16 before) unless the call keeps them in bf16; nothing is rounded after the second product."""
    state = prepare(case, seed)
    opts, hidden, w1, w2 = state["opts"], state["hidden"], state["w1"], state["w2"]
    if "logits" in state:
        topk_w, topk_ids = _routing64(case, state["logits"])
    else:
        topk_w, topk_ids = state["topk_w"].double(), state["topk_ids"].long()
    H, inter, local = case["H"], w1.shape[1] // 2, w1.shape[0]
    quantise = (lambda v: v) if _bf16_activations(case) else _mxfp4
    x = quantise(torch.nn.functional.pad(hidden.double(), (0, w1.shape[2] * 2 - H)))
    out = torch.zeros(case["tokens"], H, dtype=torch.float64, device=x.device)
    first = int(opts["expert_mask"].argmax()) if "expert_mask" in opts else 0
    for e in range(local):
        tok, slot = torch.nonzero(topk_ids == first + e, as_tuple=True)
        if not len(tok):
            continue
        y = x[tok] @ _weights64(w1, opts["w1_scale"], e).T
        if case["bias"]:
            y = y + opts["bias1"][e].double()
        gate, up = y[:, :inter], y[:, inter:]
        if case["swiglu"]:
            gate, up = gate.clamp(max=7.0), up.clamp(-7.0, 7.0) + 1.0
            a = gate * torch.sigmoid(1.702 * gate) * up
        else:
            a = gate * torch.sigmoid(gate) * up
        z = quantise(a.to(torch.bfloat16).double()) @ _weights64(w2, opts["w2_scale"], e).T
        if case["bias"]:
            z = z + opts["bias2"][e].double()
        out.index_add_(0, tok, z[:, :H] * topk_w[tok, slot, None])
    return (out, topk_w, topk_ids.int()) if "logits" in state else out
