"""Performance cases of the routed-expert path: the calls that an FFN rank of an
attention-FFN disaggregated MoE deployment serves, from a decode step of a few tokens to a
whole prefill dispatch, and the attention rank's combine.

``listed`` are fixed calls, ``draw`` gives more of the same ranges, ``prepare`` makes what a
serving program holds before the call (packed weights, the layer object, the tokens and their
routing), ``run`` is one pass through the public entry points, ``exact`` the same result in 64
bits by plain torch.

A case is a dict of plain values:

* ``kind``: "layer" (``AfdExperts.forward``), "wire" (``AfdExperts.forward_q`` on rows the
  attention rank quantized), "batch" (``AfdExperts.forward_batch``), "graph"
  (``FfnGraphRunner.run``, the HIP-graph replay of the token bucket), "combine"
  (``combine_parts``, the attention rank's sum over the FFN ranks plus its shared expert);
* ``hidden``, ``inter``, ``experts`` (global), ``local`` (this rank owns [0, local)), ``topk``;
* ``fmt`` "mxfp4" or "fp8_block", ``act`` "fp8" (the weight format's fp8 activations) or "bf16",
  ``activation`` "silu", "silu_limit" or "situ", ``walk`` the GEMMs' tile walk;
* ``tokens``, ``zipf`` (expert popularity, 0 for uniform), ``jobs`` (batch), ``parts`` (combine).
"""

from __future__ import annotations

import math
import os
import random
import sys

import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "sgl-afd-plugin_amd"))

from sgl_asap_amd.moe.dispatcher import combine_parts  # noqa: E402
from sgl_asap_amd.moe.experts import AfdExperts, pack_fp8_block_experts, pack_mxfp4_experts  # noqa: E402
from sgl_asap_amd.moe.topk import StandardTopKOutput  # noqa: E402
from sgl_asap_amd.runner.graph_runner import FfnGraphRunner  # noqa: E402

SWIGLU_LIMIT = 10.0  # the clamp of the limited SwiGLU
SITU_BETA, SITU_LINEAR_BETA = 4.0, 25.0

# one FFN rank of a DeepSeek-V4-Flash-style model (MXFP4 experts), of four
RANK = dict(hidden=4096, inter=2048, experts=256, local=64, topk=8, fmt="mxfp4")
# an ERNIE-5.5-Flash-style model's experts on one rank (FP8 128x128 blocks)
ERNIE = dict(hidden=4096, inter=1536, experts=64, local=64, topk=8, fmt="fp8_block")
# a smaller generic model, experts over four ranks
SMALL = dict(hidden=2048, inter=1024, experts=128, local=32, topk=4)


def _case(name, shape, tokens, **more):
    case = dict(kind="layer", act="fp8", activation="silu", walk="static", zipf=0.0)
    case.update(shape, tokens=tokens, **more)
    if name:
        case["name"] = name
    return case


def listed():
    return [
        # a decode step of a small batch, called on its own: a handful of experts, one row each
        _case("mx_decode_8", RANK, 8, activation="silu_limit"),
        # a decode step replayed from the token bucket's graph, as the FFN scheduler's graph
        # mode serves it (dynamic walk, skewed routing)
        _case("mx_graph_48", RANK, 48, kind="graph", walk="dynamic", zipf=1.2),
        # a larger decode dispatch whose rows came quantized over the wire
        _case("mx_wire_300", RANK, 300, kind="wire", walk="dynamic", zipf=1.2),
        # four pending jobs of two replicas' micro-batches served in one call
        _case("mx_batch_2900", RANK, 2900, kind="batch", jobs=4, walk="dynamic", zipf=1.2),
        # one micro-batch of a two-batch-overlap prefill
        _case("mx_prefill_8192", RANK, 8192, walk="dynamic", zipf=1.2),
        # the whole prefill dispatch of one attention replica (the benchmark's workload)
        _case("mx_prefill_16384", RANK, 16384),
        # the same dispatch with bf16 activations (W4A16)
        _case("mx_a16_16384", RANK, 16384, act="bf16"),
        # decode on FP8-block experts, every expert local
        _case("fp8_decode_24", ERNIE, 24, zipf=1.1),
        # a chunk of a prompt with ERNIE's own activation, an odd number of tokens
        _case("fp8_situ_1531", ERNIE, 1531, activation="situ", zipf=1.1, walk="dynamic"),
        # the whole prefill dispatch on FP8-block experts
        _case("fp8_prefill_16384", ERNIE, 16384, zipf=1.1),
        # bf16 activations on FP8-block experts (W8A16), a mixed prefill and decode batch
        _case("fp8_a16_517", ERNIE, 517, act="bf16", zipf=1.1),
        # the attention rank's combine of four FFN ranks' partial sums and the shared expert
        dict(name="combine_8192", kind="combine", hidden=4096, tokens=8192, parts=4),
    ]


def draw(rng):
    kind = rng.choice(["layer", "layer", "layer", "wire", "batch", "graph", "combine"])
    if kind == "combine":
        return dict(kind="combine", hidden=rng.choice([2048, 4096]), tokens=_log(rng, 16, 16384), parts=rng.randint(1, 4))
    shape = rng.choice([RANK, RANK, ERNIE, ERNIE, dict(SMALL, fmt="mxfp4"), dict(SMALL, fmt="fp8_block")])
    act = "fp8" if kind == "wire" else rng.choice(["fp8", "fp8", "bf16"])
    top = 256 if kind == "graph" else 8192 if act == "bf16" and shape["fmt"] == "fp8_block" else 16384
    case = _case(None, shape, _log(rng, 4, top), kind=kind, act=act,
                 activation=rng.choice(["silu", "silu", "silu_limit", "situ"]),
                 walk=rng.choice(["static", "dynamic"]), zipf=rng.choice([0.0, 1.1, 1.2]))
    if kind == "batch":
        case["jobs"] = rng.randint(2, 8)
        case["tokens"] = max(case["tokens"], 8)
    return case


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


# ---------------------------------------------------------------- inputs
def _routing(case, seed):
    """(ids int32 [n, k], w f32 [n, k]) on the CPU. The experts' popularity belongs to the
    model, so it is the same for every seed."""
    n, experts, k = case["tokens"], case["experts"], case["topk"]
    gen = torch.Generator().manual_seed(seed)
    logits = torch.randn(n, experts, generator=gen)
    if case["zipf"]:
        ranks = torch.randperm(experts, generator=torch.Generator().manual_seed(experts)).float() + 1.0
        u = torch.rand(n, experts, generator=gen).clamp_min(1e-20)
        _, ids = torch.topk(-case["zipf"] * ranks.log() - torch.log(-torch.log(u)), k, dim=-1)
        w = torch.softmax(logits.gather(1, ids), dim=-1)
    else:
        w, ids = torch.topk(torch.softmax(logits, dim=-1), k, dim=-1)
        w = w / w.sum(dim=-1, keepdim=True)
    return ids.to(torch.int32), w.float()


def _tensors(case, seed):
    """Tokens x ~ N(0, 1) in bf16 and logical expert weights ~ N(0, 0.02) in fp32, on the GPU."""
    gen = torch.Generator(device="cuda").manual_seed(seed)
    e, h, i = case["local"], case["hidden"], case["inter"]
    x = torch.randn(case["tokens"], h, generator=gen, device="cuda").to(torch.bfloat16)
    w13 = torch.randn(e, 2 * i, h, generator=gen, device="cuda").mul_(0.02)
    w2 = torch.randn(e, h, i, generator=gen, device="cuda").mul_(0.02)
    return x, w13, w2


def _job_sizes(case):
    """Sizes of a batch's jobs (uneven, each at least one token), adding up to its tokens."""
    rng = random.Random(case["tokens"])
    cuts = sorted(rng.sample(range(1, case["tokens"]), case["jobs"] - 1))
    return [b - a for a, b in zip([0] + cuts, cuts + [case["tokens"]])]


def _combine_inputs(case, seed):
    gen = torch.Generator(device="cuda").manual_seed(seed)
    return [torch.randn(case["tokens"], case["hidden"], generator=gen, device="cuda").mul_(0.3).to(torch.bfloat16)
            for _ in range(case["parts"] + 1)]


def prepare(case, seed):
    if case["kind"] == "combine":
        *parts, shared = _combine_inputs(case, seed)
        return dict(case=case, parts=parts, ptrs=[t.data_ptr() for t in parts], shared=shared)
    x, w13, w2 = _tensors(case, seed)
    pack = pack_mxfp4_experts if case["fmt"] == "mxfp4" else pack_fp8_block_experts
    activation, alpha, limit = {"silu": ("silu", None, None), "silu_limit": ("silu", None, SWIGLU_LIMIT),
                                "situ": ("situ", SITU_BETA, SITU_LINEAR_BETA)}[case["activation"]]
    layer = AfdExperts(case["experts"], case["topk"], 0, range(case["local"]), pack(w13, w2),
                       n_max=case["tokens"], activation=activation, gemm1_alpha=alpha, gemm1_clamp_limit=limit,
                       tile_walk=case["walk"], act_format="bf16" if case["act"] == "bf16" else None)
    del w13, w2
    ids, w = (t.cuda() for t in _routing(case, seed))
    state = dict(case=case, layer=layer, x=x, topk=StandardTopKOutput(w, ids))
    if case["kind"] == "wire":
        state["xq"], state["xs"] = layer.quant_act(x)
    elif case["kind"] == "batch":
        state["jobs"], at = [], 0
        for n in _job_sizes(case):
            rows = slice(at, at + n)
            state["jobs"].append((x[rows].clone(), StandardTopKOutput(w[rows].clone(), ids[rows].clone())))
            at += n
    elif case["kind"] == "graph":
        state["runner"] = FfnGraphRunner({0: layer}, case["tokens"], layer.local)
    return state


def run(state):
    kind = state["case"]["kind"]
    if kind == "combine":
        n, h = state["shared"].shape
        return combine_parts(state["ptrs"], state["shared"], n, h, state["shared"].device)
    if kind == "wire":
        return state["layer"].forward_q(state["xq"], state["xs"], state["topk"])
    if kind == "batch":
        return state["layer"].forward_batch(state["jobs"])
    if kind == "graph":
        return state["runner"].run(0, state["x"], state["topk"].topk_ids, state["topk"].topk_weights)
    return state["layer"](state["x"], state["topk"])


# ---------------------------------------------------------------- what a pass needs
def work(case):
    n, h = case["tokens"], case["hidden"]
    if case["kind"] == "combine":
        return {"bytes": (case["parts"] + 2) * n * h * 2, "flops": case["parts"] * n * h}
    ids, _ = _routing(case, 0)
    mine = ids[ids < case["local"]]
    weight = 17 / 32 if case["fmt"] == "mxfp4" else 1.0 + 4 / 128**2
    x_bytes = h * 2 if case["kind"] != "wire" else h + h // 32 if case["fmt"] == "mxfp4" else h + h // 32
    used = int(torch.unique(mine).numel()) * 3 * h * case["inter"] * weight
    return {"bytes": int(used + n * (x_bytes + h * 2 + case["topk"] * 8)),
            "flops": 6 * h * case["inter"] * int(mine.numel())}


def tolerance(case):
    # The results are bf16, each the sum of up to topk bf16 rows: 2.3e-3 to 2.6e-3 from 64 bits
    # at every listed case. With fp8 activations a value of h near a rounding tie may also take
    # the neighbouring code (1/16 apart) under another order of the sums.
    return {"rel": 0.01}


# ---------------------------------------------------------------- the result in 64 bits
def _e4m3(v):
    return v.clamp(-448.0, 448.0).to(torch.float32).to(torch.float8_e4m3fn).to(v.dtype)


def _mx_scale(blocks, emax):
    """2^(floor(log2(amax)) - emax) per block of 32 (smallest where the block is zero)."""
    amax = blocks.abs().amax(-1, keepdim=True)
    exponent = (torch.frexp(amax).exponent - 1 - emax).clamp(-127, 127)
    return torch.where(amax > 0, torch.ldexp(torch.ones_like(amax), exponent), torch.full_like(amax, 2.0**-127))


def _scale_448(amax):
    """max(amax, 1e-10) / 448 as the IEEE fp32 quotient (by a tensor: torch multiplies by the
    reciprocal of a scalar divisor)."""
    return amax.clamp_min(1e-10) / torch.full_like(amax, 448.0)


def _quant_act(v, act):
    """v [n, K] (fp64) as the GEMMs read it."""
    if act == "bf16":
        return v.to(torch.bfloat16).double()
    if act == "mxfp4":  # MXFP8: e4m3 with a power-of-two scale per 32
        b = v.reshape(v.shape[0], -1, 32)
        s = _mx_scale(b, 8)
        return (_e4m3(b / s) * s).reshape(v.shape)
    # e4m3 with one fp32 scale per 128: the codes are those of the fp32 quotient (bf16 values
    # meet ties of the exact quotient often)
    b = v.float().reshape(v.shape[0], -1, 128)
    s = _scale_448(b.abs().amax(-1, keepdim=True))
    return (_e4m3(b / s).double() * s.double()).reshape(v.shape)


def _quant_weight(w, fmt):
    """One expert's logical weight [N, K] (fp32) as its format holds it, in fp64."""
    n, k = w.shape
    if fmt == "mxfp4":
        b = w.reshape(n, k // 32, 32)
        s = _mx_scale(b, 2)
        v = b / s
        a = v.abs()
        q = 0.5 * ((a > 0.25).double() + (a >= 0.75).double() + (a > 1.25).double() + (a >= 1.75).double())
        q += (a > 2.5).double() + (a >= 3.5).double() + 2.0 * (a > 5.0).double()
        return (torch.copysign(q, v.double()) * s.double()).reshape(n, k)
    b = w.reshape(n // 128, 128, k // 128, 128)
    s = _scale_448(b.abs().amax((1, 3), keepdim=True))
    return (_e4m3(b / s).double() * s.double()).reshape(n, k)


def _activation(g, u, name):
    if name == "silu_limit":
        g, u = g.clamp(max=SWIGLU_LIMIT), u.clamp(-SWIGLU_LIMIT, SWIGLU_LIMIT)
    if name == "situ":
        return (SITU_LINEAR_BETA * torch.tanh(u / SITU_LINEAR_BETA)) * (SITU_BETA * torch.tanh(g / SITU_BETA)) \
            * torch.sigmoid(g)
    return g * torch.sigmoid(g) * u


def exact(case, seed):
    if case["kind"] == "combine":
        return sum(t.double() for t in _combine_inputs(case, seed))
    x, w13, w2 = _tensors(case, seed)
    ids, w = (t.cuda() for t in _routing(case, seed))
    act = "bf16" if case["act"] == "bf16" else case["fmt"]
    xq = _quant_act(x.double(), act)
    out = torch.zeros(x.shape, dtype=torch.float64, device=x.device)
    for e in range(case["local"]):
        tok, slot = torch.nonzero(ids == e, as_tuple=True)
        if not tok.numel():
            continue
        gu = xq[tok] @ _quant_weight(w13[e], case["fmt"]).t()
        g, u = gu.chunk(2, dim=-1)
        h = _quant_act(_activation(g, u, case["activation"]), act)
        y = h @ _quant_weight(w2[e], case["fmt"]).t()
        out.index_add_(0, tok, y * w[tok, slot].double()[:, None])
    if case["kind"] == "batch":
        return list(out.split(_job_sizes(case)))
    return out
