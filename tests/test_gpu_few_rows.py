"""GPU: the few-rows GEMMs (calls with few tokens per expert), every weight and activation
format, at the sizes where they can go wrong: expert counts around the 32-row blocks, the
32- and 64-row groups and the row tiles (128, or 256 for FP8 block weights with fp8 activations), experts
with no row, one K stage and K stages that do not fill the register ring, one and several weight
image columns, and an expert count that is not a multiple of the 4 a lane looks up.

Above that, up to GATED tokens per local expert on a rank with a quarter of the experts, an MXFP4
call launches both the few-rows and the large-tile GEMMs and the number of local pairs decides on
the GPU; both outcomes are run. So does any call above 2560 pairs, by how the pairs are spread.

The large-tile GEMMs and the few-rows GEMMs feed every accumulator the same products in the
same order, so the same tokens inside a call large enough for the large tiles must give the
same bits; against the oracle the bar is that of the other layer tests (rel-L2 1e-2: the same
quantizers at the same points, another order of the fp32 sums)."""

import numpy as np
import pytest
import torch

from gpu_util import bits16, dev, rel_l2, say
from oracle import experts as OX
from oracle import formats as F
from sgl_asap_amd import workloads as W
from sgl_asap_amd.moe.experts import (AfdExperts, new_job_desc, pack_fp8_block_experts, pack_mxfp4_experts,
                                      set_job)
from sgl_asap_amd.moe.topk import StandardTopKOutput
from test_gpu_moe import deq_weights

pytestmark = pytest.mark.gpu

REL_L2_TOL = 1e-2
# rows of the first experts; the others get none
COUNTS = [1, 0, 31, 32, 33, 63, 64, 65, 127, 128, 129, 0, 2, 255, 256, 257, 7]
# tokens per local expert (topk 1 here) up to which a call takes the few-rows GEMMs, and up to which
# the number of local pairs decides
FEW_ROWS = 40
GATED = 140


def ids_for(counts, num_local, total, gen):
    """total tokens, top-1: counts[e] of them on expert e, the others on no local expert, in
    random order."""
    ids = torch.full((total,), num_local, dtype=torch.int32)
    at = 0
    for e, c in enumerate(counts):
        ids[at:at + c] = e
        at += c
    return ids[torch.randperm(total, generator=gen)][:, None].contiguous()


@pytest.mark.parametrize("act", ["fp8", "bf16"])
@pytest.mark.parametrize("fmt", ["mxfp4", "fp8_block"])
@pytest.mark.parametrize(
    "num_local,hidden,inter,activation",
    [
        # groups of 64 rows
        (42, 256, 128, "silu"),  # 2 and 1 K stages, one image column in each GEMM
        (42, 768, 384, "silu_limit"),  # 6 and 3 K stages, 3 columns
        (42, 1280, 1152, "situ"),  # 10 and 9 K stages
        # groups of 32 rows (the n + 300 tokens below: of 64)
        (101, 256, 128, "situ"),
        (101, 512, 384, "silu"),
    ],
)
def test_few_rows_match_large_tiles(num_local, hidden, inter, activation, fmt, act):
    n, more = sum(COUNTS) + 5, GATED * num_local + 1
    assert n <= FEW_ROWS * num_local < 3000 + n <= GATED * num_local
    say(f"few rows E={num_local} H={hidden} I={inter} {activation} {fmt} {act} n={n}")
    gen = W.generator("cpu", 17)
    x = W.tokens(n + more, hidden, gen, "cpu")
    w = torch.rand(n + more, 1, generator=gen) + 0.25
    ids = torch.cat([ids_for(COUNTS, num_local, n, gen),
                     torch.randint(0, num_local, (more, 1), generator=gen, dtype=torch.int32)])
    ids[n:n + 300] = num_local
    w13, w2 = W.expert_weights(num_local, hidden, inter, gen, "cpu")
    pack = pack_mxfp4_experts if fmt == "mxfp4" else pack_fp8_block_experts
    kw, oact = {}, {}
    if activation == "situ":
        kw = dict(activation="situ", gemm1_alpha=2.0, gemm1_clamp_limit=3.0)
        oact = dict(activation="situ", act_alpha=2.0, act_limit=3.0)
    elif activation == "silu_limit":
        kw, oact = dict(swiglu_limit=0.5), dict(activation="swiglu_limit", act_limit=0.5)
    # a rank with a quarter of the experts: more tokens launch both forms
    experts = AfdExperts(4 * num_local, 1, 0, range(num_local), pack(w13, w2, device=dev()), n_max=n + more,
                         act_format="bf16" if act == "bf16" else None, **kw)

    def call(m):
        out = experts(x[:m].to(dev()), StandardTopKOutput(w[:m].to(dev()), ids[:m].to(dev())))
        torch.cuda.synchronize()
        return bits16(out)

    few = call(n)
    # a few more tokens without a local expert (42 experts: the local pairs decide), more local pairs
    # (the large tiles, by the same decision), and beyond its range
    for m in (n + 300, 3000 + n, n + more):
        assert np.array_equal(few, call(m)[:n]), m
    quant = "bf16" if act == "bf16" else "mxfp8" if fmt == "mxfp4" else "fp8_1x128"
    ref = OX.moe_ffn(x[:n], ids[:n].numpy(), w[:n].numpy(), *deq_weights(w13, w2, fmt), 0, act=quant, **oact)
    err = rel_l2(F.bf16_to_f32(few), F.bf16_to_f32(ref))
    say(f"rel_l2={err:.3e}")
    assert err <= REL_L2_TOL, err
    # one token on one expert, alone and on the last expert
    for e in (0, num_local - 1):
        ids[:1] = e
        assert np.array_equal(call(1), call(n + more)[:1]), e


@pytest.mark.parametrize("act", ["fp8", "bf16"])
@pytest.mark.parametrize("fmt", ["mxfp4", "fp8_block"])
@pytest.mark.parametrize("num_local,counts", [(42, {40: 1601}), (101, {0: 65, 3: 32, 100: 1500})])
def test_concentrated_rows_match_large_tiles(num_local, counts, fmt, act):
    """One expert with most of a few-rows call's pairs: 26 groups of 64 rows (47 of 32 with 101
    experts), which read its weights through the cache while an expert of one group streams past
    it; the same bits as inside a call of the large tiles."""
    n, more = sum(counts.values()), GATED * num_local + 1
    assert n <= FEW_ROWS * num_local
    say(f"concentrated E={num_local} {fmt} {act} counts={counts}")
    gen = W.generator("cpu", 23)
    x = W.tokens(n + more, 512, gen, "cpu")
    w = torch.rand(n + more, 1, generator=gen) + 0.25
    ids = torch.cat([ids_for([counts.get(e, 0) for e in range(num_local)], num_local, n, gen),
                     torch.randint(0, num_local, (more, 1), generator=gen, dtype=torch.int32)])
    w13, w2 = W.expert_weights(num_local, 512, 384, gen, "cpu")
    pack = pack_mxfp4_experts if fmt == "mxfp4" else pack_fp8_block_experts
    experts = AfdExperts(num_local + 1, 1, 0, range(num_local), pack(w13, w2, device=dev()), n_max=n + more,
                         act_format="bf16" if act == "bf16" else None)

    def call(m):
        out = experts(x[:m].to(dev()), StandardTopKOutput(w[:m].to(dev()), ids[:m].to(dev())))
        torch.cuda.synchronize()
        return bits16(out)

    few = call(n)
    assert np.isfinite(F.bf16_to_f32(few)).all()
    assert np.array_equal(few, call(n + more)[:n])


# Above 2560 pairs (2048 in groups of 32 rows), if some routing could call for the large tiles, a call
# launches both forms and the router writes its
# choice: few rows if gate_up's row groups make at most two rounds of workgroups (1024 / image columns
# groups of 64 rows, 1536 / columns of 32), or there are at most 3/2 groups per expert with rows.
def spread(experts, rows, last):
    """``experts`` experts of ``rows`` rows, one more of ``last`` if any."""
    return [rows] * experts + ([last] if last else [])


# num_local, hidden, inter, counts, the router's choice (n: the counts' sum, at least 2700)
EDGES = [
    # 16 image columns of gate_up, 80 experts: groups of 64 rows, 64 of them make two rounds
    (80, 256, 2048, spread(20, 140, 64 * 4), 1),  # 64 groups on 21 experts
    (80, 256, 2048, spread(20, 140, 64 * 4 + 1), 0),  # 65
    (80, 256, 2048, spread(25, 65, 0) + spread(25, 50, 0), 1),  # 75 on 50: 3/2
    (80, 256, 2048, spread(26, 65, 0) + spread(24, 50, 0), 0),  # 76 on 50
    # 256 experts: groups of 32 rows, 96 of them make two rounds
    (256, 256, 2048, spread(31, 65, 65), 1),  # 96 groups on 32 experts
    (256, 256, 2048, spread(31, 65, 97), 0),  # 97
    (256, 256, 2048, spread(80, 33, 0) + spread(80, 1, 0), 1),  # 240 on 160: 3/2
    (256, 256, 2048, spread(81, 33, 0) + spread(79, 1, 0), 0),  # 241 on 160
    # one column: no routing makes two rounds, so the few rows run alone (no choice written); all rows
    # on the last expert
    (256, 256, 128, [0] * 255 + [4000], -1),
]


def counted(counts, num_local, total):
    return (list(counts) + [0] * num_local)[:num_local], max(total, sum(counts))


@pytest.mark.parametrize("act", ["fp8", "bf16"])
@pytest.mark.parametrize("fmt", ["mxfp4", "fp8_block"])
@pytest.mark.parametrize("edge", range(len(EDGES)))
def test_router_chooses_at_the_edge(edge, fmt, act):
    """Either choice gives the bits of the large tiles, on a poisoned workspace, from bf16 and
    quantized rows, in a batch and from a descriptor with room for more tokens."""
    num_local, hidden, inter, counts, want = EDGES[edge]
    counts, n = counted(counts, num_local, 2700)
    assert FEW_ROWS * num_local >= n > 2560
    say(f"edge E={num_local} H={hidden} I={inter} {fmt} {act} n={n} want={want}")
    more = GATED * num_local + 1
    gen = W.generator("cpu", 31 + edge)
    x = W.tokens(n + more, hidden, gen, "cpu").to(dev())
    w = (torch.rand(n + more, 1, generator=gen) + 0.25).to(dev())
    ids = torch.cat([ids_for(counts, num_local, n, gen),
                     torch.randint(0, num_local, (more, 1), generator=gen, dtype=torch.int32)]).to(dev())
    gpu = torch.Generator(device=dev()).manual_seed(7)
    w13 = torch.randn(num_local, 2 * inter, hidden, generator=gpu, device=dev()) * 0.05
    w2 = torch.randn(num_local, hidden, inter, generator=gpu, device=dev()) * 0.05
    pack = pack_mxfp4_experts if fmt == "mxfp4" else pack_fp8_block_experts
    experts = AfdExperts(num_local + 1, 1, 0, range(num_local), pack(w13, w2), n_max=n + more,
                         act_format="bf16" if act == "bf16" else None)

    def topk(a, b):
        return StandardTopKOutput(w[a:b].contiguous(), ids[a:b].contiguous())

    def poisoned():
        experts.workspace().fill_(0xFF)
        out = torch.empty(n, hidden, dtype=torch.bfloat16, device=dev())
        out.view(torch.int16).fill_(-1)
        return out

    def chosen():
        return int(experts.ws_view("num_tiles", torch.int32, 2, n)[1])

    ref = bits16(experts(x, topk(0, n + more)))[:n]  # the large tiles
    assert np.isfinite(F.bf16_to_f32(ref)).all()
    got = bits16(experts(x[:n].contiguous(), topk(0, n), out=poisoned()))
    assert chosen() == want
    assert np.array_equal(got, ref)
    if act == "fp8":
        xq, xs = experts.quant_act(x[:n].contiguous())
        got = bits16(experts.forward_q(xq, xs, topk(0, n), out=poisoned()))
        assert chosen() == want
        assert np.array_equal(got, ref)
    cut, out = n // 3, poisoned()
    experts.forward_batch([(x[:cut].contiguous(), topk(0, cut)), (x[cut:n].contiguous(), topk(cut, n))],
                          outs=[out[:cut], out[cut:]])
    torch.cuda.synchronize()
    assert chosen() == want
    assert np.array_equal(bits16(out), ref)
    if n + 8 <= FEW_ROWS * num_local:  # room for more tokens, in the same form
        desc, out, job = new_job_desc(dev()), poisoned(), topk(0, n)
        set_job(desc, ids=job.topk_ids, w=job.topk_weights, out=out, x=x[:n].contiguous())
        experts.call_job(desc, n + 8)
        torch.cuda.synchronize()
        assert int(experts.ws_view("num_tiles", torch.int32, 2, n + 8)[1]) == want
        assert np.array_equal(bits16(out), ref)


@pytest.mark.parametrize("act", ["fp8", "bf16"])
@pytest.mark.parametrize("extra,want", [(0, 1), (1, 0)])
def test_local_pairs_at_the_line(extra, want, act):
    """An MXFP4 call above the few-rows line: local pairs exactly at 40 per local expert, and one
    more."""
    num_local, hidden, inter = 42, 256, 128
    counts = spread(num_local - 1, FEW_ROWS, FEW_ROWS + extra)
    n, more = FEW_ROWS * num_local + 301, GATED * num_local + 1
    gen = W.generator("cpu", 41)
    x = W.tokens(n + more, hidden, gen, "cpu")
    w = torch.rand(n + more, 1, generator=gen) + 0.25
    ids = torch.cat([ids_for(counts, num_local, n, gen),
                     torch.randint(0, num_local, (more, 1), generator=gen, dtype=torch.int32)])
    w13, w2 = W.expert_weights(num_local, hidden, inter, gen, "cpu")
    experts = AfdExperts(4 * num_local, 1, 0, range(num_local), pack_mxfp4_experts(w13, w2, device=dev()),
                         n_max=n + more, act_format="bf16" if act == "bf16" else None)

    def call(m):
        experts.workspace().fill_(0xFF)
        out = experts(x[:m].to(dev()), StandardTopKOutput(w[:m].to(dev()), ids[:m].to(dev())))
        torch.cuda.synchronize()
        return bits16(out)

    got = call(n)
    assert int(experts.ws_view("num_tiles", torch.int32, 2, n)[1]) == want
    assert np.array_equal(got, call(n + more)[:n])


@pytest.mark.parametrize("act", ["fp8", "bf16"])
@pytest.mark.parametrize("n,want", [(3, 1), (210, 1), (211, 0), (400, 0)])
def test_capacity_above_the_line(n, want, act):
    """A descriptor call with room for 50 pairs per local expert, all experts local: by the tokens it
    has (40 pairs per expert, and one token more), the few rows or the large tiles."""
    num_local, k, cap = 42, 8, 400
    gen = W.generator("cpu", 43)
    x = W.tokens(cap, 512, gen, "cpu").to(dev())
    ids, w = W.route_uniform(cap, num_local, k, gen, "cpu")
    w13, w2 = W.expert_weights(num_local, 512, 256, gen, "cpu")
    experts = AfdExperts(num_local, k, 0, range(num_local), pack_mxfp4_experts(w13, w2, device=dev()), n_max=cap,
                         act_format="bf16" if act == "bf16" else None)
    ids, w = ids.to(torch.int32).to(dev()), w.float().to(dev())
    experts.workspace().fill_(0xFF)
    desc, out = new_job_desc(dev()), torch.full((n, 512), float("nan"), dtype=torch.bfloat16, device=dev())
    set_job(desc, ids=ids[:n], w=w[:n], out=out, x=x[:n])
    experts.call_job(desc, cap)
    torch.cuda.synchronize()
    assert int(experts.ws_view("num_tiles", torch.int32, 2, cap)[1]) == want
    whole = experts(x, StandardTopKOutput(w, ids))  # its 400 tokens by value: the large tiles
    torch.cuda.synchronize()
    assert np.array_equal(bits16(out), bits16(whole)[:n])


@pytest.mark.parametrize("act", ["fp8", "bf16"])
@pytest.mark.parametrize("fmt", ["mxfp4", "fp8_block"])
def test_one_local_expert(fmt, act):
    """One expert: 1 to 40 of its rows, from one group of 32 rows to one of 64, and none."""
    gen = W.generator("cpu", 47)
    x = W.tokens(300, 512, gen, "cpu").to(dev())
    w13, w2 = W.expert_weights(1, 512, 256, gen, "cpu")
    pack = pack_mxfp4_experts if fmt == "mxfp4" else pack_fp8_block_experts
    experts = AfdExperts(9, 1, 0, range(4, 5), pack(w13, w2, device=dev()), n_max=300,
                         act_format="bf16" if act == "bf16" else None)
    w = (torch.rand(300, 1, generator=gen) + 0.25).to(dev())
    ids = torch.full((300, 1), 4, dtype=torch.int32, device=dev())

    def call(m, which):
        experts.workspace().fill_(0xFF)
        out = experts(x[:m], StandardTopKOutput(w[:m], which[:m]))
        torch.cuda.synchronize()
        return bits16(out)

    whole = call(300, ids)  # large tiles
    for n in (1, 16, 17, 32, 33, 40):
        assert np.array_equal(call(n, ids), whole[:n]), n
    assert not call(40, ids + 1).any()
