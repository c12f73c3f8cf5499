"""CPU: which GEMMs an expert call runs (afd_rows_rule.h, compiled here as host code).

The few-rows GEMMs read an expert's weights once per group of 64 (or 32) rows, so with the pairs
concentrated on few experts they lose to the large tiles, on 256 experts by up to 2.2 times. A call
launches them alone only while it is too small for that; a larger one launches both forms and the
router's counts choose."""

import os
import random
import shutil
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
HIPCC = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
LARGE, FEW, BOTH = 0, 1, 2
MXFP4, FP8_BLOCK = 1, 2


def n_pairs(case):
    return case["n"] * case.get("topk", 8)


@pytest.fixture(scope="module")
def rule(tmp_path_factory):
    if not os.path.exists(HIPCC):
        pytest.skip("hipcc is not available to build the host program")
    exe = tmp_path_factory.mktemp("rows_rule") / "rows_rule"
    subprocess.run([HIPCC, "-O1", "-std=c++17", "-x", "hip", "--cuda-host-only", os.path.join(HERE, "rows_rule.cpp"),
                    "-o", str(exe)], check=True, stdout=subprocess.PIPE, stderr=subprocess.STDOUT)

    def run(cases):
        """cases: dicts; returns (form, group rows, the router's choice) of each. ``counts``: rows per
        expert; ``capacity``: the call's descriptor holds its tokens, n is the most."""
        lines = []
        for c in cases:
            n, k, local = c["n"], c.get("topk", 8), c["local"]
            rows = 32 if n * k <= 16 * local else 64
            counts = c.get("counts", [])
            lines.append(f"{c['fmt']} {c.get('inter', 2048)} {k} {c.get('lo', 0)} {local} {c.get('walk', 0)} {n} "
                         f"{c.get('capacity', 0)} "
                         f"{sum(counts)} {sum(-(-v // rows) for v in counts)} {sum(v > 0 for v in counts)}")
        res = subprocess.run([str(exe)], input="\n".join(lines) + "\n", stdout=subprocess.PIPE, text=True, timeout=60,
                             check=True)
        got = [tuple(int(v) for v in line.split()) for line in res.stdout.splitlines()]
        for c, (form, rows, choice, grid_groups) in zip(cases, got):  # the launch covers whatever runs
            groups = sum(-(-v // rows) for v in c.get("counts", []))
            assert form == LARGE or form == BOTH and not choice or groups <= grid_groups, c
            # alone above 2560 pairs only where no routing makes the counts say otherwise
            assert form != FEW or n_pairs(c) <= 2560 or choice, c
        return [g[:3] for g in got]

    return run


@pytest.mark.parametrize("fmt", [MXFP4, FP8_BLOCK])
def test_form_and_group_rows_at_the_lines(rule, fmt):
    cases = [
        (dict(local=64, n=1), (FEW, 32)),
        (dict(local=64, n=128), (FEW, 32)),  # 16 pairs per expert
        (dict(local=64, n=129), (FEW, 64)),
        (dict(local=64, n=320), (FEW, 64)),  # 40 pairs per expert, 2560 pairs
        (dict(local=64, n=321), (BOTH if fmt == MXFP4 else LARGE, 64)),
        (dict(local=65, n=2560, topk=1), (FEW, 64)),
        (dict(local=65, n=2561, topk=1), (BOTH, 64)),
        (dict(local=256, n=256), (FEW, 32)),  # 2048 pairs
        (dict(local=256, n=257), (BOTH, 32)),
        (dict(local=256, n=512), (BOTH, 32)),
        (dict(local=256, n=513), (BOTH, 64)),
        (dict(local=256, n=1280), (BOTH, 64)),
        (dict(local=1, n=5), (FEW, 64)),
        (dict(local=1, n=2, topk=8), (FEW, 32)),
        (dict(local=64, n=131071), (LARGE, 64)),
    ]
    got = rule([dict(c, fmt=fmt) for c, _ in cases])
    assert [g[:2] for g in got] == [want for _, want in cases]


@pytest.mark.parametrize("fmt", [MXFP4, FP8_BLOCK])
def test_concentrated_routing_takes_the_large_tiles(rule, fmt):
    """Routings measured: those the few-rows GEMMs lost by 20% and more go to the large tiles, even
    loads and Zipf-like ones stay with the few rows."""
    hot = lambda total, m, local: [total // m] * m + [0] * (local - m)
    large = [dict(local=256, n=1280, counts=hot(10240, m, 256)) for m in (8, 32, 64, 128)]
    large += [dict(local=256, n=510, counts=hot(4080, m, 256)) for m in (16, 32, 64)]
    large += [dict(local=128, n=640, counts=hot(5120, m, 128)) for m in (12, 16, 32, 64)]
    few = [dict(local=256, n=1280, counts=[40] * 256), dict(local=256, n=510, counts=[15] * 256),
           dict(local=128, n=640, counts=[40] * 128),
           dict(local=256, n=1280, counts=[700, 300, 200, 100] + [35] * 252)]
    got = rule([dict(c, fmt=fmt) for c in large + few])
    assert all(form == BOTH for form, _, _ in got)
    assert [choice for _, _, choice in got] == [0] * len(large) + [1] * len(few)


@pytest.mark.parametrize("local,inter", [(64, 2048), (65, 1536), (128, 2048), (256, 512), (256, 1024), (256, 2048)])
@pytest.mark.parametrize("fmt", [MXFP4, FP8_BLOCK])
def test_few_rows_run_alone_only_in_small_calls(rule, fmt, local, inter):
    sizes = list(range(1, 6 * local))
    cases = [dict(fmt=fmt, local=local, inter=inter, n=n, walk=4 * local << 8 | n % 2) for n in sizes]
    for n, (form, rows, _) in zip(sizes, rule(cases)):
        pairs = 8 * n
        if pairs > 40 * local:
            assert form == (BOTH if fmt == MXFP4 and pairs <= 140 * local else LARGE), n
        else:
            rounds = (1536 if rows == 32 else 1024) // (inter // 128)  # row groups of two rounds
            alone = pairs <= (2048 if rows == 32 else 2560) or 3 * pairs <= rounds * rows
            assert form == (FEW if alone else BOTH), n
            assert rows == (32 if pairs <= 16 * local else 64), n


@pytest.mark.parametrize("lo,said,last", [
    (0, 64, 320),  # all local
    (0, 65, 320), (0, 80, 350),  # the few-rows line itself; 35 pairs per expert of the model
    (0, 128, 560), (64, 128, 560),  # half
    (0, 256, 1120), (192, 256, 1120), (0, 0, 1120), (64, 0, 1120),  # a quarter; not said
    (0, 512, 1120),  # an eighth: measured up to a quarter
])
def test_both_forms_are_launched_only_near_the_line(rule, lo, said, last):
    """An MXFP4 rank launches both forms for the count of local pairs only where its share of the
    experts makes few local pairs likely: with all experts local it never does."""
    sizes = range(1, 1500)
    got = rule([dict(fmt=MXFP4, local=64, lo=lo, n=n, walk=said << 8 | n % 2) for n in sizes])
    assert [form for form, _, _ in got] == [FEW if n <= 320 else BOTH if n <= last else LARGE for n in sizes]
    got = rule([dict(fmt=FP8_BLOCK, local=64, lo=lo, n=n, walk=said << 8 | n % 2) for n in sizes])
    assert [form for form, _, _ in got] == [FEW if n <= 320 else LARGE for n in sizes]
    # a capacity: the job may have few tokens, so the count decides up to 140 pairs per expert
    got = rule([dict(fmt=MXFP4, local=64, lo=lo, n=n, walk=said << 8 | n % 2, capacity=1) for n in sizes])
    assert [form for form, _, _ in got] == [FEW if n <= 320 else BOTH if n <= 1120 else LARGE for n in sizes]


def test_the_launch_covers_every_routing(rule):
    """Random loads, even to concentrated: the few-rows grid has a group for each that can be."""
    rng = random.Random(3)
    cases = []
    for _ in range(4000):
        local = rng.choice([1, 2, 5, 64, 65, 128, 256])
        k = rng.randint(1, 8)
        n = rng.randint(1, max(1, 45 * local // k))
        hot = rng.randint(1, local)
        counts = [0] * local
        left = rng.choice([n * k, rng.randint(0, n * k)])
        for e in range(hot):
            counts[e] = left // hot + (e < left % hot)
        for _ in range(hot):
            a, b = rng.randrange(hot), rng.randrange(hot)
            moved = rng.randint(0, counts[a])
            counts[a] -= moved
            counts[b] += moved
        cases.append(dict(fmt=rng.choice([MXFP4, FP8_BLOCK]), local=local, topk=k, n=n, counts=counts,
                          inter=rng.choice([128, 1024, 2048, 16384]), walk=4 * local << 8))
    rule(cases)
