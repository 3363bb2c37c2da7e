"""Performance cases of the Helix all-to-all: the calls a serving program makes, over the sizes it makes them at.

A decode step of a model served with decode context parallelism ends every attention layer with one
exchange over ``cp`` ranks, here the logical ranks of one GPU. A program gets there in one of these ways:

* ``alltoall``  ``helix_a2a.alltoall`` once per rank, the reference's signature;
* ``loopback``  ``helix_a2a.alltoall_loopback``, all ranks in one call;
* ``plan``      ``LoopbackPlan.run()``, a loop with buffers that stay where they are;
* ``combine``   ``helix_a2a.alltoall_combine_loopback``, exchange and LSE-weighted combine, (max, sum) statistics;
* ``combine_plan``  the same, replayed from a ``CombinePlan``;
* ``reduce``    ``helix_a2a.dcp_a2a_lse_reduce``, what the serving integration calls: ``[B, H, D]`` and
                ``[B, H]`` log-sum-exps per rank in, ``[B, H/cp, D]`` per rank out.

Shapes are those of the repository's workloads (cp, tokens, query heads, head width), of its pipeline
benchmark (64 heads of 128, 16 heads of 512, batches of 1 to 512) and of its tests.
"""
from __future__ import annotations

import os
import sys

import torch

sys.path.insert(0, os.path.join(os.getcwd(), "helix-a2a_amd"))  # the package's folder in the tree this runs in
import helix_a2a  # noqa: E402
from helix_a2a import _ops  # noqa: E402

_DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16}
_EXCHANGES = ("alltoall", "loopback", "plan")


def _case(name, call, cp, tokens, heads, dim, dtype="bf16", per_head=False, lse=False, base2=False, masked=0.0):
    case = {"call": call, "cp": cp, "tokens": tokens, "heads": heads, "dim": dim, "dtype": dtype,
            "per_head": per_head, "lse": lse, "base2": base2, "masked": masked}
    return {"name": name, **case} if name else case


def listed():
    return [
        # one user decoding: the smallest call, launch and host time are everything
        _case("reduce_batch1", "reduce", 8, 1, 64, 128),
        # sixteen wide heads (latent attention) with the combined log-sum-exp in base 2, an odd small batch
        _case("reduce_wide_heads_lse", "reduce", 8, 33, 16, 512, lse=True, base2=True),
        # a full batch of grouped-query heads, half precision
        _case("reduce_batch512_fp16", "reduce", 8, 512, 64, 128, dtype="fp16"),
        # many ranks, short rows, some heads masked on a rank: the largest reduce
        _case("reduce_16_ranks", "reduce", 16, 1024, 32, 128, masked=0.01),
        # an ordinary decode step with running (max, sum) statistics, eager
        _case("combine_4_ranks", "combine", 4, 64, 32, 128, lse=True),
        # 128 latent heads of 512, buffers kept: the largest message rows through the combine
        _case("combine_plan_latent", "combine_plan", 8, 128, 128, 512),
        # the reference's signature at a small and at an ordinary decode step
        _case("alltoall_4_ranks", "alltoall", 4, 64, 32, 128),
        _case("alltoall_8_ranks", "alltoall", 8, 256, 64, 128),
        # the serving integration's layout: one entry per (token, head), 8-byte statistics rows
        _case("alltoall_per_head", "alltoall", 8, 256, 64, 128, per_head=True),
        # ragged: odd token count, rows that are no power of two, masked heads
        _case("loopback_ragged_fp16", "loopback", 4, 37, 24, 96, dtype="fp16", masked=0.01),
        # large message rows, all ranks in one call
        _case("loopback_latent", "loopback", 8, 128, 128, 512),
        # many short rows between many ranks: the largest exchange
        _case("plan_16_ranks", "plan", 16, 1024, 32, 128, masked=0.01),
    ]


# every call with more than one decode step's worth of data stays within the largest listed case
_MAX_INPUT_BYTES = 16 * 1024 * 32 * 128 * 2


def draw(rng):
    call = rng.choice(("alltoall", "loopback", "plan", "combine", "combine_plan", "reduce", "reduce", "reduce"))
    while True:
        cp = rng.choice((2, 3, 4, 6, 8, 8, 8, 12, 16))
        tokens = int(round(2.0 ** rng.uniform(0.0, 10.0)))
        if tokens > 2 and rng.random() < 0.5:
            tokens |= 1
        heads = cp * rng.choice((1, 2, 3, 4, 5, 8, 8, 16))
        dim = rng.choice((64, 80, 96, 128, 128, 128, 192, 256, 512))
        if cp * tokens * heads * dim * 2 <= _MAX_INPUT_BYTES:
            break
    exchange = call in _EXCHANGES
    return _case(None, call, cp, tokens, heads, dim, dtype=rng.choice(("bf16", "bf16", "fp16")),
                 per_head=exchange and rng.random() < 0.3, lse=not exchange and rng.random() < 0.5,
                 base2=call == "reduce" and rng.random() < 0.3, masked=rng.choice((0.0, 0.0, 0.01)))


def prepare(case, seed):
    cp, tokens, heads, dim = case["cp"], case["tokens"], case["heads"], case["dim"]
    hp, dtype, call = heads // cp, _DTYPES[case["dtype"]], case["call"]
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    # partial outputs are averages of value vectors, normal at unit scale; running maxima are spread over a few
    # units, running sums over the length of a rank's shard of the sequence
    o = torch.randn(cp, tokens, heads, dim, generator=g, device="cuda", dtype=torch.float32).to(dtype)
    top = torch.randn(cp, tokens, heads, generator=g, device="cuda") * 3.0
    total = 1.0 + torch.rand(cp, tokens, heads, generator=g, device="cuda") * 8191.0
    if case["masked"] > 0:
        masked = torch.rand(cp, tokens, heads, generator=g, device="cuda") < case["masked"]
        top = torch.where(masked, torch.full_like(top, float("-inf")), top)
    state = {"call": call, "cp": cp, "lse": case["lse"], "base2": case["base2"]}
    ws = helix_a2a.allocate_workspace(cp, 0)
    for r in range(cp):
        helix_a2a.init_workspace(ws, r, cp)
    state["ws"] = ws
    if call == "reduce":
        lse = top + total.log()
        if case["base2"]:
            lse = lse * 1.4426950408889634
        # a tensor of its own per rank: every rank's attention kernel has written it
        state["o"], state["s"] = [t.clone() for t in o], [t.clone() for t in lse]
        return state
    stats = torch.stack((top, total), dim=-1)
    if case["per_head"]:
        o = o.view(cp, tokens, cp, hp, dim).permute(0, 1, 3, 2, 4).reshape(cp, tokens * hp, cp, dim)
        stats = stats.view(cp, tokens, cp, hp, 2).permute(0, 1, 3, 2, 4).reshape(cp, tokens * hp, cp, 2)
    else:
        o, stats = o.view(cp, tokens, cp, hp * dim), stats.view(cp, tokens, cp, hp * 2)
    ins_o, ins_s = [t.clone() for t in o], [t.clone() for t in stats]
    if call == "plan":
        state["plan"] = _ops.LoopbackPlan(ins_o, ins_s, ws)
    elif call == "combine_plan":
        state["plan"] = _ops.CombinePlan(ins_o, ins_s, ws, helix_a2a.STATS_MAX_SUM, case["lse"])
    else:
        state["o"], state["s"] = ins_o, ins_s
    return state


def run(state):
    call = state["call"]
    if call == "reduce":
        return helix_a2a.dcp_a2a_lse_reduce(state["o"], state["s"], state["ws"], return_lse=state["lse"],
                                            is_lse_base_on_e=not state["base2"])
    if call == "alltoall":
        cp = state["cp"]
        return [helix_a2a.alltoall(state["o"][r], state["s"][r], state["ws"], r, cp) for r in range(cp)]
    if call == "loopback":
        return helix_a2a.alltoall_loopback(state["o"], state["s"], state["ws"])
    if call == "combine":
        return helix_a2a.alltoall_combine_loopback(state["o"], state["s"], state["ws"], helix_a2a.STATS_MAX_SUM, state["lse"])
    return state["plan"].run()


def work(case):
    """Every input read once, every output written once; the weighted sum of the combine is two operations a term."""
    cp, tokens, heads, dim = case["cp"], case["tokens"], case["heads"], case["dim"]
    values = cp * tokens * heads * dim
    stats = cp * tokens * heads * (4 if case["call"] == "reduce" else 8)
    if case["call"] in _EXCHANGES:
        return {"bytes": 2 * (2 * values + stats), "flops": 0}
    out = 2 * values // cp + (4 * tokens * heads if case["lse"] else 0)
    return {"bytes": 2 * values + stats + out, "flops": 2 * values}


def tolerance(case):
    """The exchange moves bytes. The combine sums in fp32 and rounds once to the type of its inputs: half an ulp of
    bf16 is 2^-9, of fp16 2^-12 of a value, a third to a half of that in the 2-norm over many values; the combined
    log-sum-exp is an fp32 sum. Against the same combine in double precision: bf16 1.7e-3 and at most 3.9e-3 of a
    value, fp16 2.1e-4 and 4.9e-4; four times that here."""
    if case["call"] in _EXCHANGES:
        return "exact"
    return {"rel": 6e-3, "max": 1.6e-2} if case["dtype"] == "bf16" else {"rel": 8e-4, "max": 2e-3}
