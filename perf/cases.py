"""The work a user of this package has it do, as cases that can be timed.

    listed()          the cases by name
    draw(rng)         one more case of the same ranges
    prepare(case, s)  what a program holds before the call: tensors on the GPU, and the plan where it keeps one
    run(state)        one pass through the public entry points, and its outputs
    work(case)        bytes and operations a pass cannot do without
    tolerance(case)   how far another correct implementation of the same precision may be off

A case is a dict of plain values:
    path    which entry points a pass goes through (see PATHS)
    lens    tokens per rank, "4096*8" (eight equal ranks) or "640,512,384,512"
    batch, heads, kv_heads, dim, dtype, causal, zigzag
    sigma   standard deviation of the Q and K entries (how peaked the softmax is)
    graph   a forward replayed as a captured graph
    half    per-step partial O kept in fp16
    rows    per-step partials of a row next to each other
    rank    the rank of the calls that run one rank
"""
import numpy as np
import torch

from ringattention_amd import api, torch_ops

PATHS = ("forward",          # all ranks of the ring in one call on a plan: what bench.py times
         "step_partials",    # the same on a plan that keeps the ring steps apart
         "torch_op",         # the dispatcher op: plan and outputs are its own business
         "rank_call",        # the reference-shaped call, one head and one rank, blocking
         "rank_call_noalloc",  # the same without allocation or synchronisation: serving loops
         "rank_ring",        # one process's share of a ring over several GPUs: its steps one by one, then the merge
         "merge_ring")       # merge of the per-step partials of all ranks
TORCH = {"fp16": torch.float16, "bf16": torch.bfloat16}
DEFAULTS = {"batch": 1, "heads": 1, "kv_heads": 0, "dim": 128, "dtype": "fp16", "causal": False, "zigzag": False, "sigma": 1.0,
            "graph": False, "half": False, "rows": False, "rank": 0}


def _case(path, lens, **more):
    return dict(DEFAULTS, path=path, lens=lens, **more)


def listed():
    cases = [
        # the smallest ring: four ranks of 128 tokens, one head.  A forward is a few microseconds of GPU work, so what
        # counts is the call, the launch and the latency of one short walk
        _case("forward", "128*4", name="tiny_ring", dim=64),
        # the reference's own program: two ranks of 8192 tokens, one head, fp16, d = 64; a rank per call, blocking
        _case("rank_call", "8192*2", name="reference_call", dim=64),
        # the same kind of call in a loop that may not allocate: unequal ranks, causal, bf16, the last rank's rows
        _case("rank_call_noalloc", "640,512,384,512", name="serving_call", dtype="bf16", causal=True, rank=3),
        # eight heads, 8 x 1024 tokens, d = 64: one workgroup per compute unit
        _case("forward", "1024*8", name="ring_d64", heads=8, dim=64),
        # many short ranks, batched, graph replay
        _case("forward", "512*32", name="short_ranks", batch=4, heads=16, graph=True),
        # the headline: causal, 32 heads, 32 K tokens in eight ranks
        _case("forward", "4096*8", name="causal_32k", heads=32, dtype="bf16", causal=True),
        # the longest: 128 K tokens without a mask, peaked softmax (N(0, 9) logits before the scale)
        _case("forward", "8192*16", name="long_128k", heads=16, sigma=3.0),
        # tensors as a program has them: ragged ranks, grouped-query heads, causal, through the torch op
        _case("torch_op", "1021,777,1300,64,905,333", name="ragged_gqa", heads=16, kv_heads=4, dtype="bf16", causal=True),
        # the forward with the ring steps kept apart, fp16 partials
        _case("step_partials", "512*32", name="steps_apart", batch=4, heads=16, half=True),
        # one GPU's share of the headline over a ring of eight: balanced causal layout, eight launches and a merge
        _case("rank_ring", "4096*8", name="rank_ring_zigzag", heads=32, dtype="bf16", causal=True, zigzag=True, rank=5),
        # the same for a short ring of few heads, where a step is a small launch
        _case("rank_ring", "1024*8", name="rank_ring_short", heads=8, dim=64, rank=3),
        # the merge of the headline's per-step partials
        _case("merge_ring", "4096*8", name="merge_32k", heads=32, dtype="bf16", causal=True),
    ]
    return cases


def _log_int(rng, lo, hi):
    return int(round(lo * (hi / lo) ** rng.random()))


MAX_FLOPS = 2e13          # a drawn case does at most this (the longest listed one does 1.4e14)
MAX_PARTIAL_BYTES = 9e9   # per-step partials of a drawn case (the listed ones hold 2.7e9 to 9e9)


def draw(rng):
    """Sizes over the whole range: rings of 1 to 32 ranks, 64 to 8192 tokens per rank (equal, multiples of 32, or ragged),
    1 to 64 heads in all."""
    while True:
        path = rng.choice(("forward", "forward", "forward", "torch_op", "torch_op", "rank_call", "rank_call_noalloc", "step_partials",
                           "rank_ring", "merge_ring"))
        ranks = _log_int(rng, 1, 32)
        chunk = _log_int(rng, 64, 8192)
        causal = rng.random() < 0.5
        zigzag = causal and rng.random() < 0.4
        kind = rng.choice(("equal", "rounded", "ragged"))
        if kind == "equal":
            grain = rng.choice((64, 128, 256))
            lens = "%d*%d" % (max(grain, chunk // grain * grain), ranks)
        else:
            grain = 32 if kind == "rounded" else 1
            ls = [max(grain, int(chunk * (0.4 + 1.2 * rng.random())) // grain * grain) for _ in range(ranks)]
            lens = ",".join(str(n - n % 2 if zigzag else n) for n in ls)
        c = _case(path, lens, dim=rng.choice((64, 128)), dtype=rng.choice(("fp16", "bf16")), causal=causal, zigzag=zigzag,
                  sigma=rng.choice((1.0, 1.0, 1.0, 3.0)), rank=rng.randrange(ranks))
        if path.startswith("rank_call"):
            c["zigzag"] = False
        else:
            c["batch"] = rng.choice((1, 1, 1, 2, 4))
            c["heads"] = rng.choice((1, 2, 4, 6, 8, 12, 16))
            if rng.random() < 0.3:
                c["kv_heads"] = rng.choice([g for g in range(1, c["heads"] + 1) if c["heads"] % g == 0])
        if path == "forward":
            c["graph"] = rng.random() < 0.15
        if path in ("step_partials", "rank_ring", "merge_ring"):
            c["half"] = rng.random() < 0.4
        if path in ("rank_ring", "merge_ring"):
            c["rows"] = rng.random() < 0.4
        parts = c["batch"] * c["heads"] * sum(_lens(c)) * ranks * (c["dim"] + 1) * 4
        if work(c)["flops"] <= MAX_FLOPS and (path not in ("step_partials", "rank_ring", "merge_ring") or parts <= MAX_PARTIAL_BYTES):
            return c


def _lens(c):
    if "*" in c["lens"]:
        n, ranks = c["lens"].split("*")
        return [int(n)] * int(ranks)
    return [int(x) for x in c["lens"].split(",")]


class _Inputs:
    def __init__(self, case, seed):
        self.gen = torch.Generator(device="cuda").manual_seed(seed)
        self.dtype = TORCH[case["dtype"]]

    def normal(self, shape, sigma=1.0, dtype=None):
        x = torch.randn(shape, generator=self.gen, device="cuda", dtype=dtype or self.dtype)
        return x if sigma == 1.0 else x.mul_(sigma)


def _plan(c, **more):
    return api.RingAttention(len(_lens(c)), _lens(c), c["dim"], c["batch"], c["heads"], c["dtype"], c["causal"], kv_heads=c["kv_heads"],
                             layout="zigzag" if c["zigzag"] else "contiguous", **more)


def prepare(case, seed):
    c, x, lens = case, _Inputs(case, seed), _lens(case)
    B, H, d, S, P, path = c["batch"], c["heads"], c["dim"], sum(lens), len(lens), c["path"]
    s = {"case": c}
    if path in ("rank_call", "rank_call_noalloc"):
        rows = lens[c["rank"]]
        s.update(q=x.normal((rows, d), c["sigma"]), k=x.normal((S, d), c["sigma"]), v=x.normal((S, d)), lens=lens,
                 out=torch.empty(rows, d, dtype=x.dtype, device="cuda"), lse=torch.empty(rows, dtype=torch.float32, device="cuda"))
        return s
    hkv = c["kv_heads"] or H
    if path in ("forward", "step_partials", "torch_op"):
        s.update(q=x.normal((B, H, S, d), c["sigma"]), k=x.normal((B, hkv, S, d), c["sigma"]), v=x.normal((B, hkv, S, d)))
        if path == "torch_op":
            s["lens"] = lens
            return s
        s["plan"] = _plan(c, graph=c["graph"]) if path == "forward" else _plan(c, step_partials=True, half_partials=c["half"])
        s.update(out=torch.empty_like(s["q"]), lse=torch.empty(B, H, S, dtype=torch.float32, device="cuda"))
        return s
    s["plan"] = plan = _plan(c, half_partials=c["half"], row_partials=c["rows"])
    if path == "rank_ring":
        # the rank's own queries, and the K/V chunk of every step as the exchange delivers it
        r = c["rank"]
        s["q"] = x.normal((B, H, lens[r], d), c["sigma"])
        s["chunks"] = [(x.normal((B, hkv, lens[(r + t) % P], d), c["sigma"]), x.normal((B, hkv, lens[(r + t) % P], d))) for t in range(P)]
        o_shape, l_shape = plan.rank_parts_shapes(r)
        s.update(o_parts=torch.zeros(o_shape, dtype=plan.part_dtype, device="cuda"), l_parts=torch.zeros(l_shape, device="cuda"),
                 out=torch.empty_like(s["q"]), lse=torch.empty(B, H, lens[r], dtype=torch.float32, device="cuda"))
        return s
    # merge_ring: partials as the steps leave them, rows averaging some V rows and LSEs of similar size
    o_shape, l_shape = plan.parts_shapes()
    s.update(o_parts=x.normal(o_shape, 0.1, plan.part_dtype), l_parts=x.normal(l_shape, 1.0, torch.float32).add_(8.0),
             out=torch.empty(B, H, S, d, dtype=x.dtype, device="cuda"), lse=torch.empty(B, H, S, dtype=torch.float32, device="cuda"))
    return s


def run(s):
    c = s["case"]
    path = c["path"]
    if path in ("forward", "step_partials"):
        return s["plan"].forward(s["q"], s["k"], s["v"], s["out"], s["lse"])
    if path == "torch_op":
        return torch_ops.ring_attention_fwd(s["q"], s["k"], s["v"], s["lens"], c["causal"], zigzag=c["zigzag"])
    if path in ("rank_call", "rank_call_noalloc"):
        call = api.ring_attention if path == "rank_call" else api.ring_attention_noalloc
        lens = s["lens"]
        call(s["q"], s["k"], s["v"], s["out"], len(lens), c["rank"], lens, c["dim"], max(lens), lse=s["lse"], causal=c["causal"])
        return s["out"], s["lse"]
    plan = s["plan"]
    if path == "rank_ring":
        o, l = s["o_parts"], s["l_parts"]
        for t, (k, v) in enumerate(s["chunks"]):
            plan.rank_step_forward(c["rank"], t, s["q"], k, v, o if c["rows"] else o[t], l if c["rows"] else l[t])
        return plan.rank_merge(c["rank"], o, l, s["out"], s["lse"]) + (o, l)
    return plan.merge_ring(s["o_parts"], s["l_parts"], s["out"], s["lse"])


def _positions(c):
    """(first sequence position, rows) of the runs of every rank's rows, in memory order."""
    lens = _lens(c)
    if not c["zigzag"]:
        at = np.concatenate(([0], np.cumsum(lens)))
        return [[(int(at[r]), n)] for r, n in enumerate(lens)]
    half = [n // 2 for n in lens]
    low = np.concatenate(([0], np.cumsum(half)))
    high = low[-1] + np.concatenate(([0], np.cumsum(half[::-1])))
    P = len(lens)
    return [[(int(low[r]), half[r]), (int(high[P - 1 - r]), half[r])] for r in range(P)]


def _pairs(c, rank=None):
    """Visible (query, key) pairs of a head: of all ranks, or of one."""
    S, lens = sum(_lens(c)), _lens(c)
    if not c["causal"]:
        return (S if rank is None else lens[rank]) * S
    runs = [run for r, own in enumerate(_positions(c)) if rank in (None, r) for run in own]
    return sum(n * at + n * (n + 1) // 2 for at, n in runs)


def work(case):
    c, lens = case, _lens(case)
    B, H, d, S, P = c["batch"], c["heads"], c["dim"], sum(lens), len(lens)
    hkv = c["kv_heads"] or H
    if c["path"] in ("rank_call", "rank_call_noalloc"):
        r = c["rank"]
        keys = sum(lens[:r + 1]) if c["causal"] else S
        return {"bytes": lens[r] * (4 * d + 4) + keys * 4 * d, "flops": 4 * d * _pairs(c, r)}
    if c["path"] in ("forward", "step_partials", "torch_op"):
        return {"bytes": B * H * S * (4 * d + 4) + B * hkv * S * 4 * d, "flops": 4 * d * B * H * _pairs(c)}
    part = d * (2 if c["half"] else 4) + 4   # a partial row
    own = [c["rank"]] if c["path"] == "rank_ring" else range(P)
    part_rows = 0    # partial rows the steps of a head write: those that see a key of the visited chunk
    kv_rows = 0
    for r in own:
        for t in range(P):
            j = (r + t) % P
            if not c["causal"] or j == r:
                part_rows, kv_rows = part_rows + lens[r], kv_rows + lens[j]
            elif not c["zigzag"] and j < r:
                part_rows, kv_rows = part_rows + lens[r], kv_rows + lens[j]
            elif c["zigzag"]:
                part_rows += lens[r] if j < r else lens[r] // 2
                kv_rows += lens[j] // 2 if j < r else lens[j]
    rows = sum(lens[r] for r in own)
    merge = {"bytes": B * H * (part_rows * part + rows * (2 * d + 4)), "flops": B * H * part_rows * 2 * d}
    if c["path"] == "merge_ring":
        return merge
    # every partial is an output of its step and an input of the merge; the queries once
    return {"bytes": merge["bytes"] + B * H * (part_rows * part + rows * 2 * d) + B * hkv * kv_rows * 4 * d,
            "flops": merge["flops"] + 4 * d * B * H * _pairs(c, c["rank"])}


def tolerance(case):
    """About four times what the paths show against the same computation in fp64.  What separates two correct
    implementations is the rounding of the probabilities and of O to the storage type: relative 2-norm 2.0e-4 to 3.6e-4 in
    fp16 and 1.8e-3 to 2.4e-3 in bf16.  The largest single entry (against its own size or the rms, whichever is more)
    was 1.7e-3 / 1.1e-2 without a mask; under the causal mask the rows of few keys, whose entries are far above the
    rms, reach 6.3e-3 / 4.8e-2.  A merge only rounds its result: 2.1e-4 / 1.7e-3, largest 5e-4 / 3.9e-3.  (LSEs, in fp32,
    are within 2e-7 everywhere.)"""
    fp16 = case["dtype"] == "fp16"
    if case["path"] == "merge_ring":
        return {"rel": 8.5e-4, "max": 2e-3} if fp16 else {"rel": 6.8e-3, "max": 1.6e-2}
    if fp16:
        return {"rel": 1.4e-3, "max": 2.5e-2 if case["causal"] else 7e-3}
    return {"rel": 9.6e-3, "max": 0.19 if case["causal"] else 4.5e-2}
