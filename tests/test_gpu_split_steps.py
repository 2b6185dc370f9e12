"""steps::ring_split_kernel (ringattn_split_steps.hip): the ring steps apart, their keys split over the eight waves of a workgroup.  Its
partials are documented to have the same bits in every launch of a plan -- a step of one rank, of all ranks, the forward that
merges them: the bound between these is equality -- and are held to the oracle like any other's.  Sizes where it can go
wrong: ranges of one tile, around the lengths that one, two, four and eight waves share (4, 8, 16 tiles), several rounds of ranges, more
ranges than waves, tails of one key, q tiles that end early, zigzag halves that are no multiple of a tile, diagonals, keys
hidden in the first tiles, references that move in every tile."""
import numpy as np
import pytest
import torch

from launched import kernels
from ringattention_amd import api
from ringattention_amd.configs import Workload
from test_gpu_parity import check_rows
from test_kernel_resources import compile_to_asm
from test_kernel_resources import test_no_lds_transfer_reads_a_scalar_register_fresh_from_a_vector_instruction as _hazards

SWITCHES = ("RINGATTN_WIDE", "RINGATTN_WIDE_PARTIALS", "RINGATTN_SPLIT", "RINGATTN_THIN", "RINGATTN_SPLIT_STEPS")


@pytest.fixture(autouse=True)
def no_switches(monkeypatch):
    for name in SWITCHES:
        monkeypatch.delenv(name, raising=False)


@pytest.mark.gpu
@pytest.mark.parametrize("half", [False, True])
@pytest.mark.parametrize("d", [64, 128])
@pytest.mark.parametrize("lens,causal,zigzag,kind", [
    ((1,), False, False, "flat"),
    ((128, 129, 31), False, False, "flat"),                # 4 and 5 tiles
    ((256, 257, 255), True, False, "flat"),                # 8 and 9
    ((512, 513, 40), True, False, "rising"),               # 16 and 17
    ((33,) * 12 + (290,), True, False, "flat"),            # two rounds of short ranges, one longer
    ((130, 70, 2, 258, 18) * 2, True, True, "rising"),     # halves of 65, 35, 1, 129 and 9 rows
    ((9,) * 63 + (321,), False, False, "flat"),            # as many ranges as there may be
    ((1000, 24), False, False, "steep"),
    ((300, 500), True, False, "hidden"),
    ((700, 300), False, False, "hidden"),
])
def test_steps_and_forward_give_the_same_bits_and_the_oracles_numbers(oracle, monkeypatch, lens, causal, zigzag, kind, d, half):
    monkeypatch.setenv("RINGATTN_SPLIT_STEPS", "1")
    P, S, B, H = len(lens), sum(lens), 1, 3
    dtype = "fp16" if (d == 64) == half else "bf16"
    w = Workload("split_steps", B, H, d, 1, S, dtype, 1500 + S, causal)
    bits = list(api.make_qkv_bits(w))
    q, k, v = (api.bits_to_tensor(np.ascontiguousarray(x), dtype) for x in bits)
    at = np.concatenate(([0], np.cumsum(lens)))
    if kind in ("rising", "steep"):   # scores grow along the sequence, beyond fp16's range of exponentials in between
        q[..., 0] = 8.0
        k[..., 0] = (torch.arange(S, device="cuda", dtype=torch.float32) * (0.02 if kind == "rising" else 0.2)).to(k.dtype)
    if kind == "hidden":              # no finite score in the first 70 keys of a chunk (the first row's own excepted)
        q[..., 0] = 1.0
        for a in at[:-1]:
            k[:, :, a + (1 if causal else 0):a + 70, 0] = float("-inf")
    plan = api.RingAttention(P, list(lens), d, B, H, dtype, causal, layout="zigzag" if zigzag else "contiguous", step_partials=True,
                             half_partials=half)
    assert plan.forward_kernel() == "ring_split_kernel"
    out_buf = torch.full((B * H * S + 64, d), 7.0, dtype=q.dtype, device="cuda")
    out, lse = plan.forward(q, k, v, out_buf[:B * H * S].view(B, H, S, d))
    o_shape, l_shape = plan.parts_shapes()
    o_parts = torch.full(o_shape, float("nan"), dtype=plan.part_dtype, device="cuda")   # nobody may read what no step wrote
    l_parts = torch.full(l_shape, float("-inf"), dtype=torch.float32, device="cuda")
    for s in range(P):
        plan.block_forward(s, q, k, v, o_parts[s], l_parts[s])
    out_m, lse_m = plan.merge_ring(o_parts, l_parts)
    torch.cuda.synchronize()
    assert bool((out_buf[B * H * S:] == 7.0).all()) and not torch.isnan(out).any()
    assert torch.equal(out, out_m) and torch.equal(lse, lse_m)
    for r in {0, P // 2, P - 1}:
        rows = slice(at[r], at[r + 1])
        q_r = q[:, :, rows].contiguous()
        for s in {0, 1 % P, P - 1}:
            j = (r + s) % P
            k_j, v_j = (x[:, :, at[j]:at[j + 1]].contiguous() for x in (k, v))
            o_r, l_r = torch.full((B, H, lens[r], d), float("nan"), dtype=plan.part_dtype, device="cuda"), torch.full((B, H, lens[r]), float("-inf"), device="cuda")
            plan.rank_step_forward(r, s, q_r, k_j, v_j, o_r, l_r)
            torch.cuda.synchronize()
            assert torch.equal(torch.nan_to_num(o_r, 7.0), torch.nan_to_num(o_parts[s][:, :, rows], 7.0)) and torch.equal(l_r, l_parts[s][:, :, rows])
    plan.close()
    if kind != "hidden" and not (zigzag and kind == "rising"):
        order = torch.from_numpy(np.argsort(api.zigzag_order(lens)) if zigzag else np.arange(S)).cuda()
        seq = [x[:, :, order].contiguous().view(torch.int16).cpu().numpy().view(np.uint16) for x in (q, k, v)]
        check_rows(oracle, w, *seq, out[:, :, order].contiguous(), lse[:, :, order].contiguous(), np.arange(w.rows), half_partials=half)


@pytest.mark.gpu
@pytest.mark.parametrize("d,lens,heads,causal,taken", [
    (64, (512,) * 4, 4, False, True),
    (64, (1024,) * 8, 8, False, False),      # all steps at once would take half as long again
    (128, (256,) * 8, 4, False, True),
    (128, (2048,) * 4, 2, False, True),
    (128, (512,) * 32, 2, False, False),
    (128, (777,) * 4, 4, True, True),
    (64, (100,), 4, False, False),           # one range of few tiles
    (64, (40,) * 6, 2, False, False),
])
def test_which_plans_run_on_it(monkeypatch, d, lens, heads, causal, taken):
    """One choice for all launches of a plan, whether or not its forward keeps the steps apart: single steps of all ranks and of one, and
    the forward that merges them, launch what they do with the choice forced to what it should be, and not what they do with the other."""
    x = torch.zeros(1, heads, sum(lens), d, dtype=torch.float16, device="cuda")
    r = len(lens) - 1
    own = x[:, :, :lens[r]].contiguous()
    for apart in (True, False):
        plan = api.RingAttention(len(lens), list(lens), d, 1, heads, "fp16", causal, step_partials=apart)
        o, l = plan.block_forward(0, x, x, x)
        o_r, l_r = plan.rank_step_forward(r, 0, own, own, own)
        out, lse = plan.forward(x, x, x)
        calls = [lambda stream: plan.block_forward(0, x, x, x, o, l, stream), lambda stream: plan.rank_step_forward(r, 0, own, own, own, o_r, l_r, stream)]
        if apart:
            calls.append(lambda stream: plan.forward(x, x, x, out, lse, stream))
            assert (plan.forward_kernel() == "ring_split_kernel") == taken
        for call in calls:
            chosen = kernels(call)
            monkeypatch.setenv("RINGATTN_SPLIT_STEPS", "1" if taken else "0")
            assert kernels(call) == chosen
            monkeypatch.setenv("RINGATTN_SPLIT_STEPS", "0" if taken else "1")
            assert kernels(call) != chosen
            monkeypatch.delenv("RINGATTN_SPLIT_STEPS")
        plan.close()


def test_resources_and_hazards(tmp_path):
    """No scratch, two waves per SIMD at d = 128, two workgroups a compute unit at d = 64; the wait states in front of the
    direct-to-LDS loads."""
    _, usage = compile_to_asm("ringattn_split_steps.hip", tmp_path / "steps.s")
    kernels = {n: u for n, u in usage.items() if "ring_split_kernel" in n}
    assert len(kernels) == 16   # {fp16, bf16} x {64, 128} x {partials rounded to fp16 or not} x {stored, merged}
    for n, u in kernels.items():
        d64 = "ELi64E" in n
        assert u["ScratchSize [bytes/lane]"] == 0 and u["VGPRs"] <= (128 if d64 else 256), (n, u)
        assert (2 if d64 else 1) * u["LDS Size [bytes/block]"] <= 160 * 1024, (n, u)
    _hazards("ringattn_split_steps.hip", tmp_path)
