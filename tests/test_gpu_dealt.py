"""dealt::ring_walk_kernel (ringattn_dealt.hip) against ring_walk_kernel: the same operations on a row in the same order, so the bound is
equality of the partials, of steps of one rank and of all.  Sizes where its rounds of four tiles can go wrong: one tile, one tile less and
more than a round, than the rings of four rounds hold, tails of one key, q tiles that end early, diagonals, zigzag halves, references
that move in every tile, rows hidden in their first tiles, infinite scores; and which launches it is chosen for."""
import numpy as np
import pytest
import torch

from launched import launched
from ringattention_amd import api
from ringattention_amd.configs import Workload
from test_kernel_resources import compile_to_asm
from test_kernel_resources import test_no_lds_transfer_reads_a_scalar_register_fresh_from_a_vector_instruction as _hazards

SWITCHES = ("RINGATTN_WIDE", "RINGATTN_WIDE_PARTIALS", "RINGATTN_SPLIT", "RINGATTN_THIN", "RINGATTN_DEALT", "RINGATTN_SPLIT_STEPS")


@pytest.fixture(autouse=True)
def no_switches(monkeypatch):
    for name in SWITCHES:
        monkeypatch.delenv(name, raising=False)


def use(monkeypatch, kernel):
    monkeypatch.setenv("RINGATTN_SPLIT_STEPS", "0")
    monkeypatch.delenv("RINGATTN_THIN", raising=False)
    monkeypatch.delenv("RINGATTN_DEALT", raising=False)
    monkeypatch.setenv(*{"walk": ("RINGATTN_THIN", "0"), "dealt": ("RINGATTN_DEALT", "1")}[kernel])


@pytest.mark.gpu
@pytest.mark.parametrize("half,by_rows", [(False, False), (True, False), (False, True), (True, True)])
@pytest.mark.parametrize("lens,causal,zigzag,kind", [
    ((1,), False, False, "flat"),
    ((32, 33, 31), False, False, "flat"),
    ((65, 128, 160, 161), True, False, "flat"),              # a round, and one tile more
    ((96, 480, 512, 513, 544), False, False, "flat"),         # four rounds, one tile less and more
    ((513, 1100), True, False, "rising"),
    ((1000, 24), False, False, "steep"),
    ((320, 256, 192), True, True, "rising"),
    ((130, 70, 2, 258), True, True, "flat"),
    ((300, 200), False, False, "hidden"),
    ((700, 300), True, False, "hidden"),
    ((400, 161), False, False, "infinite"),
])
def test_bits_of_ring_walk_kernel(monkeypatch, lens, causal, zigzag, kind, half, by_rows):
    P, S, B, H, hkv, d = len(lens), sum(lens), 2, 4, 2, 64
    at = np.concatenate(([0], np.cumsum(lens)))
    for dtype in ("fp16", "bf16"):
        q = api.bits_to_tensor(api.make_qkv_bits(Workload("dealt", B, H, d, 1, S, dtype, 2200 + S, causal))[0], dtype)
        k, v = (api.bits_to_tensor(x, dtype) for x in api.make_qkv_bits(Workload("dealt", B, hkv, d, 1, S, dtype, 2300 + S, causal))[1:])
        if kind in ("rising", "steep"):   # scores grow along the sequence, beyond fp16's range of exponentials in between
            ramp = torch.arange(S, device="cuda", dtype=torch.float32) * (0.02 if kind == "rising" else 0.2)
            q[..., 0] = 8.0
            k[..., 0] = ramp.to(k.dtype)
        if kind == "hidden":              # no finite score in the first 70 keys of a chunk
            q[..., 0] = 1.0
            for a in at[:-1]:
                k[:, :, a:a + 70, 0] = float("-inf")
        if kind == "infinite":            # a score of +inf in the middle of a round, one of NaN further on
            q[..., 0] = 1.0
            k[:, :, 45, 0] = float("inf")
            k[:, :, 300, 0] = float("nan")
        results = []
        for kernel in ("walk", "dealt"):
            use(monkeypatch, kernel)
            plan = api.RingAttention(P, list(lens), d, B, H, dtype, causal, kv_heads=hkv, layout="zigzag" if zigzag else "contiguous",
                                     half_partials=half, row_partials=by_rows)
            parts = []
            o_shape, l_shape = plan.parts_shapes()
            o = torch.full(o_shape, 7.0, dtype=plan.part_dtype, device="cuda")
            l = torch.full(l_shape, 7.0, dtype=torch.float32, device="cuda")
            at_step = (lambda x, s: x) if by_rows else (lambda x, s: x[s])
            for s in range(P):
                plan.block_forward(s, q, k, v, at_step(o, s), at_step(l, s))
            parts += [o, l]
            for r in range(P):
                o_shape, l_shape = plan.rank_parts_shapes(r)
                o = torch.full(o_shape, 7.0, dtype=plan.part_dtype, device="cuda")
                l = torch.full(l_shape, 7.0, dtype=torch.float32, device="cuda")
                own = q[:, :, at[r]:at[r + 1]].contiguous()
                for s in range(P):
                    j = (r + s) % P
                    plan.rank_step_forward(r, s, own, k[:, :, at[j]:at[j + 1]].contiguous(), v[:, :, at[j]:at[j + 1]].contiguous(),
                                           at_step(o, s), at_step(l, s))
                parts += [o, l]
            threads = 384 if kernel == "dealt" else 512
            o, l = parts[0], parts[1]
            assert [t for t, _ in launched(lambda stream: plan.block_forward(0, q, k, v, at_step(o, 0), at_step(l, 0), stream))] == [threads]
            torch.cuda.synchronize()
            plan.close()
            results.append(parts)
        for x, y in zip(*results):
            ints = torch.int32 if x.dtype == torch.float32 else torch.int16
            nan = torch.isnan(x)          # (which NaN is nobody's promise)
            assert torch.equal(nan, torch.isnan(y)) and torch.equal(x.view(ints)[~nan], y.view(ints)[~nan]), dtype


@pytest.mark.gpu
@pytest.mark.parametrize("tokens,heads,step,threads", [
    (1024, 8, 1, 384),     # 256 q tiles of 32 rows
    (1024, 9, 1, 256),     # thin::ring_walk_kernel
    (353, 8, 1, 384),      # twelve tiles
    (352, 8, 1, 256),
    (97, 8, 0, 384),       # four, under the diagonal
    (96, 8, 0, 256),
    (1024, 16, 0, 384),    # 512 under the diagonal
    (1056, 16, 0, 256),
    (512, 16, 0, 384),     # 256
    (512, 17, 0, 256),     # 272 of sixteen tiles
    (544, 16, 0, 384),     # 272 of seventeen
    (223, 64, 0, 256),     # 448 of seven
])
def test_which_launches_it_is_chosen_for(monkeypatch, tokens, heads, step, threads):
    monkeypatch.setenv("RINGATTN_SPLIT_STEPS", "0")
    x = torch.zeros(1, heads, tokens, 64, dtype=torch.float16, device="cuda")
    plan = api.RingAttention(2, tokens, 64, 1, heads, "fp16", step == 0)
    o, l = plan.rank_step_forward(0, step, x, x, x)
    assert [t for t, _ in launched(lambda stream: plan.rank_step_forward(0, step, x, x, x, o, l, stream))] == [threads]
    plan.close()


def test_resources_and_hazards(tmp_path):
    """One workgroup on a compute unit, no scratch; and the wait states in front of the direct-to-LDS loads."""
    _, usage = compile_to_asm("ringattn_dealt.hip", tmp_path / "dealt.s")
    found = {n: u for n, u in usage.items() if "ring_walk_kernel" in n}
    assert len(found) == 4
    for n, u in found.items():
        assert u["ScratchSize [bytes/lane]"] == 0, (n, u)
        assert u["VGPRs"] <= 256, (n, u)
        assert u["LDS Size [bytes/block]"] <= 160 * 1024, (n, u)
    _hazards("ringattn_dealt.hip", tmp_path)
