"""thin::ring_walk_kernel (ringattn_thin.hip) against ring_walk_kernel: the same operations on a row in the same order, so the bound is
equality -- of the partials of single steps and of the forward with the steps merged.  Sizes where its pipeline can go wrong: one
tile, fewer and more than its rings hold, tails of one key, q tiles that end early, diagonals, references that move in
every tile, rows hidden in their first tiles.  And which launches it is chosen for is invisible but in time."""
import numpy as np
import pytest
import torch

from launched import launched
from ringattention_amd import api
from ringattention_amd.configs import Workload


@pytest.mark.gpu
@pytest.mark.parametrize("half", [False, True])
@pytest.mark.parametrize("lens,causal,zigzag,kind", [
    ((1,), False, False, "flat"),
    ((32, 33, 31), False, False, "flat"),
    ((65, 128, 160, 161), True, False, "flat"),
    ((224, 225, 256, 257, 288, 289), False, False, "flat"),   # 7, 8 and 9 tiles: the rings, one less, one more
    ((513, 480), True, False, "rising"),
    ((1000, 24), False, False, "steep"),
    ((320, 256, 192), True, True, "rising"),
    ((300, 200), False, False, "hidden"),
    ((700, 300), True, False, "hidden"),
])
def test_bits_of_ring_walk_kernel(monkeypatch, lens, causal, zigzag, kind, half):
    for name in ("RINGATTN_WIDE", "RINGATTN_WIDE_PARTIALS", "RINGATTN_THIN"):
        monkeypatch.delenv(name, raising=False)
    P, S, B, H, d = len(lens), sum(lens), 1, 3, 64
    for dtype in ("fp16", "bf16"):
        w = Workload("thin", B, H, d, 1, S, dtype, 1200 + S, causal)
        q, k, v = (api.bits_to_tensor(np.ascontiguousarray(x), w.dtype) for x in api.make_qkv_bits(w))
        if kind in ("rising", "steep"):   # scores grow along the sequence, beyond fp16's range of exponentials in between
            ramp = torch.arange(S, device="cuda", dtype=torch.float32) * (0.02 if kind == "rising" else 0.2)
            q[..., 0] = 8.0
            k[..., 0] = ramp.to(k.dtype)
        if kind == "hidden":              # no finite score in the first 70 keys of a chunk
            q[..., 0] = 1.0
            at = np.concatenate(([0], np.cumsum(lens)))[:-1]
            for a in at:
                k[:, :, a:a + 70, 0] = float("-inf")
        results = []
        for choice in ("0", "1"):
            monkeypatch.setenv("RINGATTN_THIN", choice)
            plan = api.RingAttention(P, list(lens), d, B, H, dtype, causal, layout="zigzag" if zigzag else "contiguous",
                                     step_partials=True, half_partials=half)
            out, lse = plan.forward(q, k, v)
            o_shape, l_shape = plan.parts_shapes()
            o_parts = torch.full(o_shape, 7.0, dtype=plan.part_dtype, device="cuda")
            l_parts = torch.full(l_shape, 7.0, dtype=torch.float32, device="cuda")
            for s in range(P):
                plan.block_forward(s, q, k, v, o_parts[s], l_parts[s])
            threads = 256 if choice == "1" else 512
            assert [t for t, _ in launched(lambda stream: plan.forward(q, k, v, out, lse, stream))] == [threads]
            assert [t for t, _ in launched(lambda stream: plan.block_forward(0, q, k, v, o_parts[0], l_parts[0], stream))] == [threads]
            torch.cuda.synchronize()
            plan.close()
            results.append((out, lse, o_parts, l_parts))
        for x, y in zip(*results):
            ints = torch.int32 if x.dtype == torch.float32 else torch.int16
            assert torch.equal(x.view(ints), y.view(ints)), dtype


@pytest.mark.gpu
@pytest.mark.parametrize("d,tokens,heads,thin", [
    (64, 512, 64, True),     # 128 q tiles of 256 rows in all
    (64, 512, 66, False),
    (64, 257, 64, True),     # as many, the second of a head one row long
    (128, 512, 2, False),
])
def test_which_launches_it_is_chosen_for(monkeypatch, d, tokens, heads, thin):
    for name in ("RINGATTN_WIDE", "RINGATTN_WIDE_PARTIALS", "RINGATTN_THIN"):
        monkeypatch.delenv(name, raising=False)
    x = torch.zeros(1, heads, 2 * tokens, d, dtype=torch.float16, device="cuda")
    own = x[:, :, :tokens].contiguous()
    plan = api.RingAttention(2, tokens, d, 1, heads, "fp16")
    o, l = plan.rank_step_forward(0, 1, own, own, own)
    assert [t for t, _ in launched(lambda stream: plan.rank_step_forward(0, 1, own, own, own, o, l, stream))] == [256 if thin else 512]
    plan.close()
    if heads % 2 == 0:   # two ranks of half as many heads are as many q tiles
        half = x[:, :heads // 2].contiguous()
        plan = api.RingAttention(2, tokens, d, 1, heads // 2, "fp16", step_partials=True)
        out, lse = plan.forward(half, half, half)
        assert [t for t, _ in launched(lambda stream: plan.forward(half, half, half, out, lse, stream))] == [256 if thin else 512]
        plan.close()
