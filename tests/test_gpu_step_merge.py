"""The forward with the steps apart on ring_walk_kernel, which merges the partial of a step where it arises (ringattn_steps.hip; at d = 64
thin::ring_walk_kernel as well), where the walk from step to step can go wrong: one part and two, up to the 64 a plan may
have; a q tile that ends after one row, in the middle of a wave or exactly; chunks of less than a tile; rows that see only some of
the parts; the masked part last.  It is documented to give the bits of ringattn_block_fwd per step and
ringattn_merge_ring, whose merge kernel is other code: the bound is equality."""
import numpy as np
import pytest
import torch

from launched import launched
from ringattention_amd import api
from ringattention_amd.configs import Workload


@pytest.mark.gpu
@pytest.mark.parametrize("d,thin", [(64, False), (64, True), (128, False)])
@pytest.mark.parametrize("half", [False, True])
@pytest.mark.parametrize("lens,causal,zigzag", [
    ((257,), False, False),
    ((300, 41), False, False),
    ((129, 384), True, False),
    ((256, 1, 64), False, False),
    ((40,) * 8, True, False),
    ((300, 31) + (37,) * 7, False, False),
    ((33,) * 12 + (290,), True, False),
    ((64,) * 17, False, False),
    ((130, 70, 2, 258, 18) * 2, True, True),
    ((9,) * 63 + (321,), False, False),
    ((17,) * 64, True, False),
])
def test_forward_with_the_steps_apart_gives_the_bits_of_steps_and_merge(monkeypatch, lens, causal, zigzag, half, d, thin):
    monkeypatch.setenv("RINGATTN_WIDE_PARTIALS", "0")
    monkeypatch.setenv("RINGATTN_THIN", "1" if thin else "0")
    P, S, B, H = len(lens), sum(lens), 1, 3
    w = Workload("step_merge", B, H, d, 1, S, "fp16" if d == 128 else "bf16", 700 + S, causal)
    q, k, v = (api.bits_to_tensor(np.ascontiguousarray(x), w.dtype) for x in api.make_qkv_bits(w))
    plan = api.RingAttention(P, list(lens), d, B, H, w.dtype, causal, layout="zigzag" if zigzag else "contiguous",
                             step_partials=True, half_partials=half)
    try:
        assert plan.forward_kernel() == "ring_walk_kernel"
        out, lse = plan.forward(q, k, v)
        assert launched(lambda stream: plan.forward(q, k, v, out, lse, stream)) == [(256 if thin else 512, 0)]
        o_shape, l_shape = plan.parts_shapes()
        o_parts = torch.full(o_shape, float("nan"), dtype=plan.part_dtype, device="cuda")   # nobody may read what no step wrote
        l_parts = torch.full(l_shape, float("-inf"), dtype=torch.float32, device="cuda")
        for s in range(P):
            plan.block_forward(s, q, k, v, o_parts[s], l_parts[s])
        out_m, lse_m = plan.merge_ring(o_parts, l_parts)
        torch.cuda.synchronize()
    finally:
        plan.close()
    assert not torch.isnan(out).any()
    assert torch.equal(out, out_m) and torch.equal(lse, lse_m)
