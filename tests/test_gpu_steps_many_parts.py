"""The forward with the steps apart on ring_walk64_kernel where the LSEs of the steps leave its staged merge no room (more than 24
of them: merge_job_rows in ringattn_walk64.hip), and with one step less.  It is documented to give the bits of
ringattn_block_fwd per step and ringattn_merge_ring, whose merge kernel is other code: the bound is equality."""
import pytest
import torch

from ringattention_amd import api
from ringattention_amd.configs import Workload


@pytest.mark.gpu
@pytest.mark.parametrize("half", [False, True])
@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("ranks", [24, 25, 33, 64])
def test_bits_of_steps_and_merge(monkeypatch, ranks, causal, half):
    monkeypatch.delenv("RINGATTN_WIDE", raising=False)
    monkeypatch.setenv("RINGATTN_WIDE_PARTIALS", "1")
    w = Workload("many_parts", 1, 1, 128, ranks, 160, "bf16", 900 + ranks, causal)
    q, k, v = (api.bits_to_tensor(x, w.dtype) for x in api.make_qkv_bits(w))
    plan = api.RingAttention(ranks, w.chunk, w.dim, w.batch, w.heads, w.dtype, causal, step_partials=True, half_partials=half)
    try:
        assert plan.forward_kernel() == "ring_walk64_kernel"
        out, lse = plan.forward(q, k, v)
        o_shape, l_shape = plan.parts_shapes()
        o_parts = torch.full(o_shape, float("nan"), dtype=plan.part_dtype, device="cuda")   # nobody may read what no step wrote
        l_parts = torch.full(l_shape, float("-inf"), dtype=torch.float32, device="cuda")
        for s in range(ranks):
            plan.block_forward(s, q, k, v, o_parts[s], l_parts[s])
        out_m, lse_m = plan.merge_ring(o_parts, l_parts)
        torch.cuda.synchronize()
    finally:
        plan.close()
    assert not torch.isnan(out).any()
    assert torch.equal(out, out_m) and torch.equal(lse, lse_m)
