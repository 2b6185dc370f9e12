"""Steps, merges and forwards of a plan whose first use they are, or that only forwards without tables in memory have warmed up, in a
stream capture: the plan's device tables are made then and there, and every replay gives the eager bits."""
import pytest
import torch

from ringattention_amd import api
from ringattention_amd.configs import Workload


def steps_and_merge(plan, t, o, l, out, lse):
    for s in range(plan.npes):
        plan.block_forward(s, t["q"], t["k"], t["v"], o[s], l[s])
    return plan.merge_ring(o, l, out, lse)


def rank_steps_and_merge(plan, t, o, l, out, lse, rank=2):
    for s in range(plan.npes):
        c = (rank + s) % plan.npes
        plan.rank_step_forward(rank, s, t["q_%d" % rank], t["k_%d" % c], t["v_%d" % c], o[s], l[s])
    return plan.rank_merge(rank, o, l, out, lse)


def whole_forward(plan, t, o, l, out, lse):
    return plan.forward(t["q"], t["k"], t["v"], out, lse)


@pytest.mark.gpu
@pytest.mark.parametrize("layout", ["contiguous", "zigzag"])
@pytest.mark.parametrize("warm", [True, False])
@pytest.mark.parametrize("work", [steps_and_merge, rank_steps_and_merge, whole_forward])
def test_capture_after_forwards_only(layout, warm, work):
    P, c, H, d = 4, 96, 2, 64
    S, rank = P * c, 2
    w = Workload("capture", 1, H, d, 1, S, "fp16", 77, True)
    t = dict(zip("qkv", (api.bits_to_tensor(x, w.dtype) for x in api.make_qkv_bits(w))))
    for r in range(P):
        for name in "qkv":
            t["%s_%d" % (name, r)] = t[name][:, :, r * c:(r + 1) * c].contiguous()
    rows = c if work is rank_steps_and_merge else S

    def buffers(plan):
        o_shape, l_shape = plan.rank_parts_shapes(rank) if work is rank_steps_and_merge else plan.parts_shapes()
        return (torch.zeros(o_shape, device="cuda"), torch.full(l_shape, float("-inf"), device="cuda"),
                torch.empty(1, H, rows, d, dtype=torch.float16, device="cuda"), torch.empty(1, H, rows, device="cuda"))

    make = lambda: api.RingAttention(P, c, d, 1, H, w.dtype, True, layout=layout)
    eager, plan = make(), make()
    try:
        out_e, lse_e = work(eager, t, *buffers(eager))
        if warm:
            plan.forward(t["q"], t["k"], t["v"])
        b = buffers(plan)
        torch.cuda.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            out, lse = work(plan, t, *b)
        for _ in range(3):
            for x in b[2:]:
                x.fill_(7.0)
            graph.replay()
            torch.cuda.synchronize()
            assert torch.equal(out, out_e) and torch.equal(lse, lse_e)
            plan.forward(t["q"], t["k"], t["v"])
            torch.cuda.synchronize()
    finally:
        eager.close()
        plan.close()
