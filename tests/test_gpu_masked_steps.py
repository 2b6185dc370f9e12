"""Single ring steps at d = 64 on ring_walk_kernel, two workgroups of which a compute unit holds: launches that keep to one at a time, and
those whose second lap of workgroups runs in reverse (ringattn_walk.hip).  The order says nothing about a row: the bound
is equality, with the same step on thin::ring_walk_kernel, which gives the same bits in another order.  Sizes: around one and
two laps of the eight XCDs (256 and 512 workgroups), heads that the XCDs share, several segments, q tiles that end early."""
import pytest
import torch

from launched import launched
from ringattention_amd import api


@pytest.fixture(autouse=True)
def no_switches(monkeypatch):
    for name in ("RINGATTN_WIDE", "RINGATTN_WIDE_PARTIALS", "RINGATTN_THIN"):
        monkeypatch.delenv(name, raising=False)


@pytest.mark.gpu
@pytest.mark.parametrize("half", [False, True])
@pytest.mark.parametrize("lens,heads,zigzag", [
    ((2048, 40), 31, False),     # 248 workgroups, one at a time
    ((2020, 40), 33, False),     # a compute unit too few
    ((2017, 40), 51, False),     # the second lap in reverse, three heads that the XCDs share; a q tile of 225 rows
    ((2300, 40), 50, False),     # nine q tiles a head
    ((2048, 40), 64, False),     # both laps full
    ((2048, 40), 65, False),     # a third begins
    ((2100, 40), 75, False),
    ((520, 100), 107, False),    # short walks: as they come
    ((1000, 2100), 33, True),    # two segments a rank in the steps that follow
])
def test_every_row_of_a_masked_step(monkeypatch, lens, heads, zigzag, half):
    gen = torch.Generator(device="cuda").manual_seed(heads)
    q, k, v = (torch.randn(1, heads, sum(lens), 64, generator=gen, device="cuda").half() for _ in range(3))
    results = []
    for thin in ("0", "1"):
        monkeypatch.setenv("RINGATTN_THIN", thin)
        plan = api.RingAttention(len(lens), list(lens), 64, 1, heads, "fp16", True, layout="zigzag" if zigzag else "contiguous",
                                 half_partials=half)
        o = torch.full(q.shape, float("nan"), dtype=plan.part_dtype, device="cuda")
        l = torch.full(q.shape[:3], float("nan"), device="cuda")
        plan.block_forward(0, q, k, v, o, l)
        o_1, l_1 = torch.zeros_like(o), torch.zeros_like(l)
        plan.block_forward(1, q, k, v, o_1, l_1)
        first = slice(0, lens[0])
        rank = [x[:, :, first].contiguous() for x in (q, k, v)]
        o_r, l_r = (torch.full_like(x[:, :, first].contiguous(), float("nan")) for x in (o, l))
        plan.rank_step_forward(0, 0, *rank, o_r, l_r)
        torch.cuda.synchronize()
        plan.close()
        assert torch.equal(o_r, o[:, :, first]) and torch.equal(l_r, l[:, :, first])
        results.append((o, l, o_1, l_1))
    for x, y in zip(*results):
        assert torch.equal(x, y)   # (a NaN is unequal to itself: every row is written)


def more_lds_of_a_step(lens, heads, step, zigzag=False, rank=None):
    plan = api.RingAttention(len(lens), list(lens), 64, 1, heads, "fp16", True, layout="zigzag" if zigzag else "contiguous")
    rows = sum(lens) if rank is None else lens[rank]
    x = torch.zeros(1, heads, rows, 64, dtype=torch.float16, device="cuda")
    o, l = torch.empty(x.shape, device="cuda"), torch.empty(x.shape[:3], device="cuda")

    def call(stream=None):
        if rank is None:
            plan.block_forward(step, x, x, x, o, l, stream)
        else:
            plan.rank_step_forward(rank, step, x, x, x, o, l, stream)

    call()   # (makes the plan's tables)
    (threads, more_lds), = launched(call)
    plan.close()
    assert threads == 512
    return more_lds


@pytest.mark.gpu
@pytest.mark.parametrize("tokens,heads,step,alone", [
    (2048, 32, 0, True),     # 256 workgroups: as many as compute units
    (2048, 50, 0, True),     # 400
    (2048, 51, 0, False),
    (1024, 72, 0, True),     # 288 of shorter walks
    (1024, 73, 0, False),
    (512, 130, 0, False),    # 260 of still shorter ones
    (2048, 33, 1, False),    # walks of one length
])
def test_few_workgroups_of_a_rank_run_one_at_a_time(tokens, heads, step, alone):
    assert (more_lds_of_a_step((tokens, tokens), heads, step, rank=1) > 0) == alone


@pytest.mark.gpu
@pytest.mark.parametrize("lens,heads,step,zigzag,alone", [
    ((1024,) * 8, 11, 1, True, True),      # 198 workgroups in a grid of 352
    ((4096,) * 4, 8, 1, True, True),       # 320, of two lengths
    ((4096,) * 4, 11, 1, True, False),     # 440
    ((2048,) * 4, 11, 0, False, True),     # 352 of the masked step of all ranks
    ((2048,) * 8, 6, 0, False, False),     # 384
    ((2048, 256, 256, 256), 20, 0, False, True),   # 220 in a grid of 640
])
def test_few_workgroups_of_all_ranks_run_one_at_a_time(lens, heads, step, zigzag, alone):
    assert (more_lds_of_a_step(lens, heads, step, zigzag) > 0) == alone
