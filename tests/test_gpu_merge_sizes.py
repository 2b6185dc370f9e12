"""merge_kernel with a batch of parts ahead (more than 256 MiB of parts) and without: the same operations on a row in the same order, so
the bound is equality, of the rows of a large merge with merges of few rows.  One part to several batches, none of them
whole but by chance; rows without any visible key among them."""
import pytest
import torch

from launched import kernels
from ringattention_amd import api

LINE = 256 << 20   # bytes of parts


def parts(shape, dtype, seed):
    gen = torch.Generator(device="cuda").manual_seed(seed)
    o = torch.randn(shape, generator=gen, device="cuda", dtype=dtype)
    l = torch.randn(shape[:-1], generator=gen, device="cuda") * 4
    hidden = torch.rand(shape[:-1], generator=gen, device="cuda") < 0.1
    hidden[..., 5] = True
    return o.masked_fill_(hidden[..., None], float("nan")), l.masked_fill_(hidden, float("-inf"))


@pytest.mark.gpu
@pytest.mark.parametrize("d", [64, 128])
@pytest.mark.parametrize("n", [1, 3, 4, 5, 8, 9, 17, 64])
def test_merge_of_many_rows(n, d):
    rows = LINE // (n * (d * 4 + 4)) + 3
    o, l = parts((n, rows, d), torch.float32, n)
    out, lse = api.merge(o, l, "fp16")
    some = rows // 3
    few = [x[:, :some].contiguous() for x in (o, l)]
    assert kernels(lambda s: api.merge(o, l, "fp16", s)) != kernels(lambda s: api.merge(*few, "fp16", s))
    for a, b in ((0, 1001), (some, some + 777), (rows - 99, rows)):
        out_s, lse_s = api.merge(o[:, a:b].contiguous(), l[:, a:b].contiguous(), "fp16")
        assert torch.equal(out[a:b], out_s) and torch.equal(lse[a:b], lse_s)
    assert not torch.isnan(out).any() and bool((lse[5] == float("-inf")).all()) and bool((out[5] == 0).all())


@pytest.mark.gpu
@pytest.mark.parametrize("half,rows_first,d", [(False, False, 64), (True, False, 128), (True, True, 64), (False, True, 128)])
def test_merge_of_all_ranks_and_of_one(half, rows_first, d):
    P, causal = 5, True
    chunk = LINE // (15 * (d * (2 if half else 4) + 4)) + 7   # fifteen of the 25 pairs of ranks are visible
    plan = api.RingAttention(P, chunk, d, 1, 1, "bf16", causal, half_partials=half, row_partials=rows_first)
    o, l = parts((P, 1, 1, P * chunk, d), plan.part_dtype, d)
    if rows_first:
        o, l = (x.movedim(0, 3).contiguous() for x in (o, l))
    out, lse = plan.merge_ring(o, l)
    for rank in (0, 2, 4):
        own = slice(rank * chunk, (rank + 1) * chunk)
        o_r, l_r = ((x[:, :, own] if rows_first else x[:, :, :, own]).contiguous() for x in (o, l))
        out_r, lse_r = plan.rank_merge(rank, o_r, l_r)
        assert torch.equal(out[:, :, own], out_r) and torch.equal(lse[:, :, own], lse_r)
        if rank == 0:
            assert kernels(lambda s: plan.merge_ring(o, l, out, lse, s)) != kernels(lambda s: plan.rank_merge(0, o_r, l_r, out_r, lse_r, s))
    plan.close()


@pytest.mark.gpu
@pytest.mark.parametrize("d", [64, 128])
def test_rows_whose_lses_are_no_numbers(d):
    """A row without any finite LSE has seen nothing: O = 0, LSE = -inf, whether its LSEs are -inf or NaN; one NaN next to a finite LSE
    makes both NaN, whichever comes first."""
    inf, nan = float("inf"), float("nan")
    nothing = [(-inf, -inf, -inf), (nan, nan, nan), (nan, -inf, nan), (-inf, nan, -inf)]
    broken = [(nan, 0.5, 0.25), (0.5, nan, -inf), (-inf, 0.5, nan), (nan, -inf, 0.5)]
    l = torch.tensor(nothing + broken, device="cuda").T.contiguous()
    o = torch.randn(3, 8, d, device="cuda")
    plan = api.RingAttention(3, [8, 2, 2], d, 1, 1, "fp16")   # (the rows of its first rank)
    o_parts, l_parts = torch.zeros(3, 1, 1, 12, d, device="cuda"), torch.zeros(3, 1, 1, 12, device="cuda")
    o_parts[:, 0, 0, :8], l_parts[:, 0, 0, :8] = o, l
    ring = [x[0, 0, :8] for x in plan.merge_ring(o_parts, l_parts)]
    rank = [x[0, 0] for x in plan.rank_merge(0, o[:, None, None].contiguous(), l[:, None, None].contiguous())]
    for out, lse in (api.merge(o, l, "fp16"), ring, rank):
        assert bool((out[:4] == 0).all()) and bool((lse[:4] == -inf).all())
        assert bool(out[4:].isnan().all()) and bool(lse[4:].isnan().all())
    plan.close()
