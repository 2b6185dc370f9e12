"""columns::ring_split_kernel (ringattn_split_columns.hip): 64 or 32 columns of V and O in a workgroup.  The columns of a row do not meet, so
its results are bit for bit those of the form with all columns (which the other tests hold to the oracle): forwards that carry the
state, calls of one rank, and single steps.  Sizes where it can go wrong: one row, tails of one key, fewer tiles than waves, walks of many
tiles, grouped heads over the XCDs, several ranges (zigzag), masked steps, both partial types and layouts."""
import pytest
import torch

from launched import kernels
from ringattention_amd import api
from test_kernel_resources import compile_to_asm
from test_kernel_resources import test_no_lds_transfer_reads_a_scalar_register_fresh_from_a_vector_instruction as _hazards

SWITCHES = ("RINGATTN_WIDE", "RINGATTN_WIDE_D64", "RINGATTN_WIDE_PARTIALS", "RINGATTN_SPLIT", "RINGATTN_PAIR", "RINGATTN_THIN",
            "RINGATTN_SPLIT_STEPS", "RINGATTN_SPLIT_COLUMNS")


@pytest.fixture(autouse=True)
def no_switches(monkeypatch):
    for name in SWITCHES:
        monkeypatch.delenv(name, raising=False)


def same_bits(monkeypatch, call, outs, dim):
    """call(stream) with all columns, 64 and 32: other kernels, the same bits, nothing behind the outputs."""
    seen, first = set(), None
    for columns in ([128] if dim == 128 else []) + [64, 32]:
        monkeypatch.setenv("RINGATTN_SPLIT_COLUMNS", str(columns))
        seen.update(kernels(call))
        for t in outs:
            t.fill_(7.0)
        call()
        torch.cuda.synchronize()
        got = [t.clone() for t in outs]
        first = first or got
        for a, b in zip(first, got):
            assert torch.equal(a.view(torch.int16), b.view(torch.int16))
            assert bool((a[-64:] == 7.0).all())
    assert len(seen) == (3 if dim == 128 else 2)


def tensors(dim, dtype, *shapes):
    gen = torch.Generator(device="cuda").manual_seed(sum(s[-1] for s in shapes) + dim)
    return [torch.randn(*s, dim, generator=gen, device="cuda", dtype=dtype) for s in shapes]


def padded(shape, dtype):
    n = 1
    for x in shape:
        n *= x
    buf = torch.empty(n + 64, dtype=dtype, device="cuda")
    return buf, buf[:n].view(shape)


@pytest.mark.gpu
@pytest.mark.parametrize("dim,waves", [(64, 8), (64, 16), (128, 8)])
@pytest.mark.parametrize("lens,B,H,hkv,dtype,causal,zigzag", [
    ((1,), 1, 1, 1, torch.float16, True, False),
    ((33,), 1, 2, 1, torch.bfloat16, False, False),
    ((255, 2), 2, 3, 3, torch.bfloat16, True, False),
    ((200, 313), 1, 9, 3, torch.float16, True, False),
    ((130, 70, 2, 258), 1, 2, 2, torch.bfloat16, True, True),
    ((1500, 1537), 1, 1, 1, torch.float16, False, False),
])
def test_forward(monkeypatch, lens, B, H, hkv, dtype, causal, zigzag, waves, dim):
    monkeypatch.setenv("RINGATTN_SPLIT", str(waves))
    S = sum(lens)
    q, k, v = tensors(dim, dtype, (B, H, S), (B, hkv, S), (B, hkv, S))
    (o_buf, out), (l_buf, lse) = padded((B, H, S, dim), dtype), padded((B, H, S), torch.float32)
    plan = api.RingAttention(len(lens), list(lens), dim, B, H, {torch.float16: "fp16", torch.bfloat16: "bf16"}[dtype], causal, kv_heads=hkv,
                             layout="zigzag" if zigzag else "contiguous")
    try:
        same_bits(monkeypatch, lambda stream=None: plan.forward(q, k, v, out, lse, stream), [o_buf, l_buf], dim)
    finally:
        plan.close()


@pytest.mark.gpu
@pytest.mark.parametrize("dim", [64, 128])
@pytest.mark.parametrize("lens,rank,causal", [((640, 512, 384, 511), 3, True), ((7, 4090), 0, False)])
def test_call_of_one_rank(monkeypatch, lens, rank, causal, dim):
    monkeypatch.setenv("RINGATTN_SPLIT", "8")
    rows, S = lens[rank], sum(lens)
    q, k, v = tensors(dim, torch.bfloat16, (rows,), (S,), (S,))
    o_buf, out = padded((rows, dim), torch.bfloat16)
    same_bits(monkeypatch, lambda stream=None: api.ring_attention_noalloc(q, k, v, out, len(lens), rank, lens, dim, max(lens), causal=causal,
                                                                          stream=stream), [o_buf], dim)


@pytest.mark.gpu
@pytest.mark.parametrize("half,by_rows", [(False, False), (True, False), (False, True)])
@pytest.mark.parametrize("dim", [64, 128])
@pytest.mark.parametrize("lens,causal,zigzag,rank,step", [
    ((128, 129, 31), False, False, 0, 1),
    ((256, 257, 255), True, False, 1, 0),
    ((300, 222), True, True, 0, 1),
    ((514, 40), True, True, 0, 0),
])
def test_step_of_one_rank(monkeypatch, lens, causal, zigzag, rank, step, dim, half, by_rows):
    monkeypatch.setenv("RINGATTN_SPLIT_STEPS", "1")
    P, H = len(lens), 3
    n, m = lens[rank], lens[(rank + step) % P]
    q, k, v = tensors(dim, torch.float16, (1, H, n), (1, H, m), (1, H, m))
    plan = api.RingAttention(P, list(lens), dim, 1, H, "fp16", causal, layout="zigzag" if zigzag else "contiguous", half_partials=half,
                             row_partials=by_rows)
    o_shape, l_shape = plan.rank_parts_shapes(rank) if by_rows else ((1, H, n, dim), (1, H, n))
    (o_buf, o), (l_buf, l) = padded(o_shape, plan.part_dtype), padded(l_shape, torch.float32)
    try:
        same_bits(monkeypatch, lambda stream=None: plan.rank_step_forward(rank, step, q, k, v, o, l, stream), [o_buf, l_buf], dim)
    finally:
        plan.close()


@pytest.mark.gpu
@pytest.mark.parametrize("dim,tokens,columns", [(128, 1024, 32), (128, 1025, 64), (128, 4096, 64), (64, 3072, 32), (64, 3073, 64)])
def test_how_many_columns(monkeypatch, dim, tokens, columns):
    """The lines of split_columns: row tiles of 32, one head."""
    monkeypatch.setenv("RINGATTN_SPLIT", "8")
    q, k, v = tensors(dim, torch.float16, (1, 1, tokens), (1, 1, tokens), (1, 1, tokens))
    out, lse = torch.empty_like(q), torch.empty(1, 1, tokens, device="cuda")
    plan = api.RingAttention(1, tokens, dim, 1, 1, "fp16", False)
    try:
        chosen = kernels(lambda stream: plan.forward(q, k, v, out, lse, stream))
        monkeypatch.setenv("RINGATTN_SPLIT_COLUMNS", str(columns))
        assert kernels(lambda stream: plan.forward(q, k, v, out, lse, stream)) == chosen
    finally:
        plan.close()


@pytest.mark.gpu
@pytest.mark.parametrize("kind", ["forward", "call", "step", "block"])
@pytest.mark.parametrize("dim", [64, 128])
def test_results_over_q(monkeypatch, dim, kind):
    """O, or fp16 partials, written over Q: a row of Q is read by the workgroup that writes it, so all columns are its own."""
    H, S = (1 if kind == "call" else 3), 300
    (q, k, v), lse = tensors(dim, torch.float16, *[(S,) if kind == "call" else (1, H, S)] * 3), torch.empty(1, H, S, device="cuda")
    plan = api.RingAttention(1, S, dim, 1, H, "fp16", True, half_partials=True)
    call = {
        "forward": lambda q, out, stream=None: plan.forward(q, k, v, out, lse, stream),
        "call": lambda q, out, stream=None: api.ring_attention_noalloc(q, k, v, out, 1, 0, [S], dim, S, causal=True, stream=stream),
        "step": lambda q, out, stream=None: plan.rank_step_forward(0, 0, q, k, v, out, lse, stream),
        "block": lambda q, out, stream=None: plan.block_forward(0, q, k, v, out, lse, stream),
    }[kind]
    monkeypatch.setenv(*(("RINGATTN_SPLIT", "8") if kind in ("forward", "call") else ("RINGATTN_SPLIT_STEPS", "1")))
    out = torch.empty_like(q)
    try:
        some, over = kernels(lambda stream: call(q, out, stream)), kernels(lambda stream: call(q, q, stream))
        monkeypatch.setenv("RINGATTN_SPLIT_COLUMNS", "32")
        assert kernels(lambda stream: call(q, out, stream)) == some != over and kernels(lambda stream: call(q, q, stream)) == over
        monkeypatch.setenv("RINGATTN_SPLIT_COLUMNS", "128")
        assert kernels(lambda stream: call(q, out, stream)) == over
        call(q, out)
        monkeypatch.delenv("RINGATTN_SPLIT_COLUMNS")
        call(q, q)
        torch.cuda.synchronize()
        assert torch.equal(q.view(torch.int16), out.view(torch.int16))
    finally:
        plan.close()


def test_resources_and_hazards(tmp_path):
    """Two waves per SIMD at d = 128, four at d = 64 (two workgroups of eight waves on a compute unit), no scratch; and the wait states
    in front of the direct-to-LDS loads."""
    _, usage = compile_to_asm("ringattn_split_columns.hip", tmp_path / "columns.s")
    found = {n: u for n, u in usage.items() if "ring_split_kernel" in n}
    assert len(found) == 20   # two types: d = 64 carried with 8 and 16 waves, partials in two types; d = 128 twice, with 8 waves
    for n, u in found.items():
        d64 = "ELi64ELi32E" in n
        assert u["ScratchSize [bytes/lane]"] == 0, (n, u)
        assert u["VGPRs"] <= (128 if d64 else 256), (n, u)
        assert u["LDS Size [bytes/block]"] <= 160 * 1024, (n, u)
    _hazards("ringattn_split_columns.hip", tmp_path)
