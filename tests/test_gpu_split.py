"""ring_split_kernel (ringattn_split.hip: 32 query rows per workgroup, the keys split over its eight or sixteen waves) against the
CPU oracle where it can go wrong: fewer tiles than waves, one tile more or less than a round of eight, a last tile of one
key, rows of a tile that see nothing of a wave's first tile (causal), several key ranges (zigzag), grouped heads, heads
that the eight XCDs share unevenly, and logits that make every wave move its reference again and again.  Bounds: those of
test_gpu_parity.check_rows, which derive from the roundings of P and O to the storage type."""
import numpy as np
import pytest
import torch

from ringattention_amd import api
from ringattention_amd.configs import Workload
from test_gpu_parity import check_rows
from launched import launched
from test_gpu_walk64 import rising_logits
from test_kernel_resources import test_no_lds_transfer_reads_a_scalar_register_fresh_from_a_vector_instruction as _hazards
from test_kernel_resources import compile_to_asm


@pytest.mark.gpu
@pytest.mark.parametrize("d", [64, 128])
@pytest.mark.parametrize("lens,B,H,hkv,dtype,causal,zigzag,slope", [
    ((1,), 1, 1, 1, "fp16", True, False, 0),
    ((33,), 1, 2, 1, "bf16", False, False, 0),                    # a second tile of one key
    ((255, 1), 1, 1, 1, "fp16", False, False, 0),                 # eight tiles: one per wave
    ((257,), 2, 3, 3, "bf16", True, False, 0),                    # nine tiles; six heads over eight XCDs
    ((200, 313), 1, 9, 3, "fp16", True, False, 0),                # one head more than the XCDs, grouped
    ((130, 70, 2, 258), 1, 2, 2, "bf16", True, True, 0),          # two segments per rank, ranges of one tile and less
    ((640, 384), 1, 2, 2, "fp16", False, False, 0.3),             # the row maximum keeps climbing
    ((640, 385), 1, 2, 2, "bf16", True, False, 0.3),
    ((1024,), 1, 1, 1, "fp16", True, False, 4.0),                 # steep enough to overflow a stale reference
])
def test_split_kernel_against_oracle(oracle, monkeypatch, lens, B, H, hkv, dtype, causal, zigzag, slope, d):
    for name in ("RINGATTN_WIDE", "RINGATTN_WIDE_PARTIALS", "RINGATTN_SPLIT"):
        monkeypatch.delenv(name, raising=False)
    check_forward(oracle, lens, B, H, hkv, dtype, causal, zigzag, slope, d)


def check_forward(oracle, lens, B, H, hkv, dtype, causal, zigzag, slope, d):
    S = sum(lens)
    w = Workload("split", B, H, d, 1, S, dtype, 900 + S, causal)
    q, _, _ = rising_logits(w, slope) if slope else api.make_qkv_bits(w)
    wk = Workload("split_kv", B, hkv, d, 1, S, dtype, 1900 + S, causal)
    _, k, v = rising_logits(wk, slope) if slope else api.make_qkv_bits(wk)
    order = api.zigzag_order(lens) if zigzag else np.arange(S)
    inv = torch.from_numpy(np.argsort(order)).cuda()
    qd, kd, vd = (api.bits_to_tensor(np.ascontiguousarray(x[:, :, order]), dtype) for x in (q, k, v))
    plan = api.RingAttention(len(lens), list(lens), d, B, H, dtype, causal, kv_heads=hkv, layout="zigzag" if zigzag else "contiguous")
    try:
        assert plan.forward_kernel() == "ring_split_kernel"
        out_buf = torch.full((B * H * S + 64, d), 7.0, dtype=qd.dtype, device="cuda")
        lse_buf = torch.full((B * H * S + 64,), 7.0, dtype=torch.float32, device="cuda")
        out, lse = plan.forward(qd, kd, vd, out_buf[:B * H * S].view(B, H, S, d), lse_buf[:B * H * S].view(B, H, S))
        torch.cuda.synchronize()
    finally:
        plan.close()
    assert bool((out_buf[B * H * S:] == 7.0).all()) and bool((lse_buf[B * H * S:] == 7.0).all())
    k_full, v_full = (np.repeat(x, H // hkv, axis=1) for x in (k, v))
    check_rows(oracle, w, q, k_full, v_full, out[:, :, inv].contiguous(), lse[:, :, inv].contiguous(), np.arange(w.rows))


@pytest.mark.gpu
@pytest.mark.parametrize("lens,B,H,hkv,dtype,causal,zigzag,slope,forced", [
    ((1,), 1, 1, 1, "fp16", True, False, 0, True),                       # fifteen waves see nothing
    ((480,), 1, 2, 1, "bf16", False, False, 0, True),                    # fifteen tiles
    ((300, 212), 1, 2, 2, "fp16", True, False, 0, True),                 # sixteen: one per wave
    ((513,), 2, 3, 3, "fp16", False, False, 0, True),                    # a seventeenth tile of one key
    ((130, 70, 2, 258), 1, 2, 2, "bf16", True, True, 0, True),           # several ranges
    ((1024, 1025), 1, 1, 1, "fp16", True, False, 0.3, True),             # the row maximum keeps climbing
    ((1536, 1601), 1, 2, 1, "fp16", True, False, 0, False),              # 99 tiles, 198 workgroups: chosen without being asked
])
def test_split_kernel_with_sixteen_waves(oracle, monkeypatch, lens, B, H, hkv, dtype, causal, zigzag, slope, forced):
    for name in ("RINGATTN_WIDE", "RINGATTN_WIDE_PARTIALS", "RINGATTN_SPLIT"):
        monkeypatch.delenv(name, raising=False)
    if forced:
        monkeypatch.setenv("RINGATTN_SPLIT", "16")
    else:
        plan = api.RingAttention(len(lens), list(lens), 64, B, H, dtype, causal, kv_heads=hkv)
        x, kv = (torch.zeros(B, h, sum(lens), 64, dtype=torch.float16, device="cuda") for h in (H, hkv))
        out, lse = torch.empty_like(x), torch.empty(B, H, sum(lens), device="cuda")
        assert launched(lambda stream: plan.forward(x, kv, kv, out, lse, stream)) == [(1024, 0)]
        plan.close()
    check_forward(oracle, lens, B, H, hkv, dtype, causal, zigzag, slope, 64)


@pytest.mark.gpu
@pytest.mark.parametrize("lens,rank,causal,waves", [
    ((3137,), 0, True, 16),          # 99 tiles
    ((3072,), 0, False, 16),         # 96
    ((3040,), 0, False, 8),          # 95
    ((8192, 8192), 0, False, 16),    # 256 workgroups
    ((333, 11968), 0, False, 16),    # 385 tiles, the last of 13 keys
    ((12000, 300), 1, True, 16),     # 385 tiles, diagonal in the last ten
])
def test_how_many_waves_share_the_keys(oracle, monkeypatch, lens, rank, causal, waves):
    """d = 64: sixteen waves where a launch leaves no compute unit a second workgroup and the walk has 96 tiles or more.  The keys of
    a row then meet sixteen references instead of eight: the result is bit for bit that of the switch that asks for as many
    waves, and another than that of the other number."""
    for name in ("RINGATTN_WIDE", "RINGATTN_WIDE_D64", "RINGATTN_WIDE_PARTIALS", "RINGATTN_SPLIT", "RINGATTN_PAIR"):
        monkeypatch.delenv(name, raising=False)
    d, S, first, rows = 64, sum(lens), sum(lens[:rank]), lens[rank]
    w = Workload("waves", 1, 1, d, 1, S, "fp16", 4000 + S, causal)
    bits = api.make_qkv_bits(w)
    q, k, v = (api.bits_to_tensor(np.ascontiguousarray(x[0, 0]), w.dtype) for x in bits)
    q = q[first:first + rows].contiguous()
    out, lse = torch.zeros(S, d, dtype=q.dtype, device="cuda"), torch.zeros(S, device="cuda")

    def call(stream=None):
        api.ring_attention_noalloc(q, k, v, out[first:first + rows], len(lens), rank, lens, d, max(lens), lse=lse[first:first + rows],
                                   causal=causal, stream=stream)

    def result():
        call()
        torch.cuda.synchronize()
        return out.clone(), lse.clone()

    assert launched(call) == [(64 * waves, 0)]
    got, results = result(), {}
    for n in (8, 16):
        monkeypatch.setenv("RINGATTN_SPLIT", str(n))
        assert launched(call) == [(64 * n, 0)]
        results[n] = result()
    assert torch.equal(got[0], results[waves][0]) and torch.equal(got[1], results[waves][1])
    assert not torch.equal(got[0], results[24 - waves][0])
    some = first + np.unique(np.concatenate([np.arange(0, rows, max(1, rows // 100)), [rows - 1]]))
    check_rows(oracle, w, *bits, *got, some)


@pytest.mark.gpu
def test_eight_waves_where_two_workgroups_share_a_compute_unit(monkeypatch):
    for name in ("RINGATTN_WIDE", "RINGATTN_WIDE_D64", "RINGATTN_WIDE_PARTIALS", "RINGATTN_SPLIT", "RINGATTN_PAIR"):
        monkeypatch.delenv(name, raising=False)
    plan = api.RingAttention(1, 4096, 64, 1, 8, "fp16", True)   # 128 tiles, 1024 workgroups
    try:
        x = torch.zeros(1, 8, 4096, 64, dtype=torch.float16, device="cuda")
        out, lse = torch.empty_like(x), torch.empty(1, 8, 4096, device="cuda")
        assert plan.forward_kernel() == "ring_split_kernel"
        assert launched(lambda stream: plan.forward(x, x, x, out, lse, stream)) == [(512, 0)]
    finally:
        plan.close()


def test_split_kernel_resources_and_hazards(tmp_path):
    """Two waves per SIMD at d = 128, four (two workgroups per compute unit) at d = 64, no scratch; and the wait states in
    front of the direct-to-LDS loads."""
    _, usage = compile_to_asm("ringattn_split.hip", tmp_path / "split.s")
    kernels = {n: u for n, u in usage.items() if "ring_split_kernel" in n}
    assert len(kernels) == 6
    for n, u in kernels.items():
        d64 = "ELi64E" in n
        assert u["ScratchSize [bytes/lane]"] == 0, (n, u)
        assert u["VGPRs"] <= (128 if d64 else 256), (n, u)
        share = 2 if d64 and "ELi8E" in n else 1  # (sixteen waves at d = 64: one workgroup, four waves per SIMD)
        assert share * u["LDS Size [bytes/block]"] <= 160 * 1024, (n, u)
    _hazards("ringattn_split.hip", tmp_path)
