"""The place of a workgroup in launches of no more workgroups than compute units (job_grid, decode_job): on both sides of the line in
number, for head counts that divide the XCDs, are multiples of them, or neither, masked and not, with two segments per rank, results
against float64; every row is written, and nothing behind the outputs."""
import numpy as np
import pytest
import torch

from ringattention_amd import api
from ringattention_amd.configs import Workload
from test_gpu_parity import check_rows


@pytest.mark.gpu
@pytest.mark.parametrize("d,H,lens,causal,zigzag,switch", [
    (64, 1, (256 * 32,), False, False, None),                    # 256 workgroups of ring_split_kernel
    (64, 1, (255 * 32 + 2, 2), True, False, ("RINGATTN_SPLIT", "8")),
    (64, 1, (256 * 32 + 1,), False, False, ("RINGATTN_SPLIT", "8")),   # 257
    (128, 8, (1000, 24), True, False, ("RINGATTN_SPLIT", "8")),   # 32 a head
    (128, 8, (1025,), True, False, ("RINGATTN_SPLIT", "8")),      # 33
    (64, 3, (300, 200), True, False, None),                      # 3 heads: as before
    (64, 16, (200, 312), False, False, None),
    (64, 4, (200, 312), True, True, ("RINGATTN_SPLIT", "8")),      # segments of 100 and 156 rows
    (128, 16, (768, 1280), True, False, ("RINGATTN_PAIR", "1")),
    (64, 32, (1024, 1024), False, False, ("RINGATTN_PAIR", "0")),  # 256 of ring_walk64_kernel
])
def test_every_row_is_found(oracle, monkeypatch, d, H, lens, causal, zigzag, switch):
    for name in ("RINGATTN_WIDE", "RINGATTN_WIDE_D64", "RINGATTN_WIDE_PARTIALS", "RINGATTN_SPLIT", "RINGATTN_PAIR", "RINGATTN_SPLIT_COLUMNS"):
        monkeypatch.delenv(name, raising=False)
    if switch:
        monkeypatch.setenv(*switch)
    S = sum(lens)
    w = Workload("few", 1, H, d, 1, S, "fp16", 3100 + S + H, causal)
    bits = api.make_qkv_bits(w)
    order = api.zigzag_order(lens) if zigzag else np.arange(S)
    inv = torch.from_numpy(np.argsort(order)).cuda()
    q, k, v = (api.bits_to_tensor(np.ascontiguousarray(x[:, :, order]), "fp16") for x in bits)
    o_buf = torch.full((H * S + 64, d), 7.0, dtype=q.dtype, device="cuda")
    l_buf = torch.full((H * S + 64,), 7.0, device="cuda")
    plan = api.RingAttention(len(lens), list(lens), d, 1, H, "fp16", causal, layout="zigzag" if zigzag else "contiguous")
    try:
        out, lse = plan.forward(q, k, v, o_buf[:H * S].view(1, H, S, d), l_buf[:H * S].view(1, H, S))
        torch.cuda.synchronize()
    finally:
        plan.close()
    assert bool((o_buf[H * S:] == 7.0).all()) and bool((l_buf[H * S:] == 7.0).all())
    assert not bool((l_buf[:H * S] == 7.0).any())
    rows = np.unique(np.concatenate([np.arange(0, w.rows, max(1, w.rows // 300)), np.arange(w.rows - 40, w.rows)]))
    check_rows(oracle, w, *bits, out[:, :, inv].contiguous(), lse[:, :, inv].contiguous(), rows)
