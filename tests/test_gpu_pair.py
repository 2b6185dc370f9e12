"""ring_pair_kernel (ringattn_pair.hip: 128 query rows per workgroup, the key tiles dealt in turn to two pairs of waves) against the
CPU oracle where it can go wrong: the four tiles it needs at least, an odd tile more, ragged ends that fall to either group and
hold one key or 31, query tiles that end early, rows that see nothing of the second group's first tile (causal), several
key ranges whose tiles change hands (zigzag), grouped heads, heads that the XCDs share unevenly, and logits that make both
groups move their references again and again.  Bounds: those of test_gpu_parity.check_rows, which derive from the roundings
of P and O to the storage type."""
import importlib.util
import os
import re

import numpy as np
import pytest
import torch

from ringattention_amd import api
from ringattention_amd.configs import Workload
from test_gpu_parity import check_rows
from test_gpu_walk64 import rising_logits
from test_kernel_resources import test_no_lds_transfer_reads_a_scalar_register_fresh_from_a_vector_instruction as _hazards
from test_kernel_resources import compile_to_asm
from test_walk64_loop import CSRC, operands, regs


@pytest.mark.gpu
@pytest.mark.parametrize("d", [64, 128])
@pytest.mark.parametrize("lens,B,H,hkv,dtype,causal,zigzag,slope", [
    ((128,), 1, 1, 1, "fp16", True, False, 0),                    # four tiles: two per group
    ((129,), 1, 2, 1, "bf16", False, False, 0),                   # a fifth of one key: group 0's third
    ((100, 91), 1, 1, 1, "fp16", False, False, 0),                # 191: six tiles, the last of 31 keys is group 1's
    ((385,), 2, 3, 3, "bf16", True, False, 0),                    # a last q tile of one row; six heads over eight XCDs
    ((200, 313), 1, 9, 3, "fp16", True, False, 0),                # one head more than the XCDs, grouped
    ((256, 512, 256), 1, 2, 2, "bf16", True, True, 0),            # two segments per rank, up to four ranges each
    ((320, 320, 320), 1, 2, 1, "fp16", True, True, 0),            # ranges of five tiles: the groups swap places
    ((640, 384), 1, 2, 2, "fp16", False, False, 0.3),             # the row maximum keeps climbing
    ((640, 385), 1, 2, 2, "bf16", True, False, 0.3),
    ((1024,), 1, 1, 1, "fp16", True, False, 4.0),                 # steep enough to overflow a stale reference
    ((2048, 77), 1, 4, 4, "bf16", False, False, 0),
])
def test_pair_kernel_against_oracle(oracle, monkeypatch, lens, B, H, hkv, dtype, causal, zigzag, slope, d):
    for name in ("RINGATTN_WIDE", "RINGATTN_WIDE_PARTIALS", "RINGATTN_SPLIT"):
        monkeypatch.delenv(name, raising=False)
    monkeypatch.setenv("RINGATTN_PAIR", "1")
    S = sum(lens)
    w = Workload("pair", B, H, d, 1, S, dtype, 700 + S, causal)
    q, _, _ = rising_logits(w, slope) if slope else api.make_qkv_bits(w)
    wk = Workload("pair_kv", B, hkv, d, 1, S, dtype, 1700 + S, causal)
    _, k, v = rising_logits(wk, slope) if slope else api.make_qkv_bits(wk)
    order = api.zigzag_order(lens) if zigzag else np.arange(S)
    inv = torch.from_numpy(np.argsort(order)).cuda()
    qd, kd, vd = (api.bits_to_tensor(np.ascontiguousarray(x[:, :, order]), dtype) for x in (q, k, v))
    plan = api.RingAttention(len(lens), list(lens), d, B, H, dtype, causal, kv_heads=hkv, layout="zigzag" if zigzag else "contiguous")
    try:
        assert plan.forward_kernel() == "ring_pair_kernel"
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
@pytest.mark.parametrize("d", [64, 128])
def test_a_row_of_nan_stays_one(monkeypatch, d):
    """A query row that is not a number gives a row that is not, with LSE -inf as on the 256-row kernels, on the kernels that
    combine several softmax states too; its neighbours keep their values."""
    S = 512
    w = Workload("nan_row", 1, 2, d, 1, S, "fp16", 41, False)
    qd, kd, vd = (api.bits_to_tensor(x, "fp16") for x in api.make_qkv_bits(w))
    qn = qd.clone()
    qn[0, 1, 77] = float("nan")
    for name in ("RINGATTN_WIDE", "RINGATTN_WIDE_PARTIALS", "RINGATTN_SPLIT"):
        monkeypatch.delenv(name, raising=False)
    for pair, kernel in (("1", "ring_pair_kernel"), ("0", "ring_split_kernel")):
        monkeypatch.setenv("RINGATTN_PAIR", pair)
        plan = api.RingAttention(1, S, d, 1, 2, "fp16", False)
        assert plan.forward_kernel() == kernel
        o_n, l_n = plan.forward(qn, kd, vd)
        o, l = plan.forward(qd, kd, vd)
        torch.cuda.synchronize()
        plan.close()
        assert o_n[0, 1, 77].isnan().all() and l_n[0, 1, 77].item() == float("-inf"), kernel
        keep = torch.ones(S, dtype=torch.bool, device="cuda")
        keep[64:128] = False   # (rows of the same wave may take another reference)
        assert torch.equal(o_n[:, :, keep], o[:, :, keep]) and torch.equal(l_n[:, :, keep], l[:, :, keep]), kernel
        assert not o_n[0, 0].isnan().any() and int(o_n.isnan().any(-1).sum()) == 1, kernel


def test_pair_kernel_resources_and_hazards(tmp_path):
    """One wave per SIMD, no scratch, the rings, lists and statistics within the LDS; and the wait states in front of the
    direct-to-LDS loads."""
    _, usage = compile_to_asm("ringattn_pair.hip", tmp_path / "pair.s")
    kernels = {n: u for n, u in usage.items() if "ring_pair_kernel" in n}
    assert len(kernels) == 4
    for n, u in kernels.items():
        assert u["ScratchSize [bytes/lane]"] == 0 and u["Occupancy [waves/SIMD]"] == 1, (n, u)
        assert u["LDS Size [bytes/block]"] <= 160 * 1024, (n, u)
    _hazards("ringattn_pair.hip", tmp_path)


@pytest.mark.parametrize("d", [128, 64])
def test_pair_loop_text(d):
    """The committed loop is what the generator writes; every iteration has one barrier, in front of its tile loads and of the
    V fragments it reads, and each MFMA finds its fragments returned; branches lead to labels that exist."""
    spec = importlib.util.spec_from_file_location("gen_walk64_loop", os.path.join(CSRC, "gen_walk64_loop.py"))
    gen = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(gen)
    with open(os.path.join(CSRC, gen.PAIR_FILES[d])) as f:
        assert f.read() == gen.render(d, 2)
    mfma = "v_mfma_f32_32x32x16_f16"
    gen.configure(d, 2)
    del gen._sites[:]
    del gen._redo[:]
    for i in range(gen.UNROLL):
        lines = [l for l in gen.iteration(i, mfma, "v_cvt_pk_f16_f32") if not l.endswith(":")]
        ops = [operands(l)[0] for l in lines]
        assert ops.count(mfma) == d // 4 and ops.count("s_barrier") == 1 and ops.count("global_load_lds_dwordx4") == d // 16
        bar = ops.index("s_barrier")
        assert lines[bar - 1] == "s_waitcnt vmcnt(%d)" % (3 * d // 32) or "s_waitcnt vmcnt(%d)" % (3 * d // 32) in lines[:bar]
        assert min(j for j, o in enumerate(ops) if o.startswith(("global_load_lds", "ds_read_b64_tr"))) > bar
        outstanding = [set(regs(gen.KF(ks))[1]) for ks in range(min(gen.PREREAD, gen.KS))]
        for line in lines:
            op, args = operands(line)
            if op.startswith("ds_read"):
                outstanding.append(set(regs(args[0])[1]))
            elif op == "s_waitcnt" and "lgkmcnt" in line:
                keep = int(re.search(r"lgkmcnt\((\d+)\)", line).group(1))
                outstanding = outstanding[max(0, len(outstanding) - keep):]
            elif op == mfma:
                read = {r for tok in args[1:3] if regs(tok)[0] == "v" for r in regs(tok)[1]}
                assert not any(read & x for x in outstanding), (i, line)
    text = gen.loop_text(mfma, "v_cvt_pk_f16_f32")
    labels = [l[:-1] for l in text if l.endswith(":")]
    assert len(labels) == len(set(labels))
    at = {l[:-1]: k for k, l in enumerate(text) if l.endswith(":")}
    for k, l in enumerate(text):
        m = re.match(r"s_c?branch\w*\s+(\d+)([fb])$", l)
        assert not m or (at[m.group(1)] > k) == (m.group(2) == "f"), l
