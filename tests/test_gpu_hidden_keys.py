"""Keys that a coordinate of -inf hides from every query (left padding), a tile of 32 of them and more at the start of the walk,
with all other logits far below zero: a row has no reference maximum until its first finite score, and whatever stands in for
one must not let that score's exponential underflow.  Every attention kernel, against the same attention in float64."""
import numpy as np
import pytest
import torch

from np_reference import bits_to_float64, float32_to_bits
from ringattention_amd import api
from ringattention_amd.configs import Workload
from test_gpu_parity import storage_ulp

KERNELS = {  # name: (environment, ranks, plan options)
    "ring_walk64_kernel": ({"RINGATTN_PAIR": "0", "RINGATTN_SPLIT": "0"}, (320, 704), {}),
    "ring_pair_kernel": ({"RINGATTN_PAIR": "1"}, (500, 601), {}),
    "ring_split_kernel": ({"RINGATTN_SPLIT": "8"}, (500, 601), {}),
    "ring_walk_kernel": ({"RINGATTN_WIDE": "0"}, (500, 601), {}),
    "ring_walk64_kernel, partials": ({"RINGATTN_WIDE_PARTIALS": "1"}, (320, 704), {"step_partials": True}),
}


def reference(q, k, v, hidden, causal, scale):
    """Attention in float64 (CPU) over the keys from `hidden` on: O, LSE and the same average of |V|."""
    q, k, v = (torch.from_numpy(x) for x in (q, k, v))
    logits = torch.matmul(q, k.transpose(-1, -2).contiguous()) * scale
    S = q.shape[2]
    seen = torch.arange(S)[None, :] >= hidden
    if causal:
        seen = seen & (torch.arange(S)[None, :] <= torch.arange(S)[:, None])
    logits = logits.masked_fill(~seen, float("-inf"))
    lse = torch.logsumexp(logits, -1)
    p = torch.exp(logits - torch.where(torch.isinf(lse), torch.zeros_like(lse), lse)[..., None])
    return (x.numpy() for x in (torch.matmul(p, v), lse, torch.matmul(p, v.abs())))


@pytest.mark.gpu
@pytest.mark.parametrize("kernel,d", [(k, d) for k in KERNELS for d in (64, 128)
                                      if d == 128 or k != "ring_walk64_kernel, partials"])   # (partials at d = 128 only)
@pytest.mark.parametrize("dtype", ["fp16", "bf16"])
@pytest.mark.parametrize("hidden,causal", [(40, False), (130, False), (40, True), (130, True)])
def test_rows_without_a_reference_in_their_first_tile(monkeypatch, kernel, d, dtype, hidden, causal):
    env, lens, options = KERNELS[kernel]
    for name in ("RINGATTN_WIDE", "RINGATTN_WIDE_D64", "RINGATTN_WIDE_PARTIALS", "RINGATTN_SPLIT", "RINGATTN_PAIR"):
        monkeypatch.delenv(name, raising=False)
    for name, value in env.items():
        monkeypatch.setenv(name, value)
    B, H, S = 1, 2, sum(lens)
    w = Workload("hidden", B, H, d, 1, S, dtype, 600 + d, causal)
    q, k, v = (bits_to_float64(x, dtype).astype(np.float32).reshape(B, H, S, d) for x in api.make_qkv_bits(w))
    q[..., 0], q[..., 1] = 1.0, 4.0
    k[..., 0] = 0.0
    k[..., 1] = -(15.0 if dtype == "fp16" else 30.0) * d ** 0.5      # every logit moves down by 60 (fp16) or 120
    bits = [float32_to_bits(x, dtype).reshape(B, H, S, d) for x in (q, k, v)]
    exact = [bits_to_float64(x, dtype).reshape(B, H, S, d) for x in bits]
    o_ref, l_ref, mean_abs_v = reference(*exact, hidden, causal, d ** -0.5)
    k[:, :, :hidden, 0] = -np.inf
    bits[1] = float32_to_bits(k, dtype).reshape(B, H, S, d)
    plan = api.RingAttention(len(lens), list(lens), d, B, H, dtype, causal, **options)
    try:
        assert plan.forward_kernel() == kernel.split(",")[0]
        out, lse = plan.forward(*(api.bits_to_tensor(x, dtype) for x in bits))
        torch.cuda.synchronize()
    finally:
        plan.close()
    out, lse = out.double().cpu().numpy(), lse.double().cpu().numpy()
    blind = np.isinf(l_ref)   # rows that see no key
    assert blind.any() == causal and (lse[blind] == -np.inf).all() and (out[blind] == 0).all()
    # half a unit in the last place for the store of O; half a unit relative for each probability, and where fp16 holds it as a
    # subnormal half of 2^-24 of the reference (the row maximum or less: of 1 or less in the sum)
    u = 2.0 ** -(11 if dtype == "fp16" else 8)
    bound = 0.5 * storage_ulp(o_ref, dtype) + u * mean_abs_v + 2.0 ** -25 * S * np.abs(exact[2]).max() + 1e-5
    assert (np.abs(out - o_ref)[~blind] <= bound[~blind]).all()
    assert (np.abs(lse[~blind] - l_ref[~blind]) <= 1e-4 * np.abs(l_ref[~blind])).all()
