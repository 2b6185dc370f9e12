"""Parity of the gfx950 path (through the C ABI) with the CPU oracle on the same seeded
inputs.  Tolerances are the ones the engine is specified with:

    O   : max-abs error <= 1e-2 against the float64 oracle (O is stored in fp16 / bf16)
    LSE : relative error <= 1e-3 (fp32)

Large workloads are compared on whole heads (cfg2 in full; one or two complete heads of cfg3 and
cfg4; complete 256-row q tiles at chunk starts, middles and ends of cfg5) plus a seeded sample of rows
(the first rows of the sequence, where causal rows see few keys and |O| is largest, are always
included), and through size-independent properties on the full output.  Where the roundings that
the algorithm prescribes (the store of O and the probabilities of the PV product, both in the storage
type) by themselves allow more than 1e-2 -- bf16 rows that average very few, large V rows -- what
they allow is the bound: see check_rows."""
import math
import os

import numpy as np
import pytest
import torch

from np_reference import bits_to_float64, float32_to_bits
from ringattention_amd import api
from ringattention_amd.configs import WORKLOADS, Workload

pytestmark = pytest.mark.gpu

O_TOL = 1e-2       # max-abs on O
LSE_RTOL = 1e-3    # relative on LSE
GOLD = os.path.join(os.path.dirname(__file__), "golden")


def to_dev(bits, dtype):
    return api.bits_to_tensor(bits, dtype)


# What keeps a forward that carries the state on one kernel, whatever its size ("": the library's own choice, for the small
# shapes of these tests ring_split_kernel or ring_pair_kernel).
FORCE = {"": {}, "ring_walk_kernel": {"RINGATTN_WIDE": "0"}, "ring_walk64_kernel": {"RINGATTN_SPLIT": "0", "RINGATTN_PAIR": "0"}}


def force(monkeypatch, kernel):
    for name in ("RINGATTN_WIDE", "RINGATTN_WIDE_D64", "RINGATTN_WIDE_PARTIALS", "RINGATTN_SPLIT", "RINGATTN_PAIR"):
        monkeypatch.delenv(name, raising=False)
    for name, value in FORCE[kernel].items():
        monkeypatch.setenv(name, value)


def forward(w, q, k, v, kernel="", **kw):
    """kernel: the one that has to run it (force() says so to the library)."""
    plan = api.RingAttention(w.npes, w.chunk, w.dim, w.batch, w.heads, w.dtype, w.causal, graph=w.graph,
                             half_partials=w.half_partials, **kw)
    try:
        assert kernel in ("", plan.forward_kernel())
        out, lse = plan.forward(to_dev(q, w.dtype), to_dev(k, w.dtype), to_dev(v, w.dtype))
        torch.cuda.synchronize()
        return out, lse
    finally:
        plan.close()


def sample_rows(w, n, seed=0):
    rng = np.random.default_rng(seed)
    first = np.arange(min(64, w.seq))                       # rows 0..63 of head 0
    last_head = (w.batch * w.heads - 1) * w.seq + np.arange(min(32, w.seq))
    chunk_edges = np.array([r * w.chunk + x for r in range(w.npes) for x in (0, w.chunk - 1)])
    return np.unique(np.concatenate([rng.integers(0, w.rows, n), first, last_head, chunk_edges]))


def storage_ulp(x, dtype):
    """Spacing of the storage type at |x| (numpy array, float64)."""
    mant, emin = (10, -14) if dtype == "fp16" else (7, -126)
    e = np.floor(np.log2(np.maximum(np.abs(x), 2.0 ** emin)))
    return 2.0 ** (e - mant)


def check_rows(oracle, w, q, k, v, out, lse, rows, scale=None, half_partials=None, plain_bound=None):
    """O against the float64 oracle: max-abs error <= 1e-2 -- or, where that is more, what the two roundings
    that the algorithm prescribes allow at that element: half a unit in the last place of the storage type for
    the store of O (csrc/ring_attention.cu:635; a bf16 value in [4, 8) is a multiple of 2^-5, so even the
    correctly rounded result can be 1.56e-2 off), plus u sum_i w_i |v_i| for the probabilities, which go into
    the PV product rounded to the storage type (:604, u = 2^-(mantissa+1) relative each) while the row sum is
    taken from the unrounded ones (:242): O = sum_i w_i (1 + delta_i) v_i with |delta_i| <= u.  sum_i w_i |v_i|
    is the attention output over |V| and comes from the oracle.  Only rows that average very few V rows -- the
    first rows of a causal sequence, or a softmax peaked by a large explicit scale -- get beyond 1e-2 this way;
    everywhere else the bound is 1e-2.
    In addition every element lies within ONE unit in the last place (of the row's largest element) of the
    oracle rounded to the storage type (two with fp16 per-step partials), except that one row in a thousand
    may use u max|V| plus half an ulp for the store instead (rows whose few dominant keys carry large V
    entries that nearly cancel).
    LSE: relative error <= 1e-3.
    plain_bound: the rounding allowance for the probabilities may not be used at all -- every element within
    max(1e-2, half an ulp of the storage type).  Always so for fp16 (half an ulp of fp16 stays below 1e-2 up to
    |O| = 16, and its probabilities carry 2^-11, not 2^-8); the five specified workloads ask for it explicitly."""
    if plain_bound is None:
        plain_bound = w.dtype == "fp16"
    o_ref, l_ref = oracle.attention_rows(q, k, v, w.dtype, causal=w.causal, rows=rows, scale=scale)
    idx = torch.from_numpy(rows).cuda()
    o_gpu = out.reshape(-1, w.dim)[idx].double().cpu().numpy()
    l_gpu = lse.reshape(-1)[idx].double().cpu().numpy()
    assert np.isfinite(o_gpu).all() and np.isfinite(l_gpu).all()
    ulp = storage_ulp(o_ref, w.dtype)
    tol = np.maximum(O_TOL, 0.5 * ulp)
    u_p = 2.0 ** -((10 if w.dtype == "fp16" else 7) + 1)
    v_max = bits_to_float64(np.array([(np.ascontiguousarray(v).view(np.uint16) & 0x7FFF).max()], dtype=np.uint16), w.dtype)[0]
    p_round = u_p * v_max
    err = np.abs(o_gpu - o_ref)
    beyond = np.unique(np.nonzero(err > tol)[0])
    if len(beyond) and not plain_bound:  # rows with an element beyond the plain bound: what do their own roundings allow?
        v_abs = (np.ascontiguousarray(v).view(np.uint16) & 0x7FFF).view(v.dtype)
        mean_abs_v, _ = oracle.attention_rows(q, k, v_abs, w.dtype, causal=w.causal, rows=rows[beyond], scale=scale)
        tol[beyond] = np.maximum(tol[beyond], 0.5 * ulp[beyond] + u_p * mean_abs_v)
        print(f"parity {w.name}: {len(beyond)} of {len(rows)} rows have an element beyond max(1e-2, half an ulp); "
              f"their own rounding bound is up to {tol[beyond].max():.3e}")
        # the allowance is for rows that average very few V rows (the first rows of a causal sequence, a softmax
        # peaked by huge logits), never for a workload at large: at most two rows in a hundred
        assert len(beyond) <= max(4, len(rows) // 50), f"{w.name}: {len(beyond)} rows beyond the plain bound"
    err_o = err.max()
    err_l = (np.abs(l_gpu - l_ref) / np.maximum(np.abs(l_ref), 1e-3)).max()
    # also against the oracle rounded to the storage type (what a perfect kernel would store)
    o_rounded = bits_to_float64(float32_to_bits(o_ref.astype(np.float32), w.dtype), w.dtype)
    err_r = np.abs(o_gpu - o_rounded)
    # ... measured in units in the last place of the ROW's largest element: the kernel rounds the
    # probabilities to the storage type before the PV product (as the reference does,
    # csrc/ring_attention.cu:604), which moves every element of a row by about that much however
    # small the element itself is
    ulp_r = storage_ulp(np.maximum(np.abs(o_gpu), np.abs(o_rounded)).max(axis=1, keepdims=True), w.dtype)
    print(f"parity {w.name}: {len(rows)} rows, max|dO| = {err_o:.3e} vs fp64, {err_r.max():.3e} vs rounded fp64 "
          f"({(err_r / ulp_r).max():.2f} ulp), max rel dLSE = {err_l:.3e}, max|O| = {np.abs(o_ref).max():.2f}, "
          f"{int((tol > O_TOL).sum())} elements where half an ulp exceeds 1e-2, "
          f"bound: {'max(1e-2, half an ulp), no allowance' if plain_bound else 'with the rounding allowance'}")
    assert (err <= tol).all(), f"{w.name}: max|dO| = {err_o:.3e}, worst excess {(err - tol).max():.3e}"
    # fp16 per-step partials (RINGATTN_FLAG_HALF_PARTIALS) round once more on the way: two units then
    ulps = 2 if (w.half_partials if half_partials is None else half_partials) else 1
    p_rounding = p_round + 0.5 * storage_ulp(o_rounded, w.dtype)
    over = int((err_r > ulps * ulp_r).any(axis=1).sum())
    if over:
        print(f"parity {w.name}: {over} of {len(rows)} rows beyond {ulps} ulp of the rounded oracle "
              f"(max {(err_r / ulp_r).max():.2f}), within the p-rounding bound {p_rounding.max():.3e}")
    assert over <= max(1, len(rows) // 1000), f"{w.name}: {over} rows beyond {ulps} ulp of the rounded oracle"
    assert (err_r <= np.maximum(ulps * ulp_r, p_rounding)).all(), \
        f"{w.name}: {(err_r / ulp_r).max():.2f} ulp from the rounded oracle, beyond the p-rounding bound"
    assert err_l <= LSE_RTOL, f"{w.name}: max rel dLSE = {err_l:.3e}"
    return err_o, err_l


def whole_head_rows(w, heads):
    """All rows of the given flat head indices (b * H + h)."""
    return np.concatenate([np.arange(h * w.seq, (h + 1) * w.seq) for h in heads])


def workload_rows(w):
    """Rows compared for each of the five workloads: whole heads where the oracle gets through them
    in seconds, complete 256-row q tiles (a workgroup's rows) at the start, middle and end of chunks for the longest one,
    plus the seeded sample (first rows of the sequence, last head, chunk edges)."""
    bh = w.batch * w.heads
    if w.name == "cfg2":
        rows = np.arange(w.rows)                                        # everything
    elif w.name == "cfg3":
        rows = np.concatenate([whole_head_rows(w, [bh - 1]), sample_rows(w, 512)])
    elif w.name == "cfg4":
        rows = np.concatenate([whole_head_rows(w, [0, bh - 1]), sample_rows(w, 384)])
    elif w.name == "cfg5":
        tiles = []
        for head, chunk, where in ((0, 0, 0), (0, 3, w.chunk // 2), (5, 7, w.chunk - 256), (bh - 1, w.npes - 1, w.chunk - 256),
                                   (bh - 1, 8, 0), (9, 15, 4096 + 256)):
            first = head * w.seq + chunk * w.chunk + where
            tiles.append(np.arange(first, first + 256))
        rows = np.concatenate(tiles + [sample_rows(w, 1400)])
    else:
        rows = sample_rows(w, 256)
    return np.unique(rows)


def test_cfg1_full_against_oracle_and_golden(oracle):
    w = WORKLOADS["cfg1"]
    q, k, v = api.make_qkv_bits(w)
    out, lse = forward(w, q, k, v)
    check_rows(oracle, w, q, k, v, out, lse, np.arange(w.rows), plain_bound=True)
    g = np.load(os.path.join(GOLD, "cfg1_expected.npz"))   # torch-library fixture, independent of the oracle
    assert np.abs(out.float().cpu().numpy() - g["o_f32"]).max() <= O_TOL
    assert np.abs(lse.double().cpu().numpy() - g["lse_f64"]).max() <= LSE_RTOL * np.abs(g["lse_f64"]).max()


def test_causal_small_golden(oracle):
    w = Workload("causal_small", 1, 2, 128, 2, 128, "bf16", 11, True)
    q, k, v = api.make_qkv_bits(w)
    out, lse = forward(w, q, k, v)
    check_rows(oracle, w, q, k, v, out, lse, np.arange(w.rows))
    g = np.load(os.path.join(GOLD, "causal_small_expected.npz"))
    assert np.abs(out.float().cpu().numpy() - g["o_f32"]).max() <= O_TOL


@pytest.mark.parametrize("name,step_partials", [("cfg2", False), ("cfg2", True), ("cfg3", False), ("cfg3", True),
                                                ("cfg4", False), ("cfg4", True), ("cfg5", False), ("cfg5", True)])
def test_workload_whole_heads(oracle, name, step_partials):
    # step_partials: the forward that keeps the ring steps apart (per-step partials in the workspace,
    # fp16 where the workload says so) instead of carrying the softmax state through them
    w = WORKLOADS[name]
    q, k, v = api.make_qkv_bits(w)
    out, lse = forward(w, q, k, v, step_partials=step_partials)
    # the five specified workloads: max(1e-2, half an ulp of the storage type) for every element, no allowance
    check_rows(oracle, w, q, k, v, out, lse, workload_rows(w), half_partials=w.half_partials and step_partials,
               plain_bound=True)
    # full-size properties: finite everywhere, convexity |O| <= max|V| (O is an average of V rows)
    assert torch.isfinite(out).all() and torch.isfinite(lse).all()
    vmax = np.abs(bits_to_float64(v, w.dtype)).max()
    assert out.abs().max().item() <= vmax * (1 + 2**-7)
    if w.causal:  # row 0 of every head sees one key: O = V[0] exactly, LSE = scale * q0.k0
        o0 = out[:, :, 0, :].double().cpu().numpy()
        assert np.array_equal(o0, bits_to_float64(v, w.dtype)[:, :, 0, :])
        dots = (bits_to_float64(q, w.dtype)[:, :, 0, :] * bits_to_float64(k, w.dtype)[:, :, 0, :]).sum(-1) / math.sqrt(w.dim)
        assert np.abs(lse[:, :, 0].double().cpu().numpy() - dots).max() <= 1e-5 + LSE_RTOL * np.abs(dots).max()


@pytest.mark.parametrize("w", [
    Workload("p1", 1, 2, 64, 1, 256, "fp16", 21, False),          # single rank: no rotation, 1-way merge
    Workload("p1c", 2, 1, 128, 1, 384, "bf16", 22, True),
    Workload("bh", 3, 5, 64, 2, 128, "bf16", 23, False),          # batch and heads, groups not a multiple of 8
    Workload("c64", 1, 3, 64, 4, 256, "fp16", 24, True),
    Workload("c128", 2, 2, 128, 3, 384, "fp16", 25, True),        # odd rank count
    Workload("p64", 1, 1, 128, 64, 128, "bf16", 26, True),        # maximum number of ranks
    Workload("big_logits", 1, 2, 128, 4, 512, "fp16", 27, False, sigma_qk=3.0),
    # d = 64 runs its softmax phase speculatively against the reference as it stands: logits whose row maximum
    # keeps climbing by many powers of two (sigma 9 and 36) make it fall back, also from an overflowed exponential
    Workload("big_logits_64", 1, 2, 64, 4, 512, "fp16", 28, False, sigma_qk=3.0),
    Workload("huge_logits_64", 1, 2, 64, 3, 384, "bf16", 29, True, sigma_qk=6.0),
    Workload("huge_logits_64h", 2, 1, 64, 2, 640, "fp16", 30, False, sigma_qk=6.0),
], ids=lambda w: w.name)
@pytest.mark.parametrize("kernel", FORCE)
def test_shapes_and_edges_full(oracle, monkeypatch, w, kernel):
    force(monkeypatch, kernel)
    q, k, v = api.make_qkv_bits(w)
    out, lse = forward(w, q, k, v, kernel)
    check_rows(oracle, w, q, k, v, out, lse, np.arange(w.rows))


@pytest.mark.parametrize("seqlen,causal,d,dtype", [
    ((128, 384, 256), False, 64, "fp16"),
    ((512, 128, 256, 128), True, 128, "bf16"),
    ((128, 640), True, 128, "fp16"),
])
def test_unequal_rank_lengths(oracle, seqlen, causal, d, dtype):
    # per-PE seqlen[] of the reference (csrc/ring_attention.cu:753): ranks of different length
    S, P = sum(seqlen), len(seqlen)
    w = Workload("ragged_ranks", 2, 2, d, 1, S, dtype, 71, causal)   # only used for the seeded inputs
    q, k, v = api.make_qkv_bits(w)
    qd, kd, vd = (to_dev(x, dtype) for x in (q, k, v))
    plan = api.RingAttention(P, list(seqlen), d, w.batch, w.heads, dtype, causal)
    out, lse = plan.forward(qd, kd, vd)
    torch.cuda.synchronize()
    rows = np.arange(w.rows)
    check_rows(oracle, w, q, k, v, out, lse, rows)
    # the per-step partials follow the ring schedule of the unequal chunks
    _, _, po, pl = oracle.ring_rows(q, k, v, dtype, list(seqlen), rows, causal=causal, tile=32, want_parts=True)
    for s in range(P):
        o_part, lse_part = plan.block_forward(s, qd, kd, vd)
        torch.cuda.synchronize()
        lg = lse_part.reshape(-1).double().cpu().numpy()
        active = np.isfinite(pl[:, s])
        assert np.array_equal(np.isfinite(lg), active)
        # fp32 partial; p is rounded to the storage type before the PV product (2^-9 relative for bf16)
        assert np.abs(o_part.reshape(-1, d).double().cpu().numpy()[active] - po[active, s]).max() <= 5e-3
    # the reference-shaped entry on the same unequal layout, one head
    q1, k1, v1 = (np.ascontiguousarray(x[0, 0]) for x in (q, k, v))
    o_ref, _ = oracle.attention_rows(q1[None, None], k1[None, None], v1[None, None], dtype, causal=causal)
    start = np.concatenate([[0], np.cumsum(seqlen)])
    for mype in range(P):
        sl = slice(start[mype], start[mype + 1])
        o1 = torch.empty((seqlen[mype], d), dtype=qd.dtype, device="cuda")
        api.ring_attention(to_dev(np.ascontiguousarray(q1[sl]), dtype), to_dev(k1, dtype), to_dev(v1, dtype), o1, P, mype,
                           list(seqlen), d, max(seqlen), causal=causal)
        assert np.abs(o1.double().cpu().numpy() - o_ref[sl]).max() <= O_TOL
    plan.close()


@pytest.mark.parametrize("seqlen,causal,d,dtype,layout", [
    ((100, 333, 1, 77), False, 64, "fp16", "contiguous"),
    ((100, 333, 1, 77), True, 128, "bf16", "contiguous"),
    ((513,), True, 128, "fp16", "contiguous"),           # one rank, one row into a third q tile
    ((31, 33), True, 64, "bf16", "contiguous"),          # shorter than one key tile / one more than it
    ((1000, 24), False, 128, "bf16", "contiguous"),
    ((130, 70, 2, 258), True, 128, "bf16", "zigzag"),
    ((1, 1, 1), True, 64, "fp16", "contiguous"),
    ((257, 1023, 769), True, 128, "bf16", "contiguous"),   # several 256-row q tiles per rank, each rank one row or one tile off
    ((1026, 514), True, 64, "fp16", "zigzag"),             # d = 64: K and V tiles loaded by different halves of the workgroup
    ((640, 384, 896), False, 64, "bf16", "contiguous"),    # whole key tiles, chunk lengths that are no multiples of four tiles
])
@pytest.mark.parametrize("kernel", ["", "ring_walk_kernel"])
def test_ragged_lengths(oracle, monkeypatch, seqlen, causal, d, dtype, layout, kernel):
    # lengths that are no multiples of the 256-row q tile or the 32-key tile: the tail
    # predication the reference leaves open (csrc/ring_attention.cu:143-145)
    force(monkeypatch, kernel)
    P, S, B, H = len(seqlen), sum(seqlen), 2, 2
    w = Workload("ragged", B, H, d, 1, S, dtype, 95, causal)
    q, k, v = api.make_qkv_bits(w)
    order = api.zigzag_order(seqlen) if layout == "zigzag" else np.arange(S)
    inv = torch.from_numpy(np.argsort(order)).cuda()
    qd, kd, vd = (to_dev(np.ascontiguousarray(x[:, :, order]), dtype) for x in (q, k, v))
    # output buffers with sentinel rows behind them: nothing may be written past the end
    out_buf = torch.full((B * H * S + 64, d), 7.0, dtype=qd.dtype, device="cuda")
    lse_buf = torch.full((B * H * S + 64,), 7.0, dtype=torch.float32, device="cuda")
    out, lse = out_buf[:B * H * S].view(B, H, S, d), lse_buf[:B * H * S].view(B, H, S)
    plan = api.RingAttention(P, list(seqlen), d, B, H, dtype, causal, layout=layout)
    assert kernel in ("", plan.forward_kernel())
    plan.forward(qd, kd, vd, out, lse)
    torch.cuda.synchronize()
    assert bool((out_buf[B * H * S:] == 7.0).all()) and bool((lse_buf[B * H * S:] == 7.0).all())
    rows = np.arange(w.rows)
    check_rows(oracle, w, q, k, v, out[:, :, inv].contiguous(), lse[:, :, inv].contiguous(), rows)
    if layout == "contiguous":
        # per-step partials against the ring form of the oracle; untouched rows stay untouched
        _, _, po, pl = oracle.ring_rows(q, k, v, dtype, list(seqlen), rows, causal=causal, tile=32, want_parts=True)
        for s in range(P):
            o_part, lse_part = plan.block_forward(s, qd, kd, vd)
            torch.cuda.synchronize()
            lg = lse_part.reshape(-1).double().cpu().numpy()
            active = np.isfinite(pl[:, s])
            assert np.array_equal(np.isfinite(lg), active)
            if active.any():
                assert np.abs(o_part.reshape(-1, d).double().cpu().numpy()[active] - po[active, s]).max() <= 5e-3
        # the reference-shaped entry, one head, rank by rank
        q1, k1, v1 = (np.ascontiguousarray(x[0, 0]) for x in (q, k, v))
        o_ref, _ = oracle.attention_rows(q1[None, None], k1[None, None], v1[None, None], dtype, causal=causal)
        start = np.concatenate([[0], np.cumsum(seqlen)])
        for mype in range(P):
            sl = slice(start[mype], start[mype + 1])
            o1 = torch.empty((seqlen[mype], d), dtype=qd.dtype, device="cuda")
            api.ring_attention(to_dev(np.ascontiguousarray(q1[sl]), dtype), to_dev(k1, dtype), to_dev(v1, dtype), o1, P, mype,
                               list(seqlen), d, max(seqlen), causal=causal)
            assert np.abs(o1.double().cpu().numpy() - o_ref[sl]).max() <= O_TOL
    plan.close()


@pytest.mark.parametrize("causal", [False, True])
def test_grouped_query_heads(oracle, causal):
    # 8 query heads share 2 KV heads: the result equals plain attention with the KV heads repeated
    B, H, HKV, P, c, d = 2, 8, 2, 4, 256, 128
    w = Workload("gqa", B, H, d, P, c, "bf16", 81, causal)
    q, _, _ = api.make_qkv_bits(w)
    wkv = Workload("gqa_kv", B, HKV, d, P, c, "bf16", 82, causal)
    _, k, v = api.make_qkv_bits(wkv)
    plan = api.RingAttention(P, c, d, B, H, "bf16", causal, kv_heads=HKV)
    out, lse = plan.forward(to_dev(q, "bf16"), to_dev(k, "bf16"), to_dev(v, "bf16"))
    torch.cuda.synchronize()
    plan.close()
    k_rep, v_rep = (np.repeat(x, H // HKV, axis=1) for x in (k, v))
    check_rows(oracle, w, q, k_rep, v_rep, out, lse, np.arange(w.rows))


@pytest.mark.parametrize("seqlen,B,H,d,dtype,hkv", [
    ((512, 512, 512, 512), 1, 2, 128, "bf16", 0),
    ((256, 768, 512), 2, 3, 64, "fp16", 0),           # unequal ranks, odd rank count
    ((1024,), 1, 2, 128, "fp16", 0),                  # one rank: zigzag degenerates to the plain causal mask
    ((256,) * 8, 1, 4, 128, "bf16", 2),               # with grouped-query heads
])
@pytest.mark.parametrize("kernel", FORCE)
def test_zigzag_layout(oracle, monkeypatch, seqlen, B, H, d, dtype, hkv, kernel):
    force(monkeypatch, kernel)
    # The sequence is generated in sequence order, stored in zigzag memory order, and the
    # result (brought back to sequence order) must equal causal attention over the sequence.
    P, S = len(seqlen), sum(seqlen)
    w = Workload("zigzag", B, H, d, 1, S, dtype, 91, True)
    q, k, v = api.make_qkv_bits(w)
    if hkv:
        _, k, v = api.make_qkv_bits(Workload("zigzag_kv", B, hkv, d, 1, S, dtype, 92, True))
    order = api.zigzag_order(seqlen)
    inv = torch.from_numpy(np.argsort(order)).cuda()
    qd, kd, vd = (to_dev(np.ascontiguousarray(x[:, :, order]), dtype) for x in (q, k, v))
    plan = api.RingAttention(P, list(seqlen), d, B, H, dtype, True, kv_heads=hkv, layout="zigzag")
    assert kernel in ("", plan.forward_kernel())
    out, lse = plan.forward(qd, kd, vd)
    torch.cuda.synchronize()
    out_seq, lse_seq = out[:, :, inv].contiguous(), lse[:, :, inv].contiguous()
    k_full, v_full = ((np.repeat(x, H // hkv, axis=1) if hkv else x) for x in (k, v))
    check_rows(oracle, w, q, k_full, v_full, out_seq, lse_seq, np.arange(w.rows))
    plan.close()
    # the forward that keeps the steps apart: same bar against the oracle ...
    plan = api.RingAttention(P, list(seqlen), d, B, H, dtype, True, kv_heads=hkv, layout="zigzag", step_partials=True)
    out, lse = plan.forward(qd, kd, vd)
    torch.cuda.synchronize()
    check_rows(oracle, w, q, k_full, v_full, out[:, :, inv].contiguous(), lse[:, :, inv].contiguous(), np.arange(w.rows))
    # ... and step by step through the C ABI: the same items, so the same bits
    o_parts = torch.zeros((P, B, H, S, d), dtype=torch.float32, device="cuda")
    lse_parts = torch.full((P, B, H, S), float("-inf"), dtype=torch.float32, device="cuda")
    for s in range(P):
        plan.block_forward(s, qd, kd, vd, o_parts[s], lse_parts[s])
    out2, lse2 = plan.merge_ring(o_parts, lse_parts)
    torch.cuda.synchronize()
    assert torch.equal(out2, out) and torch.equal(lse2, lse)
    # low halves never see a later rank: those (row, step) partials stay untouched
    start = np.concatenate([[0], np.cumsum(seqlen)])
    for r in range(P):
        for s in range(1, P):
            low = lse_parts[s, :, :, start[r]:start[r] + seqlen[r] // 2]
            assert bool(torch.isinf(low).all()) == ((r + s) % P > r)
    plan.close()


def test_zigzag_without_mask_equals_contiguous():
    w = Workload("zz_nomask", 1, 2, 128, 4, 256, "bf16", 93, False)
    q, k, v = (to_dev(x, w.dtype) for x in api.make_qkv_bits(w))
    res = []
    for layout in ("contiguous", "zigzag"):
        plan = api.RingAttention(w.npes, w.chunk, w.dim, w.batch, w.heads, w.dtype, False, layout=layout)
        res.append(plan.forward(q, k, v))
        torch.cuda.synchronize()
        plan.close()
    assert torch.equal(res[0][0], res[1][0]) and torch.equal(res[0][1], res[1][1])


def test_zigzag_cfg4_sampled_rows(oracle):
    w = WORKLOADS["cfg4"]
    q, k, v = api.make_qkv_bits(w)
    seqlen = [w.chunk] * w.npes
    order = api.zigzag_order(seqlen)
    inv = np.argsort(order)
    order_d = torch.from_numpy(order).cuda()
    qd, kd, vd = (to_dev(x, w.dtype)[:, :, order_d].contiguous() for x in (q, k, v))
    plan = api.RingAttention(w.npes, w.chunk, w.dim, w.batch, w.heads, w.dtype, True, layout="zigzag")
    out, lse = plan.forward(qd, kd, vd)
    torch.cuda.synchronize()
    plan.close()
    assert torch.isfinite(out).all() and torch.isfinite(lse).all()
    # (head, sequence position) pairs: the whole of head 17 and the seeded sample
    rows_seq = np.unique(np.concatenate([whole_head_rows(w, [17]), sample_rows(w, 384)]))
    head, posn = rows_seq // w.seq, rows_seq % w.seq
    rows_mem = torch.from_numpy(head * w.seq + inv[posn]).cuda()
    o_ref, l_ref = oracle.attention_rows(q, k, v, w.dtype, causal=True, rows=rows_seq)
    o_gpu = out.reshape(-1, w.dim)[rows_mem].double().cpu().numpy()
    l_gpu = lse.reshape(-1)[rows_mem].double().cpu().numpy()
    ulp = storage_ulp(o_ref, w.dtype)
    assert (np.abs(o_gpu - o_ref) <= np.maximum(O_TOL, 0.5 * ulp)).all()      # the rule of check_rows
    o_rounded = bits_to_float64(float32_to_bits(o_ref.astype(np.float32), w.dtype), w.dtype)
    assert (np.abs(o_gpu - o_rounded) <= storage_ulp(np.maximum(np.abs(o_gpu), np.abs(o_rounded)).max(axis=1, keepdims=True),
                                                      w.dtype)).all()
    assert (np.abs(l_gpu - l_ref) / np.maximum(np.abs(l_ref), 1e-3)).max() <= LSE_RTOL


def test_explicit_softmax_scale(oracle):
    w = Workload("scale", 1, 2, 64, 2, 256, "fp16", 31, False)
    q, k, v = api.make_qkv_bits(w)
    out, lse = forward(w, q, k, v, softmax_scale=0.3)
    check_rows(oracle, w, q, k, v, out, lse, np.arange(w.rows), scale=0.3)


def test_closed_forms_on_device(oracle):
    w = Workload("closed", 1, 2, 128, 4, 256, "bf16", 32, True)
    q, k, v = api.make_qkv_bits(w)
    zero = np.zeros_like(q)
    vf = bits_to_float64(v, w.dtype)
    # Q = 0: O = prefix mean of V, LSE = ln(row + 1)
    out, lse = forward(w, zero, k, v)
    prefix = np.cumsum(vf, axis=2) / np.arange(1, w.seq + 1)[None, None, :, None]
    assert np.abs(out.double().cpu().numpy() - prefix).max() <= O_TOL
    want = np.log(np.arange(1, w.seq + 1))
    assert np.abs(lse.double().cpu().numpy() - want[None, None]).max() <= 1e-5 + LSE_RTOL * want.max()
    # constant V: O equals the constant exactly representable value
    vc = np.full_like(v, float32_to_bits(np.array([-0.75], np.float32), w.dtype)[0])
    out, _ = forward(w, q, k, vc)
    assert torch.all(out.float() == -0.75)
    # linear in V: O(V1 + V2) = O(V1) + O(V2) up to storage rounding
    rng = np.random.default_rng(0)
    v1 = float32_to_bits(rng.integers(-8, 9, v.shape).astype(np.float32) / 8, w.dtype)
    v2 = float32_to_bits(rng.integers(-8, 9, v.shape).astype(np.float32) / 8, w.dtype)
    v12 = float32_to_bits((bits_to_float64(v1, w.dtype) + bits_to_float64(v2, w.dtype)).astype(np.float32), w.dtype)
    o1, _ = forward(w, q, k, v1)
    o2, _ = forward(w, q, k, v2)
    o12, l12 = forward(w, q, k, v12)
    assert (o12.float() - o1.float() - o2.float()).abs().max().item() <= O_TOL


def test_reference_fill_pattern_saturating_softmax(oracle, ralib):
    # the reference harness's own inputs (csrc/ring_attention.cu:731-741): 2 ranks, d = 64, fp16
    import ctypes
    P, c, d = 2, 512, 64
    buf = np.empty((P * c, d), dtype=np.uint16)
    assert ralib.ringattn_fill_reference_pattern(buf.ctypes.data_as(ctypes.c_void_p), 0, c, d) == 0
    buf[c:] = buf[:c]   # every PE fills its own block with the same pattern (initQKV, :743-748)
    w = Workload("reffill", 1, 1, d, P, c, "fp16", 0, False)
    x = buf.reshape(1, 1, P * c, d)
    out, lse = forward(w, x, x, x)
    # |O| reaches 58 here, where one fp16 ulp is 2^-5 = 0.031 > 1e-2: the storage type, not
    # the kernel, bounds the error, so the O tolerance is max(1e-2, 1 ulp of the stored value)
    o_ref, l_ref = oracle.attention_rows(x, x, x, "fp16")
    o_gpu = out.double().cpu().numpy().reshape(-1, d)
    ulp = 2.0 ** (np.floor(np.log2(np.maximum(np.abs(o_ref), 2.0**-14))) - 10)
    assert np.all(np.abs(o_gpu - o_ref) <= np.maximum(O_TOL, ulp))
    l_gpu = lse.double().cpu().numpy().reshape(-1)
    assert (np.abs(l_gpu - l_ref) / np.maximum(np.abs(l_ref), 1e-3)).max() <= LSE_RTOL
    # saturation: the late queries of each rank collapse onto the last key
    assert np.abs(o_gpu[-64:] - bits_to_float64(x, "fp16")[0, 0, -1]).max() <= 0.05


@pytest.mark.parametrize("causal", [False, True])
def test_block_step_and_merge_separately(oracle, causal):
    w = Workload("steps", 1, 2, 128, 4, 256, "fp16", 41, causal)
    q, k, v = api.make_qkv_bits(w)
    qd, kd, vd = (to_dev(x, w.dtype) for x in (q, k, v))
    plan = api.RingAttention(w.npes, w.chunk, w.dim, w.batch, w.heads, w.dtype, w.causal)
    rows = np.arange(w.rows)
    _, _, po, pl = oracle.ring_rows(q, k, v, w.dtype, [w.chunk] * w.npes, rows, causal=causal, tile=64, want_parts=True)
    parts_o, parts_l = [], []
    for s in range(w.npes):
        o_part, lse_part = plan.block_forward(s, qd, kd, vd)   # pre-filled with O = 0, LSE = -inf
        torch.cuda.synchronize()
        og = o_part.reshape(-1, w.dim).double().cpu().numpy()
        lg = lse_part.reshape(-1).double().cpu().numpy()
        active = np.isfinite(pl[:, s])
        assert np.array_equal(np.isfinite(lg), active)      # inactive (rank, step) pairs are left untouched
        assert np.all(og[~active] == 0)
        assert np.abs(og[active] - po[active, s]).max() <= 2e-3   # fp32 partial; only p is rounded to 16 bit
        assert (np.abs(lg[active] - pl[active, s]) / np.maximum(np.abs(pl[active, s]), 1e-3)).max() <= 1e-4
        parts_o.append(o_part.reshape(-1, w.dim))
        parts_l.append(lse_part.reshape(-1))
    plan.close()
    # merge kernel alone, on the device partials, against the oracle merge of the same numbers
    po_d, pl_d = torch.stack(parts_o), torch.stack(parts_l)
    out, lse = api.merge(po_d, pl_d, w.dtype)
    torch.cuda.synchronize()
    o_m, l_m = oracle.merge(po_d.double().cpu().numpy(), pl_d.double().cpu().numpy())
    ulp = 2.0**-10 if w.dtype == "fp16" else 2.0**-7
    assert np.abs(out.double().cpu().numpy() - o_m).max() <= 1e-5 + ulp * np.abs(o_m).max()
    assert np.abs(lse.double().cpu().numpy() - l_m).max() <= 1e-5
    check_rows(oracle, w, q, k, v, out, lse, rows)


@pytest.mark.parametrize("causal,half,d", [(False, False, 128), (True, False, 128), (True, True, 64), (False, True, 128)])
def test_row_major_partials_give_the_bits_of_slot_major_ones(causal, half, d):
    """RINGATTN_FLAG_ROW_PARTIALS only changes where a partial is kept ([rows, steps, d]: a row's steps next to each
    other): the steps, run one by one, write the numbers of the slot-major layout to their new places, and the ring
    merge gives the same bits."""
    w = Workload("rowparts", 2, 2, d, 4, 320, "bf16" if d == 128 else "fp16", 47, causal)
    q, k, v = api.make_qkv_bits(w)
    qd, kd, vd = (to_dev(x, w.dtype) for x in (q, k, v))
    results = []
    for row_major in (False, True):
        plan = api.RingAttention(w.npes, w.chunk, w.dim, w.batch, w.heads, w.dtype, w.causal, half_partials=half,
                                 row_partials=row_major)
        o_shape, l_shape = plan.parts_shapes()
        o_parts = torch.zeros(o_shape, dtype=plan.part_dtype, device="cuda")
        l_parts = torch.full(l_shape, float("-inf"), dtype=torch.float32, device="cuda")
        for s in range(w.npes):
            if row_major:
                plan.block_forward(s, qd, kd, vd, o_parts, l_parts)
            else:
                plan.block_forward(s, qd, kd, vd, o_parts[s], l_parts[s])
        out, lse = plan.merge_ring(o_parts, l_parts)
        torch.cuda.synchronize()
        plan.close()
        results.append((o_parts, l_parts, out, lse))
    (o_s, l_s, out_s, lse_s), (o_r, l_r, out_r, lse_r) = results
    assert torch.equal(o_s.permute(1, 2, 3, 0, 4), o_r) and torch.equal(l_s.permute(1, 2, 3, 0), l_r)
    assert torch.equal(out_s.view(torch.int16), out_r.view(torch.int16)) and torch.equal(lse_s, lse_r)


def test_merge_identity_and_random_parts(oracle):
    rng = np.random.default_rng(3)
    n, rows, d = 7, 1000, 64
    op = rng.standard_normal((n, rows, d)).astype(np.float32)
    lp = (4 * rng.standard_normal((n, rows))).astype(np.float32)
    lp[rng.random((n, rows)) < 0.3] = -np.inf
    lp[:, :5] = -np.inf                                  # rows with no contribution at all
    out, lse = api.merge(torch.from_numpy(op).cuda(), torch.from_numpy(lp).cuda(), "bf16")
    torch.cuda.synchronize()
    o_m, l_m = oracle.merge(op.astype(np.float64), lp.astype(np.float64))
    og, lg = out.double().cpu().numpy(), lse.double().cpu().numpy()
    assert np.all(og[:5] == 0) and np.all(np.isneginf(lg[:5]))
    assert np.abs(og - o_m).max() <= 1e-5 + 2.0**-8 * np.abs(o_m).max()
    fin = np.isfinite(l_m)
    assert np.array_equal(np.isfinite(lg), fin) and np.abs(lg[fin] - l_m[fin]).max() <= 1e-5


@pytest.mark.parametrize("causal", [False, True])
def test_reference_shaped_entry_per_rank(oracle, causal):
    # ring_attention(q, k, v, out, npes, mype, seqlen, dim, max_seq): one head, one rank per call
    w = Workload("refentry", 1, 1, 64, 4, 256, "fp16", 51, causal)
    q, k, v = api.make_qkv_bits(w)
    kd, vd = to_dev(k, w.dtype).reshape(w.seq, w.dim), to_dev(v, w.dtype).reshape(w.seq, w.dim)
    o_ref, l_ref = oracle.attention_rows(q, k, v, w.dtype, causal=causal)
    for mype in range(w.npes):
        sl = slice(mype * w.chunk, (mype + 1) * w.chunk)
        qd = to_dev(np.ascontiguousarray(q[0, 0, sl]), w.dtype)
        out = torch.empty_like(qd)
        lse = torch.empty(w.chunk, dtype=torch.float32, device="cuda")
        api.ring_attention(qd, kd, vd, out, w.npes, mype, [w.chunk] * w.npes, w.dim, w.chunk, lse=lse, causal=causal)
        assert np.abs(out.double().cpu().numpy() - o_ref[sl]).max() <= O_TOL
        assert (np.abs(lse.double().cpu().numpy() - l_ref[sl]) / np.maximum(np.abs(l_ref[sl]), 1e-3)).max() <= LSE_RTOL


def test_graph_replay_matches_eager(oracle):
    # the captured step loop is replayed several times, with eager work in between, and every
    # replay must reproduce the eager result bit for bit; new pointers trigger a re-capture
    w = Workload("graph", 2, 4, 128, 8, 128, "fp16", 61, False, graph=True)
    q, k, v = api.make_qkv_bits(w)
    qd, kd, vd = (to_dev(x, w.dtype) for x in (q, k, v))
    eager = api.RingAttention(w.npes, w.chunk, w.dim, w.batch, w.heads, w.dtype, w.causal, graph=False)
    graph = api.RingAttention(w.npes, w.chunk, w.dim, w.batch, w.heads, w.dtype, w.causal, graph=True)
    o_e, l_e = eager.forward(qd, kd, vd)
    torch.cuda.synchronize()
    o_g = torch.empty_like(o_e)
    l_g = torch.empty_like(l_e)
    for it in range(4):
        o_g.zero_()
        l_g.zero_()
        graph.forward(qd, kd, vd, o_g, l_g)
        torch.cuda.synchronize()
        assert torch.equal(o_g, o_e) and torch.equal(l_g, l_e), f"replay {it}"
        _ = (qd.float() * 2).sum().item()   # unrelated eager work between replays
    # different inputs and outputs through the same plan
    q2, k2, v2 = api.make_qkv_bits(Workload("graph2", 2, 4, 128, 8, 128, "fp16", 62, False))
    q2d, k2d, v2d = (to_dev(x, w.dtype) for x in (q2, k2, v2))
    o2_e, l2_e = eager.forward(q2d, k2d, v2d)
    o2_g, l2_g = graph.forward(q2d, k2d, v2d)
    torch.cuda.synchronize()
    assert torch.equal(o2_g, o2_e) and torch.equal(l2_g, l2_e)
    check_rows(oracle, w, q2, k2, v2, o2_g, l2_g, sample_rows(w, 256))
    eager.close()
    graph.close()


def test_host_api_checks_on_device():
    plan = api.RingAttention(2, 128, 64)
    x = torch.zeros(1, 1, 256, 64, dtype=torch.float16, device="cuda")
    with pytest.raises(ValueError):
        plan.forward(x.cpu(), x, x)                       # not device-resident (attention_api.cuh:12-13)
    with pytest.raises(ValueError):
        plan.forward(x.transpose(2, 3).contiguous().transpose(2, 3), x, x)   # not contiguous (:14-15)
    with pytest.raises(ValueError):
        plan.forward(x.bfloat16(), x, x)
    plan.close()
    with pytest.raises(api._lib.RingattnError):
        api.RingAttention(2, 101, 64, causal=True, layout="zigzag")   # the zigzag layout needs even lengths


@pytest.mark.parametrize("kernel", ["", "ring_walk_kernel"])
def test_random_plans_against_oracle(oracle, monkeypatch, kernel):
    force(monkeypatch, kernel)
    # seeded sweep over the whole parameter space at small sizes: ranks, ragged lengths, batch,
    # heads, grouped KV heads, head dim, dtype, mask, layout, explicit scale, graph replay
    rng = np.random.default_rng(2024)
    for case in range(40):
        P = int(rng.integers(1, 7))
        causal = bool(rng.integers(0, 2))
        zigzag = causal and bool(rng.integers(0, 2))
        lens = [int(rng.choice([1, 2, 31, 32, 33, 64, 100, 128, 129, 200, 256, 300])) for _ in range(P)]
        if zigzag:
            lens = [2 * ((c + 1) // 2) for c in lens]
        d = int(rng.choice([64, 128]))
        dtype = str(rng.choice(["fp16", "bf16"]))
        B, hkv, group = int(rng.integers(1, 3)), int(rng.integers(1, 3)), int(rng.integers(1, 4))
        H, S = hkv * group, sum(lens)
        scale = float(rng.choice([0.0, 0.05, 0.2]))
        graph = bool(rng.integers(0, 2))
        steps_apart = case % 3 == 2
        tag = (f"case {case}: P={P} lens={lens} B={B} H={H} hkv={hkv} d={d} {dtype} causal={causal} zigzag={zigzag} "
               f"scale={scale} graph={graph} step_partials={steps_apart}")
        print(tag, flush=True)
        w = Workload("rand", B, H, d, 1, S, dtype, 1000 + case, causal)
        q, _, _ = api.make_qkv_bits(w)
        _, k, v = api.make_qkv_bits(Workload("rand_kv", B, hkv, d, 1, S, dtype, 2000 + case, causal))
        order = api.zigzag_order(lens) if zigzag else np.arange(S)
        inv = torch.from_numpy(np.argsort(order)).cuda()
        qd, kd, vd = (to_dev(np.ascontiguousarray(x[:, :, order]), dtype) for x in (q, k, v))
        plan = api.RingAttention(P, lens, d, B, H, dtype, causal, softmax_scale=scale, graph=graph,
                                 kv_heads=hkv if group > 1 else 0, layout="zigzag" if zigzag else "contiguous",
                                 step_partials=steps_apart)
        assert kernel in ("", plan.forward_kernel()), tag
        out, lse = plan.forward(qd, kd, vd)
        if graph:                                   # a replay of the captured graph must give the same bits
            out2, lse2 = plan.forward(qd, kd, vd, torch.empty_like(out), torch.empty_like(lse))
            out2, lse2 = plan.forward(qd, kd, vd, out2, lse2)
            torch.cuda.synchronize()
            assert torch.equal(out, out2) and torch.equal(lse, lse2), tag
        torch.cuda.synchronize()
        plan.close()
        k_full, v_full = (np.repeat(x, group, axis=1) for x in (k, v))
        check_rows(oracle, w, q, k_full, v_full, out[:, :, inv].contiguous(), lse[:, :, inv].contiguous(),
                   np.arange(w.rows), scale=scale if scale > 0 else None)


def test_launch_times_of_a_timed_plan():
    w = Workload("timed", 1, 4, 128, 8, 256, "bf16", 97, True)
    q, k, v = (to_dev(x, w.dtype) for x in api.make_qkv_bits(w))
    plain = api.RingAttention(w.npes, w.chunk, w.dim, w.batch, w.heads, w.dtype, True)
    o_ref, l_ref = plain.forward(q, k, v)
    with pytest.raises(api._lib.RingattnError):
        plain.launch_times()                                  # no timing flag
    plain.close()
    timed = api.RingAttention(w.npes, w.chunk, w.dim, w.batch, w.heads, w.dtype, True, timing=True)
    with pytest.raises(api._lib.RingattnError):
        timed.launch_times()                                  # no forward yet
    out, lse = timed.forward(q, k, v)
    ms = timed.launch_times()
    torch.cuda.synchronize()
    n_items = len(timed.work_items(-1))
    assert 1 <= len(ms) <= 8 and n_items == 36 and all(0.0 < t < 1000.0 for t in ms)
    assert torch.equal(out, o_ref) and torch.equal(lse, l_ref)    # the flag changes nothing in the result
    timed.close()


def test_maximum_ranks_long_sequence(oracle):
    # the largest ring the ABI takes (64 ranks) at a real chunk size: S = 262 144 tokens, one head;
    # 64 partial slots of 135 MB, 2 080 work items; rows sampled (first rows, chunk edges, random)
    w = Workload("max_ring", 1, 1, 128, 64, 4096, "bf16", 99, True)
    q, k, v = api.make_qkv_bits(w)
    out, lse = forward(w, q, k, v)
    assert torch.isfinite(out).all() and torch.isfinite(lse).all()
    check_rows(oracle, w, q, k, v, out, lse, sample_rows(w, 192))


@pytest.mark.parametrize("w,layout", [
    (Workload("hp_many_steps", 2, 4, 128, 16, 256, "fp16", 101, False), "contiguous"),
    (Workload("hp_causal_bf16", 1, 4, 128, 4, 512, "bf16", 102, True), "contiguous"),
    (Workload("hp_d64_zigzag", 2, 2, 64, 3, 384, "fp16", 103, True), "zigzag"),
], ids=lambda x: x.name if isinstance(x, Workload) else x)
def test_half_precision_partials(oracle, w, layout):
    q, k, v = api.make_qkv_bits(w)
    order = api.zigzag_order([w.chunk] * w.npes) if layout == "zigzag" else np.arange(w.seq)
    inv = torch.from_numpy(np.argsort(order)).cuda()
    qd, kd, vd = (to_dev(np.ascontiguousarray(x[:, :, order]), w.dtype) for x in (q, k, v))
    full = api.RingAttention(w.npes, w.chunk, w.dim, w.batch, w.heads, w.dtype, w.causal, layout=layout, step_partials=True)
    half = api.RingAttention(w.npes, w.chunk, w.dim, w.batch, w.heads, w.dtype, w.causal, layout=layout, step_partials=True,
                             half_partials=True)
    wb = half.lib.ringattn_workspace_bytes
    assert wb(half.params) * (4 * w.dim + 4) == wb(full.params) * (2 * w.dim + 4)
    o32, l32 = full.forward(qd, kd, vd)
    o16, l16 = half.forward(qd, kd, vd)
    torch.cuda.synchronize()
    # same parity bar against the oracle, and close to the fp32-partial result: each merged part
    # carries at most half an fp16 ulp of max |V|, plus one ulp of the output type
    check_rows(oracle, w, q, k, v, o16[:, :, inv].contiguous(), l16[:, :, inv].contiguous(), np.arange(w.rows),
               half_partials=True)
    vmax = np.abs(bits_to_float64(v, w.dtype)).max()
    ulp_out = 2.0**-10 if w.dtype == "fp16" else 2.0**-7
    assert (o16.float() - o32.float()).abs().max().item() <= vmax * 2.0**-11 + ulp_out * vmax
    assert torch.equal(l16, l32)                       # the partial LSEs stay fp32
    # a step's fp16 partial is the fp32 partial rounded to nearest
    for s in (0, w.npes - 1):
        p32, pl32 = full.block_forward(s, qd, kd, vd)
        p16, pl16 = half.block_forward(s, qd, kd, vd)
        torch.cuda.synchronize()
        assert p16.dtype == torch.float16 and torch.equal(p16, p32.half()) and torch.equal(pl16, pl32)
    # merge of caller-held fp16 partials
    parts = torch.zeros((w.npes,) + tuple(o16.shape), dtype=torch.float16, device="cuda")
    lparts = torch.full((w.npes,) + tuple(l16.shape), float("-inf"), dtype=torch.float32, device="cuda")
    for s in range(w.npes):
        half.block_forward(s, qd, kd, vd, parts[s], lparts[s])
    o_m, l_m = half.merge_ring(parts, lparts)
    torch.cuda.synchronize()
    assert torch.equal(o_m, o16) and torch.equal(l_m, l16)
    full.close()
    half.close()


@pytest.mark.parametrize("seqlen,causal,layout,d,dtype,hkv,half", [
    ((256, 256, 256, 256), True, "contiguous", 128, "bf16", 0, False),
    ((256, 256, 256, 256), False, "contiguous", 64, "fp16", 0, False),
    ((512, 256, 768), True, "zigzag", 128, "bf16", 2, False),
    ((100, 334, 2, 78), True, "zigzag", 128, "fp16", 0, True),
    ((100, 333, 1, 77), True, "contiguous", 64, "bf16", 0, False),
])
def test_rank_local_ring_equals_the_all_rank_forward(seqlen, causal, layout, d, dtype, hkv, half):
    # A ring of one process per GPU, replayed rank by rank on this GPU: every rank holds only its
    # own Q rows and, at step s, the K/V chunk of rank (r + s) mod P in a buffer of its own (what
    # the exchange would have delivered).  Same work items, so the same bits as a ringattn_fwd that
    # keeps the steps apart; the default forward (state carried in registers) agrees to rounding.
    P, S, B, H = len(seqlen), sum(seqlen), 2, 4
    w = Workload("rank_local", B, H, d, 1, S, dtype, 111, causal)
    q, _, _ = api.make_qkv_bits(w)
    _, k, v = api.make_qkv_bits(Workload("rank_local_kv", B, hkv or H, d, 1, S, dtype, 112, causal))
    qd, kd, vd = (to_dev(x, dtype) for x in (q, k, v))
    plan = api.RingAttention(P, list(seqlen), d, B, H, dtype, causal, kv_heads=hkv, layout=layout, half_partials=half,
                             step_partials=True)
    out, lse = plan.forward(qd, kd, vd)
    carried = api.RingAttention(P, list(seqlen), d, B, H, dtype, causal, kv_heads=hkv, layout=layout)
    out_c, lse_c = carried.forward(qd, kd, vd)
    torch.cuda.synchronize()
    carried.close()
    # per row: within two storage ulps of the row's largest element (three with fp16 partials)
    ulp = 2.0**-10 if dtype == "fp16" else 2.0**-7
    row_max = out.float().abs().amax(-1, keepdim=True)
    exp2 = torch.exp2(torch.floor(torch.log2(row_max.clamp_min(2.0**-14))))
    assert ((out_c.float() - out.float()).abs() <= (3 if half else 2) * ulp * exp2).all()
    assert torch.allclose(lse_c, lse, rtol=1e-5, atol=1e-5)
    start = np.concatenate([[0], np.cumsum(seqlen)])
    for r in range(P):
        rows = slice(start[r], start[r + 1])
        q_r = qd[:, :, rows].contiguous()
        o_parts = torch.zeros((P, B, H, seqlen[r], d), dtype=plan.part_dtype, device="cuda")
        l_parts = torch.full((P, B, H, seqlen[r]), float("-inf"), dtype=torch.float32, device="cuda")
        for s in range(P):
            j = (r + s) % P
            k_j = kd[:, :, start[j]:start[j + 1]].contiguous()      # the chunk the ring delivered
            v_j = vd[:, :, start[j]:start[j + 1]].contiguous()
            plan.rank_step_forward(r, s, q_r, k_j, v_j, o_parts[s], l_parts[s])
        o_r, l_r = plan.rank_merge(r, o_parts, l_parts)
        torch.cuda.synchronize()
        assert torch.equal(o_r, out[:, :, rows]) and torch.equal(l_r, lse[:, :, rows]), f"rank {r}"
    plan.close()
    # the same ring with a row's steps next to each other in the rank's partials (RINGATTN_FLAG_ROW_PARTIALS)
    plan = api.RingAttention(P, list(seqlen), d, B, H, dtype, causal, kv_heads=hkv, layout=layout, half_partials=half,
                             row_partials=True)
    for r in range(P):
        rows = slice(start[r], start[r + 1])
        q_r = qd[:, :, rows].contiguous()
        o_shape, l_shape = plan.rank_parts_shapes(r)
        o_parts = torch.zeros(o_shape, dtype=plan.part_dtype, device="cuda")
        l_parts = torch.full(l_shape, float("-inf"), dtype=torch.float32, device="cuda")
        for s in range(P):
            j = (r + s) % P
            plan.rank_step_forward(r, s, q_r, kd[:, :, start[j]:start[j + 1]].contiguous(),
                                   vd[:, :, start[j]:start[j + 1]].contiguous(), o_parts, l_parts)
        o_r, l_r = plan.rank_merge(r, o_parts, l_parts)
        torch.cuda.synchronize()
        assert torch.equal(o_r, out[:, :, rows]) and torch.equal(l_r, lse[:, :, rows]), f"rank {r}, row-major partials"
    plan.close()
