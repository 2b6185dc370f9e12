"""Which kernel the host gives a forward to (ringattn_plan_forward_kernel), without a GPU."""
import pytest

from ringattention_amd import api

SWITCHES = ("RINGATTN_WIDE", "RINGATTN_WIDE_D64", "RINGATTN_WIDE_PARTIALS", "RINGATTN_SPLIT", "RINGATTN_PAIR")


def chosen(monkeypatch, lens, d, heads=1, causal=False, layout="contiguous", env=(), **more):
    for name in SWITCHES:
        monkeypatch.delenv(name, raising=False)
    for name, value in dict(env).items():
        monkeypatch.setenv(name, value)
    plan = api.RingAttention(len(lens), list(lens), d, 1, heads, "fp16", causal, layout=layout, **more)
    try:
        return plan.forward_kernel()
    finally:
        plan.close()


@pytest.mark.parametrize("d", [128, 64])
@pytest.mark.parametrize("env", [{}, {"RINGATTN_PAIR": "1"}])
def test_a_key_range_that_begins_beyond_4_gib_of_its_head(monkeypatch, d, env):
    """The generated loops keep the byte offset of a range within its head in 32 bits.  A forward whose ranges begin further on
    (zigzag, 2^32 bytes of K and more in front of a rank) runs on ring_walk_kernel, whose offsets are 64-bit; one range
    from row 0 on may be as long as it likes."""
    rows = 2 ** 32 // (2 * d)   # of a head, in 4 GiB
    loops = ("ring_walk64_kernel", "ring_pair_kernel")
    assert chosen(monkeypatch, (rows // 2, rows // 4), d, causal=True, layout="zigzag", env=env) in loops
    assert chosen(monkeypatch, (rows, 256), d, causal=True, layout="zigzag", env=env) == "ring_walk_kernel"
    assert chosen(monkeypatch, (rows, 256), d, causal=True, env=env) in loops
    assert chosen(monkeypatch, (2 * rows,), d, env=env) in loops


def test_per_step_partials_of_chunks_that_begin_beyond_4_gib(monkeypatch):
    """The same of launches that walk the chunks one by one (the plan holds caller memory it never touches here)."""
    rows = 2 ** 24
    for lens, kernel in (((rows // 2, rows // 2), "ring_walk64_kernel"), ((rows // 2, rows // 2, 4096), "ring_walk_kernel")):
        assert chosen(monkeypatch, lens, 128, causal=True, env={"RINGATTN_WIDE_PARTIALS": "1"}, step_partials=True,
                      workspace=(1 << 20, 1 << 60)) == kernel


@pytest.mark.parametrize("lens,heads,causal", [((2048,), 1, False), ((8192,), 4, False), ((4400,), 16, True), ((1024,) * 8, 8, False)])
def test_switches_that_name_a_256_row_kernel(monkeypatch, lens, heads, causal):
    """RINGATTN_WIDE=0 and, at d = 64, RINGATTN_WIDE_D64=0 keep a forward on ring_walk_kernel whatever its size; the latter
    says nothing about d = 128."""
    for d in (64, 128):
        assert chosen(monkeypatch, lens, d, heads, causal, env={"RINGATTN_WIDE": "0"}) == "ring_walk_kernel"
    assert chosen(monkeypatch, lens, 64, heads, causal, env={"RINGATTN_WIDE_D64": "0"}) == "ring_walk_kernel"
    assert chosen(monkeypatch, lens, 128, heads, causal, env={"RINGATTN_WIDE_D64": "0"}) == chosen(monkeypatch, lens, 128, heads, causal)


@pytest.mark.parametrize("d,heads,tokens,causal,kernel", [
    # us on ring_walk_kernel and ring_pair_kernel, logits N(0, 1); the same with logits N(0, 81)
    (64, 24, 3000, False, "ring_walk_kernel"),    # 91, 90; 103, 140
    (64, 16, 6001, False, "ring_walk_kernel"),    # 185, 174; 204, 247
    (64, 12, 6000, False, "ring_walk_kernel"),    # 175, 165; 193, 233
    (64, 16, 4400, True, "ring_pair_kernel"),     # 78, 62; 87, 89
    (64, 4, 8191, False, "ring_pair_kernel"),     # 129, 82; 146, 111
    (128, 16, 4400, True, "ring_pair_kernel"),    # 123, 95; 120, 129
    (128, 8, 8191, True, "ring_pair_kernel"),     # 180, 134; 204, 187
    (128, 32, 4400, False, "ring_walk_kernel"),   # 337, 322; 380, 439
])
def test_ragged_lengths_leave_ring_walk_kernel_for_a_clear_lead_only(monkeypatch, d, heads, tokens, causal, kernel):
    """Where the 256-row kernel is ring_walk_kernel (no multiple of 32), a small lead of ring_pair_kernel on flat logits is lost,
    and more, on peaked ones."""
    assert chosen(monkeypatch, (tokens,), d, heads, causal) == kernel
