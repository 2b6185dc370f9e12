"""What the compiler made of the attention kernels: every instantiation must fit two waves per
SIMD (256 registers) without scratch memory in its loops, and the steady key loops of the d = 128
ones -- the loops that hold 64 MFMAs, four 32-key blocks -- must carry one barrier per two tiles and
read their fragments ahead of the MFMAs.
Compiles the kernels to assembly for gfx950; needs hipcc but no GPU."""
import os
import re
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def loops_of(asm):
    """(label, instructions) of every innermost loop of a function body: from the block the
    compiler marks as the loop header to the last branch back to it (or to the block of wait
    and barrier it sometimes places right in front of the header)."""
    lines = asm.split("\n")
    where = {}
    for i, line in enumerate(lines):
        m = re.match(r"^(\.LBB\d+_\d+):", line)
        if m:
            where[m.group(1)] = i
    out = []
    for i, line in enumerate(lines):
        if "Inner Loop Header" not in line:
            continue
        head = max((k for k in where.values() if k <= i), default=None)
        if head is None:
            continue
        targets = {lab for lab, k in where.items() if head - 12 <= k <= head}
        last = None
        for j in range(i + 1, len(lines)):
            m = re.match(r"^\s*s_(?:cbranch_\w+|branch)\s+(\.LBB\d+_\d+)\s*$", lines[j])
            if m and m.group(1) in targets:
                last = j
        if last is not None:
            body = [l.strip() for l in lines[i + 1:last + 1]]
            out.append((lines[head].split(":")[0], [l for l in body if l and not l.startswith((";", "."))]))
    return out


def compile_to_asm(source, out):
    """Assembly of one kernel source plus the compiler's per-kernel resource remarks."""
    hipcc = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
    if not os.path.exists(hipcc):
        pytest.skip("no hipcc")
    from ringattention_amd import _build
    src = os.path.join(_build.CSRC, source)
    flags = [f for f in _build.HIPCC_FLAGS if f not in ("-shared", "-fPIC", "-pthread")]
    res = subprocess.run([hipcc] + flags + ["-S", "--cuda-device-only", "-Rpass-analysis=kernel-resource-usage",
                                            "-I", os.path.join(ROOT, "include"), "-I", _build.CSRC, src, "-o", str(out)],
                         capture_output=True, text=True, timeout=900)
    assert res.returncode == 0, res.stderr[-2000:]
    usage = {}
    name = None
    for line in res.stderr.split("\n"):
        m = re.search(r"Function Name: (\S+)", line)
        if m:
            name = m.group(1)
            usage[name] = {}
        for key in ("VGPRs", "ScratchSize [bytes/lane]", "Occupancy [waves/SIMD]", "LDS Size [bytes/block]"):
            m = re.search(re.escape(key) + r": (\d+)", line)
            if m and name:
                usage[name][key] = int(m.group(1))
    return out.read_text(), usage


def steady_loops(asm, kernel):
    start = asm.index("\n" + kernel + ":")
    end = asm.index(".amdhsa_kernel " + kernel, start)
    return [(lab, ins) for lab, ins in loops_of(asm[start:end]) if sum(i.startswith("v_mfma") for i in ins) == 64]


def body_of(asm, kernel):
    start = asm.index("\n" + kernel + ":")
    return asm[start:asm.index(".amdhsa_kernel " + kernel, start)]


def check_steady_loops(asm, n, barriers):
    """The four loops of a d = 128 instantiation: plain and masked groups, for each half of the workgroup."""
    steady = steady_loops(asm, n)
    assert len(steady) == 4, (n, len(steady))
    for lab, ins in steady:
        assert sum(i.startswith("s_barrier") for i in ins) in barriers, (n, lab)   # one per two tiles
        # fragments are read six and more ahead: a wait for the last read comes at the end of a phase and not at every MFMA
        assert sum(bool(re.match(r"s_waitcnt .*lgkmcnt\(0\)", i)) for i in ins) <= 12, (n, lab)


def test_walk_kernel_runs_two_waves_per_simd_without_spills(tmp_path):
    asm, usage = compile_to_asm("ringattn_walk.hip", tmp_path / "walk.s")
    walks = {n: u for n, u in usage.items() if "ring_walk_kernel" in n}
    # {fp16, bf16} x {64, 128} x {carried state; partials as fp32; partials as fp16}
    assert len(walks) == 12
    for n, u in walks.items():
        carried = n.endswith("Lb0ELb1EEEvNS_9BlockArgsE")
        d64 = "Li64E" in n
        # (a register of the d = 64 variants that store partials waits in scratch from the start to the stores)
        assert u["ScratchSize [bytes/lane]"] <= (8 if d64 and not carried else 0), (n, u)
        assert not any(i.startswith("scratch_") for _, ins in loops_of(body_of(asm, n)) for i in ins), n
        # eight waves per workgroup; d = 64: two workgroups per compute unit (+12 % measured)
        assert u["VGPRs"] <= (128 if d64 else 256), (n, u)
        assert u["LDS Size [bytes/block]"] == (32768 if d64 else 65536), (n, u)   # K and V rings, four tiles of 32 keys each
        if not d64:
            # (where partials are stored the first barrier of a chunk may have been taken before the stores, which puts
            # it on a side path of the loop)
            check_steady_loops(asm, n, (2,) if carried else (1, 2))


def test_walk_kernel_that_merges_its_steps(tmp_path):
    """The same program with the result of the rows in 32 registers more and, at d = 128, 64 KB of LDS."""
    asm, usage = compile_to_asm("ringattn_steps.hip", tmp_path / "steps.s")
    kernels = {n: u for n, u in usage.items() if "ring_walk_kernel" in n}
    assert len(kernels) == 8   # {fp16, bf16} x {64, 128} x {partials rounded to fp16 or not}
    for n, u in kernels.items():
        d64 = "Li64E" in n
        assert u["ScratchSize [bytes/lane]"] == 0 and u["VGPRs"] <= 256, (n, u)
        assert u["LDS Size [bytes/block]"] == (32768 if d64 else 131072), (n, u)
        if not d64:
            check_steady_loops(asm, n, (2,))


def test_thin_walk_kernel(tmp_path):
    """thin::ring_walk_kernel: four waves that a compute unit may hold twice, rings of eight tiles, and one loop of eight tiles (64
    MFMAs) with a barrier per two."""
    asm, usage = compile_to_asm("ringattn_thin.hip", tmp_path / "thin.s")
    kernels = {n: u for n, u in usage.items() if "ring_walk_kernel" in n}
    assert len(kernels) == 8   # {fp16, bf16} x {fp32, fp16 partials} x {stored, merged}
    for n, u in kernels.items():
        assert u["ScratchSize [bytes/lane]"] == 0 and u["VGPRs"] <= 256, (n, u)
        assert u["LDS Size [bytes/block]"] == 65536, (n, u)
        (_, ins), = steady_loops(asm, n)
        assert sum(i.startswith("s_barrier") for i in ins) == 4, n


def test_walk64_kernel_runs_one_wave_per_simd(tmp_path):
    """ring_walk64_kernel (64 query rows per wave) is laid out for one wave per SIMD: more than 256 registers, the two
    eight-tile rings plus the chunk list in LDS, and no scratch."""
    asm, usage = compile_to_asm("ringattn_walk64.hip", tmp_path / "walk64.s")
    kernels = {n: u for n, u in usage.items() if "ring_walk64_kernel" in n}
    # fp16, bf16 x (d = 128: state carried, fp32 partials, fp16 partials; d = 64: state carried)
    assert len(kernels) == 8
    for n, u in kernels.items():
        d64 = "ELi64E" in n
        assert u["Occupancy [waves/SIMD]"] == 1, (n, u)
        assert u["LDS Size [bytes/block]"] == 2 * 8 * (4096 if d64 else 8192) + 8 * (64 + 4), (n, u)
        assert u["ScratchSize [bytes/lane]"] == 0, (n, u)
        start = asm.index("\n" + n + ":")
        body = asm[start:asm.index(".amdhsa_kernel " + n, start)]
        blocks = body.split(";;#ASMSTART")[1:]
        loop = max((b.split(";;#ASMEND")[0] for b in blocks), key=len)
        assert loop.count("v_mfma_f32_32x32x16") >= 8 * (16 if d64 else 32)    # eight unrolled iterations of 32 (16) MFMAs, and the tails
        assert "scratch_" not in loop


def test_every_wave_of_the_workgroup_enters_the_hand_scheduled_loop(tmp_path):
    """The loop holds the workgroup's barriers and each wave's share of the tile loads: from the last barrier in front of it on
    no branch may lead past it."""
    for source, kernel in (("ringattn_walk64.hip", "ring_walk64_kernel"), ("ringattn_pair.hip", "ring_pair_kernel")):
        asm, usage = compile_to_asm(source, tmp_path / "loop.s")
        for n in (n for n in usage if kernel in n):
            start = asm.index("\n" + n + ":")
            lines = asm[start:asm.index(".amdhsa_kernel " + n, start)].split("\n")
            at = {m.group(1): i for i, m in enumerate(re.match(r"(\.LBB\d+_\d+):", l) for l in lines) if m}
            begins = [i for i, l in enumerate(lines) if ";;#ASMSTART" in l]
            ends = [next(j for j in range(i, len(lines)) if ";;#ASMEND" in lines[j]) for i in begins]
            begin, end = max(zip(begins, ends), key=lambda x: x[1] - x[0])
            barrier = max(i for i in range(begin) if lines[i].strip() == "s_barrier")
            for l in lines[barrier:begin]:
                m = re.match(r"\s*s_c?branch\S*\s+(\.LBB\d+_\d+)", l)
                assert not m or at[m.group(1)] < end, (n, l)


@pytest.mark.parametrize("source", ["ringattn_walk.hip", "ringattn_steps.hip", "ringattn_thin.hip", "ringattn_walk64.hip"])
def test_no_lds_transfer_reads_a_scalar_register_fresh_from_a_vector_instruction(source, tmp_path):
    """A vector instruction that writes a scalar register (v_readfirstlane, v_readlane, a compare into a register
    pair) must be five wait states ahead of a memory instruction that reads that register as its base address; the
    direct-to-LDS loads of these kernels sit in inline assembly, where the compiler inserts no such wait.  Every
    global_load_lds in the compiled code is checked against the instructions in front of it."""
    asm, _ = compile_to_asm(source, tmp_path / "hazard.s")
    lines = asm.split("\n")
    loads = 0
    for i, line in enumerate(lines):
        m = re.search(r"global_load_lds_dwordx4 \S+, s\[(\d+):(\d+)\]", line)
        if not m:
            continue
        loads += 1
        lo, hi = int(m.group(1)), int(m.group(2))
        wait_states, j = 0, i - 1
        while j > 0 and wait_states < 5:
            t = lines[j].strip()
            j -= 1
            if not t or t[0] in ";." or t.endswith(":"):
                continue
            w = re.match(r"(?:v_readfirstlane_b32|v_readlane_b32) s(\d+),", t) or re.match(r"v_cmp\S* s\[(\d+):", t)
            assert not (w and lo <= int(w.group(1)) <= hi), (i, t, line.strip(), wait_states)
            nop = re.match(r"s_nop (\d+)", t)
            wait_states += int(nop.group(1)) + 1 if nop else 1
    assert loads > 100
