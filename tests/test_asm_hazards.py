"""Some kernels issue LDS reads, and the prefill attention MFMAs too, as hand-written instructions whose results the compiler
believes to be present as soon as the instruction has been issued.  Two classes of mistakes follow from that, both
silent at compile time and sporadic at run time:

  * an instruction the compiler places (a register copy on a branch edge, a spill, an address computation in a register
    it considers free) touches a register while the read that fills it is still in flight;
  * an instruction the compiler places reads an MFMA's result without the wait states the hardware needs between the
    two, because the compiler keeps that distance only for MFMAs it can see.

These tests compile the kernels' translation unit to gfx950 assembly (no GPU needed).  The prefill attention is scanned in
listing order for both, with the stricter rule that no branch is reached while a read is in flight; every kernel with
hand-written reads (the prefill GEMMs fetch ahead under a branch between a read and its wait) is scanned for the first along
all paths.  The scanners are themselves checked against short listings that contain each mistake.
"""
import os
import re
import subprocess

import pytest

from seq2seqsharp_amd import build as B

KERNEL = re.compile(r"^(_ZN5tship\w+):")
ATTENTION = "attn_mfma_prefill_kernel"


def _regs(tok):
    m = re.fullmatch(r"v\[(\d+):(\d+)\]", tok)
    if m:
        return set(range(int(m.group(1)), int(m.group(2)) + 1))
    m = re.fullmatch(r"v(\d+)", tok)
    return {int(m.group(1))} if m else set()


def _kernels(text):
    """-> {name: [(line number, instruction text, written by hand)]}"""
    out, name, inasm = {}, None, False
    for ln, line in enumerate(text.split("\n"), 1):
        m = KERNEL.match(line)
        if m:
            name = m.group(1)
            out[name] = []
            continue
        if name is None:
            continue
        if line.startswith(".Lfunc_end"):
            name = None
            continue
        s = line.strip()
        if s.startswith(";;#ASMSTART"):
            inasm = True
        elif s.startswith(";;#ASMEND"):
            inasm = False
        elif s and not s.startswith(";") and (not s.startswith(".") or s.startswith(".LBB")):
            out[name].append((ln, s, inasm))
    return out


def reads_in_flight(instrs):
    """Findings: instructions that touch the destination of a hand-written ds_read_b128 before an lgkmcnt wait covers
    it, and branches or labels reached with such reads pending (the compiler may copy registers on an edge)."""
    pend, bad = [], []
    for ln, s, inasm in instrs:
        op = s.split()[0]
        toks = [t.strip(",") for t in s.split()[1:]]
        if s.startswith(".LBB"):
            if pend:
                bad.append((ln, "label with %d reads pending" % len(pend)))
            continue
        if op == "s_waitcnt":
            m = re.search(r"lgkmcnt\((\d+)\)", s)
            if m:
                n = int(m.group(1))
                pend = pend[len(pend) - n:] if n else []
            continue
        if op == "ds_read_b128" and inasm:
            pend.append(_regs(toks[0]))
            continue
        if op.startswith("s_cbranch") or op == "s_branch":
            if pend:
                bad.append((ln, "branch with %d reads pending" % len(pend)))
            continue
        used = set().union(*[_regs(t) for t in toks]) if toks else set()
        hot = set().union(*pend) if pend else set()
        if used & hot:
            bad.append((ln, "'%s' touches registers of a read in flight" % s))
    return bad


def reads_in_flight_on_paths(instrs):
    """The same for code that branches between a read and its wait: instructions that touch the destination of a hand-written
    ds_read_b128 (or take their address from one) before a wait covers it, on any path through the branches."""
    at = {s.split(":")[0]: i for i, (_, s, _) in enumerate(instrs) if s.startswith(".LBB")}
    bad, seen, todo = set(), set(), [(0, ())]
    while todo:
        i, pend = todo.pop()
        while i < len(instrs):
            ln, s, inasm = instrs[i]
            op = s.split()[0]
            toks = [t.strip(",") for t in s.split()[1:]]
            if s.startswith(".LBB"):
                if (i, pend) in seen:
                    break
                seen.add((i, pend))
            elif op == "s_waitcnt":
                m = re.search(r"lgkmcnt\((\d+)\)", s)
                if m:
                    pend = pend[max(0, len(pend) - int(m.group(1))):]
            elif op == "s_branch":
                i = at[toks[0]]
                continue
            elif op.startswith("s_cbranch"):
                todo.append((at[toks[0]], pend))
            elif op == "s_endpgm":
                break
            else:
                hand_read = op == "ds_read_b128" and inasm
                hot = set().union(*pend) if pend else set()
                if set().union(*[_regs(t) for t in toks[1 if hand_read else 0:]], set()) & hot:
                    bad.add((ln, "'%s' touches registers of a read in flight" % s))
                if hand_read:
                    pend += (frozenset(_regs(toks[0])),)
            i += 1
    return sorted(bad)


def requests_before_the_first_wait(instrs):
    """Vector loads in front of the first wait for one, and vector loads in all."""
    ops = [s for _, s, _ in instrs]
    first = next((i for i, s in enumerate(ops) if s.startswith("s_waitcnt") and "vmcnt" in s), len(ops))
    return sum(s.startswith("global_load_dwordx4") for s in ops[:first]), sum(s.startswith("global_load_dwordx4") for s in ops)


def mfma_results_read_early(instrs, distance=20):
    """Findings: instructions other than MFMAs that use the destination of a hand-written MFMA fewer than `distance`
    issue slots behind it (s_nop n counts n + 1; the hardware's largest requirement for this MFMA shape is below 20)."""
    bad, n = [], len(instrs)
    for i, (l0, s0, a0) in enumerate(instrs):
        if not (a0 and s0.startswith("v_mfma")):
            continue
        dst = _regs(s0.split()[1].strip(","))
        dist = 0
        for j in range(i + 1, min(n, i + 60)):
            l1, s1, _ = instrs[j]
            op = s1.split()[0]
            if op == "s_nop":
                dist += int(s1.split()[1]) + 1
            elif op == "s_branch":
                break
            elif op.startswith("s_") or s1.startswith(".LBB") or op.startswith("ds_") or op.startswith("global_"):
                dist += 1
            else:
                used = set().union(*[_regs(t.strip(",")) for t in s1.split()[1:]])
                if used & dst and not op.startswith("v_mfma"):
                    bad.append((l1, "'%s' %d slots behind the MFMA at line %d" % (s1, dist, l0)))
                dist += 4 if op.startswith("v_mfma") else 1
            if dist >= distance:
                break
    return bad


def _listing(body):
    return "_ZN5tship24attn_mfma_prefill_kernelILi64ELi4ELb0ELi1EEEvNS_8AttnArgsE:\n" + body + "\n.Lfunc_end0:\n"


def test_scanners_find_each_mistake():
    asm = lambda s: ";;#ASMSTART\n\t%s\n;;#ASMEND" % s
    ok = _listing("\n".join([asm("ds_read_b128 v[2:5], v9 offset:0"), "\tv_add_f32_e32 v8, v7, v6",
                             asm("s_waitcnt lgkmcnt(0)"), "\tv_mov_b32_e32 v4, v10"]))
    assert reads_in_flight(_kernels(ok).popitem()[1]) == []
    # a register of the read used as an address before the wait
    late = _listing("\n".join([asm("ds_read_b128 v[2:5], v9 offset:0"), "\tv_lshl_add_u64 v[4:5], s[4:5], 0, v[68:69]",
                               asm("s_waitcnt lgkmcnt(0)")]))
    assert reads_in_flight(_kernels(late).popitem()[1])
    # a wait count that leaves the read outstanding
    count = _listing("\n".join([asm("ds_read_b128 v[2:5], v9 offset:0"), asm("ds_read_b128 v[12:15], v9 offset:1024"),
                                asm("s_waitcnt lgkmcnt(1)"), "\tv_mov_b32_e32 v20, v13"]))
    assert reads_in_flight(_kernels(count).popitem()[1])
    # a copy on a branch edge before the wait
    edge = _listing("\n".join([asm("ds_read_b128 v[2:5], v9 offset:0"), "\ts_cbranch_scc1 .LBB0_2", ".LBB0_2:",
                               "\tv_mov_b64_e32 v[20:21], v[2:3]", asm("s_waitcnt lgkmcnt(0)")]))
    assert reads_in_flight(_kernels(edge).popitem()[1])
    # an MFMA's result copied two instructions behind it; fine behind enough idle instructions
    mf = asm("v_mfma_f32_16x16x32_f16 v[26:29], v[50:53], v[60:63], v[26:29]")
    early = _listing("\n".join([mf, "\tv_max_f32_e32 v1, v2, v3", "\tv_mov_b32_e32 v40, v27"]))
    assert mfma_results_read_early(_kernels(early).popitem()[1])
    padded = _listing("\n".join([mf, asm("s_nop 15\n\ts_nop 15"), "\tv_mov_b32_e32 v40, v27"]))
    assert mfma_results_read_early(_kernels(padded).popitem()[1]) == []


    # the same mistakes behind a branch that leaves the wait out, and a loop laid out behind another one
    branch = lambda wait: _listing("\n".join([asm("ds_read_b128 v[2:5], v9 offset:0"), "\ts_cbranch_scc1 .LBB0_2", "\tv_add_f32_e32 v8, v7, v6",
                                              asm("s_waitcnt lgkmcnt(0)") if wait else "\ts_nop 0", ".LBB0_3:", "\tv_mov_b32_e32 v10, v4", "\ts_endpgm",
                                              ".LBB0_2:", asm("s_waitcnt lgkmcnt(0)"), "\ts_branch .LBB0_3"]))
    assert reads_in_flight_on_paths(_kernels(branch(True)).popitem()[1]) == []
    assert reads_in_flight_on_paths(_kernels(branch(False)).popitem()[1])
    for listing in (late, count, edge):
        assert reads_in_flight_on_paths(_kernels(listing).popitem()[1])
    assert reads_in_flight_on_paths(_kernels(ok).popitem()[1]) == []
    address = _listing("\n".join([asm("ds_read_b128 v[2:5], v9 offset:0"), asm("ds_read_b128 v[12:15], v3 offset:0"), asm("s_waitcnt lgkmcnt(0)")]))
    assert reads_in_flight_on_paths(_kernels(address).popitem()[1])
    serial = _listing("\tglobal_load_dwordx4 v[2:5], v[0:1], off\n\ts_waitcnt vmcnt(0)\n\tglobal_load_dwordx4 v[6:9], v[0:1], off")
    assert requests_before_the_first_wait(_kernels(serial).popitem()[1]) == (1, 2)


@pytest.fixture(scope="module")
def assembly(tmp_path_factory):
    if not os.path.exists(B.HIPCC):
        pytest.skip("hipcc is not installed")
    out = tmp_path_factory.mktemp("asm") / "tship_gpt.s"
    cmd = [B.HIPCC] + B.FLAGS + ["--cuda-device-only", "-S", os.path.join(B.CSRC, "tship_gpt.hip"), "-o", str(out)]
    r = subprocess.run(cmd, capture_output=True, text=True)
    assert r.returncode == 0, r.stderr[-2000:]
    return out.read_text()


@pytest.mark.timeout(900)
def test_prefill_attention_assembly_has_neither_mistake(assembly):
    kernels = {n: i for n, i in _kernels(assembly).items() if ATTENTION in n}
    assert len(kernels) >= 32                      # head sizes 64 / 128, 1 / 2 / 4 / 8 query heads per KV head, plain / padded, one / two column groups
    for name, instrs in kernels.items():
        assert any(a and s.startswith("ds_read_b128") for _, s, a in instrs), name
        assert any(a and s.startswith("v_mfma") for _, s, a in instrs), name
        assert reads_in_flight(instrs) == [], name
        assert mfma_results_read_early(instrs) == [], name


@pytest.mark.timeout(900)
def test_no_kernel_touches_a_read_in_flight(assembly):
    kernels = {n: i for n, i in _kernels(assembly).items() if any(a and s.startswith("ds_read_b128") for _, s, a in i)}
    for kernel, instances in (("mid_gemm_f16_kernel", 15), ("big_gemm3_f16_kernel", 3), (ATTENTION, 32)):
        assert sum(kernel in n for n in kernels) >= instances, kernel
    for name, instrs in kernels.items():
        assert reads_in_flight_on_paths(instrs) == [], name


@pytest.mark.timeout(900)
def test_moved_cache_rows_are_in_flight_together(assembly):
    """rows_move_kernel: a thread's 16 bytes of all rows are requested before it waits for the first, and stay in registers."""
    kernels = {n: i for n, i in _kernels(assembly).items() if "rows_move_kernel" in n}
    rows = sorted(int(re.search(r"rows_move_kernelILi(\d+)", n).group(1)) for n in kernels)
    assert rows == [4, 8, 16]
    for name, instrs in kernels.items():
        n = int(re.search(r"rows_move_kernelILi(\d+)", name).group(1))
        assert requests_before_the_first_wait(instrs) == (n, n), name
        assert not any("scratch_" in s or s.startswith("ds_") for _, s, _ in instrs), name
