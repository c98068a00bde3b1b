"""Static check of the GEMM and attention kernels' ISA (no GPU needed: hipcc cross-compiles).

The scale-accumulate MFMA of csrc/jf_gemm.hip is written as inline asm (its accumulator input has to be an inline
constant), so the compiler's hazard recogniser does not know it is an MFMA.  A vector instruction that reads or
writes an MFMA's destination registers needs up to 19 wait states after the MFMA issues; the kernel guarantees
them by program order (the result is consumed one accumulation later).  This test compiles the file to assembly
and verifies that guarantee for every such MFMA in every instantiation, that the table of scale products which two waves
fill together is written before the barrier behind it, and that neither these kernels nor those of
csrc/jf_attention.hip spill in their main loops."""
import os
import re
import shutil
import subprocess
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
PKG = os.path.join(ROOT, "jetfire-int8training_amd")
WAIT_STATES = 19


def _regs(text):
    out = set()
    for m in re.finditer(r"\bv\[(\d+):(\d+)\]|\bv(\d+)\b", text):
        if m.group(1):
            out |= set(range(int(m.group(1)), int(m.group(2)) + 1))
        else:
            out.add(int(m.group(3)))
    return out


def _isa(tmp_path_factory, source):
    hipcc = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
    if not os.path.exists(hipcc):
        pytest.skip("hipcc not available")
    sys.path.insert(0, PKG)
    import build_ext
    out = tmp_path_factory.mktemp("isa") / "out.s"
    flags = [f for f in build_ext.HIP_FLAGS if f not in ("-shared", "-fPIC")]
    subprocess.check_call([hipcc] + flags + ["-S", "--cuda-device-only", "-o", str(out),
                                             os.path.join(PKG, "csrc", source)], stderr=subprocess.DEVNULL)
    return out.read_text().split("\n")


@pytest.fixture(scope="module")
def gemm_isa(tmp_path_factory):
    return _isa(tmp_path_factory, "jf_gemm.hip")


@pytest.fixture(scope="module")
def attention_isa(tmp_path_factory):
    return _isa(tmp_path_factory, "jf_attention.hip")


def test_asm_mfma_results_are_not_touched_too_early(gemm_isa):
    lines = gemm_isa
    found = 0
    for i, line in enumerate(lines):
        code = line.split(";")[0]
        if "v_mfma" not in code or "0x3e22f983" not in code:
            continue
        found += 1
        dst = _regs(code.split(",")[0])
        ws, j = 0, i + 1
        while ws < WAIT_STATES and j < len(lines):
            t = lines[j].split(";")[0].strip()
            j += 1
            if not t or t.startswith(".") or t.endswith(":"):
                continue
            m = re.match(r"s_nop (\d+)", t)
            if m:
                ws += int(m.group(1)) + 1
                continue
            assert not t.startswith(("s_branch", "s_cbranch", "s_endpgm", "s_setpc")), \
                f"line {i + 1}: control flow {t!r} within {WAIT_STATES} wait states of an asm MFMA"
            assert not (_regs(t) & dst), f"line {i + 1}: {code.strip()!r} -> line {j}: {t!r} touches its destination"
            ws += 1
    assert found >= 16, "the scale-accumulate MFMAs were not found (did the kernel change?)"


def _functions(lines):
    """(number of the first line, name, instructions and labels) of every function."""
    start = None
    for i, line in enumerate(lines):
        m = re.match(r"(_Z\w+):", line)
        if m:
            start, name = i + 1, m.group(1)
        elif start is not None and line.startswith(".Lfunc_end"):
            yield start + 1, name, [t.split(";")[0].strip() for t in lines[start:i]]
            start = None


def _successors(body):
    label = {t[:-1]: i for i, t in enumerate(body) if t.endswith(":")}
    out = []
    for i, t in enumerate(body):
        assert not t.startswith(("s_setpc", "s_swappc", "s_call")), t
        m = re.match(r"s_(c?)branch\w*\s+(\S+)", t)
        out.append(([label[m.group(2)]] if m else []) + ([i + 1] if not t.startswith(("s_branch", "s_endpgm")) and i + 1 < len(body) else []))
    return out


def _barriers_behind_pending_table_writes(lines):
    """Number of the kernels whose blocks two waves share (they alone use v_mfma_i32_16x16x32_i8), and the lines of the barriers that
    one of a block's waves can reach while its writes to their common table of scale products are outstanding.  The factors of that
    table, and of no other, are negated: times -2^26, 0xcc800000.  A barrier does not wait for LDS writes, and those of different waves
    are not kept in order: without lgkmcnt(0) in front of it the other wave may read what was there before."""
    kernels, bad = 0, []
    for at, _, body in _functions(lines):
        if not any("v_mfma_i32_16x16x32_i8" in t for t in body):
            continue
        kernels += 1
        writes = []
        for i, t in enumerate(body):
            m = re.match(r"v_mul_f32\S* (v\d+), 0xcc800000, ", t)
            if m:
                assert re.match(r"ds_write_b32 v\d+, %s$" % m.group(1), body[i + 1]), f"line {at + i}: a factor of the table goes elsewhere"
                writes.append(i + 1)
        assert writes, f"line {at}: the table's writes were not found (did the kernel change?)"
        succ, seen, todo = _successors(body), set(), [i + 1 for i in writes]
        while todo:
            i = todo.pop()
            if i in seen or re.match(r"s_waitcnt .*lgkmcnt\(0\)", body[i]):
                continue
            seen.add(i)
            todo += succ[i]
        bad += [at + i for i in sorted(seen) if body[i].startswith("s_barrier")]
    return kernels, bad


def test_tables_of_two_waves_are_written_before_the_barrier(gemm_isa):
    kernels, bad = _barriers_behind_pending_table_writes(gemm_isa)
    assert kernels >= 14, "the kernels whose blocks two waves share were not found"
    assert not bad, f"barriers with LDS writes of the shared table outstanding: lines {bad}"


def _scalars_parked_in_main_loops(lines):
    """Number of the loops over two stages of two blocks per wave (16 products) in kernels of one tile size, and the lines of those that write
    scalar values to lanes of a vector register: four more vector instructions per K block cost 3 %."""
    loops, bad = 0, []
    for at, name, body in _functions(lines):
        if "igemm_nt_kernel" not in name:
            continue
        label = {t[:-1]: i for i, t in enumerate(body) if t.endswith(":")}
        for i, t in enumerate(body):
            m = re.match(r"s_c?branch\w*\s+(\S+)", t)
            if m and label[m.group(1)] < i:
                loop = body[label[m.group(1)]:i]
                if sum(t.startswith("v_mfma") for t in loop) == 16:
                    loops += 1
                    if any(t.startswith("v_writelane") for t in loop):
                        bad.append(at + i)
    return loops, bad


def test_main_loops_park_no_scalars(gemm_isa):
    loops, bad = _scalars_parked_in_main_loops(gemm_isa)
    assert loops >= 60, "the main loops were not found"
    assert not bad, f"scalar values written to lanes inside the loops that end at lines {bad}"


def _no_scratch_in_loops(lines):
    in_loop_depth = None
    for i, line in enumerate(lines):
        m = re.search(r"Loop Header: Depth=(\d+)|in Loop: Header=\S+ Depth=(\d+)", line)
        if re.match(r"^\.LBB\d+_\d+:", line):
            in_loop_depth = int(m.group(1) or m.group(2)) if m else None
        if in_loop_depth and re.match(r"\s*scratch_(load|store)", line):
            raise AssertionError(f"line {i + 1}: scratch access inside a loop: {line.strip()}")


def test_main_loops_do_not_spill(gemm_isa):
    """Scratch accesses are tolerated outside loops (a few values parked across the K loop in the binary16-scale
    kernels), never inside one."""
    _no_scratch_in_loops(gemm_isa)


def test_attention_tile_loops_do_not_spill(attention_isa):
    """A reload inside a tile loop would wait for the next tile's loads as well (values are parked across the loop of the dK/dV
    kernel with heads 64 wide)."""
    assert sum("v_mfma_f32_32x32x16_f16" in line for line in attention_isa) >= 200
    _no_scratch_in_loops(attention_isa)
