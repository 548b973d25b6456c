"""What the compiler cannot see in the matrix kernels' hand-written loads, checked in the code that it made of them (the device code of the
in-tree library, disassembled; no GPU)."""
import glob
import os
import re
import shutil
import subprocess

import pytest

from gpreempt_amd import capi as gp

OBJDUMP = "/opt/rocm/llvm/bin/llvm-objdump"
READELF = "/opt/rocm/llvm/bin/llvm-readelf"
pytestmark = pytest.mark.skipif(not os.path.exists(OBJDUMP), reason="no disassembler")
WORD = re.compile(r"^\s+([a-z]\S*)\s*(.*?)\s*// ([0-9A-F]+):(.*)$")


@pytest.fixture(scope="module")
def kernels(tmp_path_factory):
    """{name: [(address, mnemonic, operands, branch target or None)]} of every kernel that loads to LDS"""
    work = tmp_path_factory.mktemp("isa")
    lib = shutil.copy(gp.LIB_PATH, work)
    subprocess.run([OBJDUMP, "--offloading", os.path.basename(lib)], cwd=work, check=True, capture_output=True)
    found = {}
    for part in glob.glob(os.path.join(work, "*gfx950*")):
        name, code = None, []
        for line in subprocess.run([OBJDUMP, "-d", part], check=True, capture_output=True, text=True).stdout.splitlines():
            if line.endswith(">:") and not line.startswith(" "):
                name, code = line[line.index("<") + 1:-2], []
                found[os.path.basename(part) + name] = code
                continue
            m = WORD.match(line)
            if m and name:
                to = re.search(r"\+0x([0-9a-f]+)>$", m.group(4)) if m.group(1).startswith(("s_branch", "s_cbranch")) else None
                code.append((int(m.group(3), 16), m.group(1), m.group(2), int(to.group(1), 16) if to else None))
    found = {k: v for k, v in found.items() if any((op.startswith("buffer_load") and args.endswith(" lds")) or op.startswith("global_load_lds") for _, op, args, _ in v)}
    assert len(found) > 400
    return found


def scalars(operand):
    m = re.match(r"^s(?:\[(\d+):(\d+)\]|(\d+))$", operand)
    return range(int(m.group(1) or m.group(3)), int(m.group(2) or m.group(3)) + 1) if m else ()


def test_a_scalar_written_by_a_vector_instruction_is_read_by_a_load_five_wait_states_later(kernels):
    """... or later: the hardware does not wait, and the compiler does not look into the loads, which are inline assembly"""
    bad = []
    for name, code in kernels.items():
        at, written = 0, {}  # wait states so far; scalar -> when it was last written
        for _, op, args, _ in code:
            parts = [p for p in re.split(r"[,\s]+", args) if p]
            if op.startswith(("buffer_", "global_", "scratch_")):
                bad += [(name, op, args) for p in parts for s in scalars(p) if at - written.get(s, -9) - 1 < 5]
            elif op.startswith("v_") and parts:
                for s in scalars(parts[0]):
                    written[s] = at
            at += int(parts[0], 0) + 1 if op == "s_nop" else 1
    assert not bad, (len(bad), bad[:4])


def test_no_barrier_is_reached_with_lds_reads_outstanding(kernels):
    """behind a stage's barrier the buffer that they read is loaded into again, which the compiler does not know"""
    bad = []
    for name, code in kernels.items():
        index = {a: i for i, (a, *_) in enumerate(code)}
        most, work = [-1] * len(code), [(0, 0)]  # reads and writes outstanding in front of an instruction, on the worst way there
        while work:
            i, n = work.pop()
            while i < len(code) and n > most[i]:
                most[i] = n
                a, op, args, to = code[i]
                if op.startswith("ds_"):
                    n = min(n + 1, 15)
                elif op == "s_waitcnt" and "lgkmcnt" in args:
                    n = min(n, int(re.search(r"lgkmcnt\((\d+)\)", args).group(1)))
                elif op == "s_barrier" and n:
                    bad.append((name, hex(a), n))
                elif op == "s_endpgm":
                    break
                if to is not None:
                    j = index[code[0][0] + to]
                    if op == "s_branch":
                        i = j
                        continue
                    work.append((j, n))
                i += 1
    assert not bad, (len(bad), bad[:4])


def loops_of(code, mfmas):
    """the innermost ways back over that many matrix instructions"""
    index = {a: i for i, (a, *_) in enumerate(code)}
    before = [0]
    for _, op, _, _ in code:
        before.append(before[-1] + op.startswith("v_mfma"))
    back = [(index[code[0][0] + to], i) for i, (_, _, _, to) in enumerate(code) if to is not None and index[code[0][0] + to] <= i]
    back = [(j, i) for j, i in back if before[i + 1] - before[j] == mfmas]
    return [code[j:i + 1] for j, i in back if not any((a, b) != (j, i) and j <= a and b <= i for a, b in back)]


def test_the_loop_of_256_tiles_in_phases_waits_for_nothing_it_need_not(kernels):
    """Operands are asked for two K-steps ahead: no wait for everything that is on its way stands in the loop, and no register comes back from
    scratch memory, behind which the compiler puts one"""
    loops = {k: loops_of(v, 32) for k, v in kernels.items() if re.search(r"PipeKernelIDF16.Li256ELi256ELi2ELi0ELb0ELb[01]ELi8ELb0ELb1E", k)}
    assert len(loops) == 10 and all(loops.values())
    for name, loop in ((k, l) for k, ls in loops.items() for l in ls):
        assert not [op for _, op, _, _ in loop if op.startswith("scratch_")], name
        assert [a for _, op, a, _ in loop if op == "s_waitcnt" and "vmcnt" in a] == ["vmcnt(8)", "vmcnt(6)"], name


@pytest.fixture(scope="module")
def spilled(tmp_path_factory):
    """{name: vector registers that the compiler spilled} of the kernels that run one tile of 256 x 256: the forms without claims (1), with fixed claims (2), and with looks (3)"""
    work = tmp_path_factory.mktemp("notes")
    lib = shutil.copy(gp.LIB_PATH, work)
    subprocess.run([OBJDUMP, "--offloading", os.path.basename(lib)], cwd=work, check=True, capture_output=True)
    found = {}
    for part in glob.glob(os.path.join(work, "*gfx950*")):
        notes = subprocess.run([READELF, "--notes", part], check=True, capture_output=True, text=True).stdout
        for kernel in re.split(r"\n\s+- \.agpr_count:", notes)[1:]:
            name = re.search(r"\.name:\s+(\S+)", kernel).group(1)
            form = re.search(r"mat_kernelINS_10PipeKernelI\S+?Li256ELi256ELi2E\S*Li([123])E", name)
            if form:
                found[name] = int(re.search(r"\.vgpr_spill_count:\s+(\d+)", kernel).group(1))
    assert len(found) == 15
    return found


def test_tiles_of_256_keep_to_their_registers(spilled):
    """... all but the addresses that the forms with looks park across a main loop that fetches stage by stage"""
    bad = {k: n for k, n in spilled.items() if n > (9 if "ELb0EEELi3E" in k else 0)}
    assert not bad, bad
