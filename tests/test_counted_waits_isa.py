"""Static checks of the built library's kernels that wait for their loads by counts (no GPU): ``s_waitcnt vmcnt(n)`` with
n > 0 rests on loads that return in the order of their requests, and on n being counted from the loads that the compiler
really emits."""
import os
import re
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
LIB = os.path.join(ROOT, "intel-extension-for-pytorch_amd", "lib", "libwoq_hip.so")
OBJDUMP = "/opt/rocm/llvm/bin/llvm-objdump"
pytestmark = pytest.mark.skipif(not os.path.exists(LIB) or not os.path.exists(OBJDUMP), reason="needs the built library and llvm-objdump")


@pytest.fixture(scope="module")
def kernels(tmp_path_factory):
    """{mangled name: [(address, instruction)]} of the prefill and decode kernels."""
    d = tmp_path_factory.mktemp("isa")
    shutil.copy(LIB, d / "lib.so")
    subprocess.run([OBJDUMP, "--offloading", "lib.so"], cwd=d, check=True, capture_output=True)
    out = {}
    for name in sorted(os.listdir(d)):
        if not name.endswith("gfx950"):
            continue
        with open(d / name, "rb") as f:
            code = f.read()
        if b"woq_gemm_w4_kernel" not in code and b"woq_decode_dq_kernel" not in code and b"woq_decode_kernel" not in code and b"woq_gemm_dense_kernel" not in code:
            continue
        body = None
        for line in subprocess.run([OBJDUMP, "-d", "--no-show-raw-insn", name], cwd=d, check=True, capture_output=True, text=True).stdout.split("\n"):
            m = re.match(r"^[0-9a-f]+ <(\w+)>:", line)
            if m:
                body = out.setdefault(m.group(1), [])
            else:
                m = re.match(r"^\t(.*?)\s*// ([0-9A-F]+):", line)
                if m:
                    body.append((int(m.group(2), 16), m.group(1)))
    return out


def test_no_flat_accesses(kernels):
    """After a FLAT load (generic address) only a wait for zero is defined: every address must be known to be global."""
    seen = 0
    for name, body in kernels.items():
        if re.search("woq_gemm_w4_kernel|woq_decode_dq_kernel|woq_decode_kernel|woq_decode_m1_kernel", name):
            seen += 1
            assert not [t for _, t in body if t.startswith("flat_")], name
    assert seen >= 100, seen


def test_prefill_waits_count_no_more_loads_than_a_step_has(kernels):
    """The prefill kernel's K loop reads a step's packed tiles from LDS after vmcnt(n), n the loads of one whole step: with
    fewer loads in the compiled loop than n, the wait would let the tiles' own loads be outstanding still."""
    seen = 0
    for name, body in kernels.items():
        if "woq_gemm_w4_kernel" not in name:
            continue
        at = {a: i for i, (a, _) in enumerate(body)}
        loops = []
        for i, (a, t) in enumerate(body):
            m = re.match(r"s_c?branch\S* (\d+)", t)
            if m:
                off = int(m.group(1))
                first = at.get(a + 4 + 4 * (off - 65536 if off >= 32768 else off))
                if first is not None and first < i:
                    loop = [x for _, x in body[first:i]]
                    loops.append((sum(x.startswith("v_mfma") for x in loop), -len(loop), loop))
        mfmas, _, loop = max(loops)
        loads = sum(x.startswith("global_load") for x in loop)
        waits = [int(n) for x in loop for n in re.findall(r"^s_waitcnt.*vmcnt\((\d+)\)", x)]
        assert mfmas >= 32 and waits, name
        assert max(waits) <= loads, (name, waits, loads)
        seen += 1
    assert seen >= 40, seen


def _loops(body):
    """Instruction ranges of the backward branches of a kernel that hold an MFMA and no smaller such range."""
    at = {a: i for i, (a, _) in enumerate(body)}
    ranges = []
    for i, (a, t) in enumerate(body):
        m = re.match(r"s_c?branch\S* (\d+)", t)
        if m:
            off = int(m.group(1))
            first = at.get(a + 4 + 4 * (off - 65536 if off >= 32768 else off))
            if first is not None and first < i and any(x.startswith("v_mfma") for _, x in body[first:i]):
                ranges.append((first, i))
    return [[x for _, x in body[f:l + 1]] for f, l in ranges if not any(f <= f2 and l2 <= l and (f, l) != (f2, l2) for f2, l2 in ranges)]


def test_every_prefill_loop_has_its_reads_back_at_the_barrier(kernels):
    """Behind the barrier of a K step the other waves refill the activation buffer that the step has read, so no read of it may
    be outstanding there.  Outstanding may be the packed tiles that a wave alone reads (8-bit weights: two) in the blocks of
    the last sub-step before the one with the barrier, number NTW - 2 (16 row tiles: NTW - 1) at most.  All loops of a kernel:
    the grouped ones have a body each for 32, 64 and 128 rows."""
    seen = 0
    for name, body in kernels.items():
        shape = re.search(r"woq_gemm_w4_kernel.*G4ShapeILi(\d+)ELi(\d+)ELi(\d+)EEELi(\d)E", name)
        if not shape:
            continue
        mt, ntw, tps = int(shape.group(1)), int(shape.group(2)), int(shape.group(4)) // 4
        for loop in _loops(body):
            reads = []  # outstanding, oldest first; NF4's table reads are of eight bytes and of a table that stays
            for _ in range(2):  # (the second time with those of the step before)
                for t in loop:
                    if t.startswith(("ds_read", "ds_write")):
                        reads.append(t.startswith("ds_read_b128"))
                    m = re.match(r"s_waitcnt\b.*lgkmcnt\((\d+)\)", t)
                    if m:
                        reads = reads[max(0, len(reads) - int(m.group(1))):]
                    if t.startswith("s_barrier"):
                        assert sum(reads) <= (ntw - (1 if mt >= 16 else 2)) * tps, (name, sum(reads))
                        seen += 1
            loads = sum(x.startswith("global_load") for x in loop)
            waits = [int(n) for x in loop for n in re.findall(r"^s_waitcnt.*vmcnt\((\d+)\)", x)]
            assert waits and max(waits) <= loads, (name, waits, loads)
    assert seen >= 100, seen


def test_every_loop_of_the_dense_kernel_has_its_reads_back_at_the_barrier(kernels):
    """As above; this kernel reads nothing but activations from LDS."""
    seen = 0
    for name, body in kernels.items():
        if "woq_gemm_dense_kernel" not in name:
            continue
        for loop in _loops(body):
            reads = 0
            for t in loop + loop:
                reads += t.startswith("ds_read")
                m = re.match(r"s_waitcnt\b.*lgkmcnt\((\d+)\)", t)
                if m:
                    reads = min(reads, int(m.group(1)))
                if t.startswith("s_barrier"):
                    assert reads == 0, (name, reads)
                    seen += 1
    assert seen >= 6, seen
