"""No LDS write is in flight when a wave arrives at a workgroup barrier, in the code that the compiler makes of the
kernels (CPU: hipcc's gfx950 assembly of this repository's sources).

A barrier does not wait for a wave's LDS writes: one that was only issued may land after another wave has read the same
place behind the barrier, now and then and without an error, so a test of results rarely sees it.  Where the kernels
use a barrier without __syncthreads' fence (dma_tile.h), the wait is theirs to write; this follows the instructions of
every kernel from its LDS writes to the barriers that they reach."""
import os
import re
import shutil
import subprocess

import pytest

from scratchtape_amd import build

READS = ("ds_read", "ds_bpermute", "ds_permute", "ds_swizzle", "ds_nop")
HIPCC = shutil.which(build.HIPCC) or shutil.which("hipcc")


def kernels(asm):
    """name -> instruction lines (labels included) of each function in an AMD assembly file."""
    out, name = {}, None
    for line in asm.splitlines():
        line = line.split(";")[0].split("//")[0].strip()
        m = re.match(r"^(_Z\w+):$", line)
        if m:
            name = m.group(1)
            out[name] = []
        elif name and (re.match(r"^\.L\w+:$", line) or re.match(r"^[a-z]\w+(\s|$)", line)):
            out[name].append(line)
            if line.startswith("s_endpgm") and ".Lfunc_end" in line:
                name = None
        elif line.startswith(".Lfunc_end"):
            name = None
    return out


def barriers_with_writes_in_flight(lines):
    """Indexes of the s_barrier instructions that an LDS write reaches without an lgkmcnt(0) in between, over all paths
    (forward data flow of one bit: some LDS write may be in flight)."""
    label = {l[:-1]: i for i, l in enumerate(lines) if l.endswith(":")}
    flying = [None] * (len(lines) + 1)  # on entry to the instruction
    todo, bad = [(0, False)], set()
    while todo:
        i, f = todo.pop()
        while i < len(lines):
            if flying[i] is not None and (flying[i] or not f):
                break
            flying[i] = f
            op, _, rest = lines[i].partition(" ")
            if op.startswith("ds_") and not op.startswith(READS):
                f = True
            elif op == "s_waitcnt" and ("lgkmcnt(0)" in rest or rest.strip() == "0"):
                f = False
            elif op == "s_barrier" and f:
                bad.add(i)
            elif op in ("s_branch", "s_endpgm"):
                if op == "s_branch":
                    todo.append((label[rest.strip()], f))
                break
            elif op.startswith("s_cbranch"):
                todo.append((label[rest.strip()], f))
            i += 1
    return sorted(bad)


def test_the_flow_sees_a_missing_wait():
    code = """
_Zk:
\ts_cbranch_scc0 .LBB0_2
\tds_write_b32 v0, v1
.LBB0_2:
\ts_barrier
\tds_read_b32 v2, v0
\ts_waitcnt lgkmcnt(0)
\ts_barrier
\ts_branch .LBB0_2
.Lfunc_end0:
"""
    (lines,) = kernels(code).values()
    assert barriers_with_writes_in_flight(lines) == [lines.index("s_barrier")]
    wait = "s_waitcnt vmcnt(1) lgkmcnt(0)"
    fixed = [x for line in lines for x in ([line, wait] if line.startswith("ds_w") else [line])]
    assert barriers_with_writes_in_flight(fixed) == []


@pytest.mark.skipif(HIPCC is None, reason="needs hipcc")
@pytest.mark.parametrize("src", ["gemm_dma.hip", "gemm_group.hip"])  # the sources with barriers of their own
def test_no_lds_write_is_in_flight_at_a_barrier(src, tmp_path):
    out = str(tmp_path / "k.s")
    flags = [f for f in build.CFLAGS if f != "-fPIC"]
    subprocess.run([HIPCC, *flags, "-S", "--cuda-device-only", os.path.join(build.CSRC, src), "-o", out], check=True,
                   capture_output=True)
    found = {n: l for n, l in kernels(open(out).read()).items() if "s_barrier" in l}
    assert len(found) >= 4, list(found)
    bad = {n: b for n, l in found.items() if (b := barriers_with_writes_in_flight(l))}
    assert not bad, f"{len(bad)} of {len(found)} kernels: {bad}"
