"""Rows that load straight into LDS land in buffers that were read a stage
before.  In the built gfx950 code of the kernels that do this, no path leads
from an LDS read to such a load, or to a barrier behind which another wave
issues one, without a wait for the reads (lgkmcnt(0)): that a read has
returned otherwise follows only from where the compiler puts its uses."""
import os
import re

import pytest

from fingering_dynamics_amd import build
from test_build_flags import _disassemble

TARGET = re.compile(r"<(\S+?)(?:\+0x([0-9a-f]+))?>\s*$")


def _functions(asm):
    """{name: [(address, mnemonic, operands, branch target or None)]}"""
    out, name = {}, None
    for line in asm.splitlines():
        m = re.match(r"^([0-9a-f]+) <(.*)>:$", line)
        if m:
            name, base = m.group(2), int(m.group(1), 16)
            out[name] = []
            continue
        m = re.match(r"^\s+(\S+)\s*(.*?)\s*// ([0-9A-F]+):(.*)$", line)
        if name is None or not m:
            continue
        op, args, addr, rest = m.group(1), m.group(2), int(m.group(3), 16), m.group(4)
        target = None
        if op.startswith(("s_cbranch", "s_branch")):
            t = TARGET.search(rest)
            assert t and t.group(1) == name, line
            target = base + int(t.group(2) or "0", 16)
        out[name].append((addr, op, args, target))
    return out


def unwaited(code):
    """Instructions of a function that load into LDS, or are a barrier, with
    an LDS read of the same wave possibly outstanding."""
    at = {addr: i for i, (addr, _, _, _) in enumerate(code)}
    pending = [None] * len(code)           # LDS reads outstanding before the instruction; None: not reached
    todo = [(0, False)]
    while todo:
        i, p = todo.pop()
        while i < len(code) and not (pending[i] is not None and (pending[i] or not p)):
            pending[i] = p
            _, op, args, target = code[i]
            if op.startswith("ds_read"):
                p = True
            elif op == "s_waitcnt" and "lgkmcnt(0)" in args:
                p = False
            if target is not None:
                todo.append((at[target], p))
            if op in ("s_branch", "s_endpgm"):
                break
            i += 1
    return [code[i] for i in range(len(code)) if pending[i] and
            (code[i][1] == "s_barrier" or (code[i][1].startswith("buffer_load") and code[i][2].endswith(" lds")))]


def test_the_check_finds_a_missing_wait():
    read, load, wait = (0, "ds_read_b32", "v0, v1", None), (4, "buffer_load_dwordx4", "v1, s[0:3], 0 offen lds", None), \
        (8, "s_waitcnt", "lgkmcnt(0)", None)
    end = (16, "s_endpgm", "", None)
    assert unwaited([read, load, end]) == [load]
    assert unwaited([read, wait, load, end]) == []
    back = (12, "s_cbranch_scc0", "65532", 4)         # around a loop: the load comes before the read
    loop = [(0, "s_nop", "0", None), load, (8, "ds_read_b32", "v0, v1", None), back, end]
    assert unwaited(loop) == [load]


@pytest.mark.parametrize("name,kernel,count", [("libfdsurr.so", "conv_wgrad", 12), ("libfdlbm.so", "fused", 10)])
def test_lds_reads_have_returned_before_their_rows_are_overwritten(tmp_path, name, kernel, count):
    code = {k: v for k, v in _functions(_disassemble(os.path.join(build.LIBDIR, name), tmp_path)).items()
            if kernel in k and any(" lds" in a for _, o, a, _ in v if o.startswith("buffer_load"))}
    assert len(code) == count, sorted(code)
    for k, v in code.items():
        assert not unwaited(v), (k, unwaited(v)[:4])
