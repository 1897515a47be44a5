"""The per-replica boundary kernel branches on flags of the replica's state that
its thread 0 rewrites for the next step, so every wave has to hold them before
any wave may write one.  Shown on the compiled gfx950 code, over every path from
the kernel's entry: no store to global memory ahead of the first barrier, and no
wave that leaves behind the first barrier decides so by what it reads from the
copy in LDS there (thread 0 may be rewriting it)."""
import os
import re
import shutil
import subprocess

import pytest

from conftest import ROOT

OBJDUMP = os.path.join(os.environ.get("ROCM_PATH", "/opt/rocm"), "llvm", "bin", "llvm-objdump")
STORE = re.compile(r"^(global|flat|buffer|scratch)_(store|atomic)")


def _kernels(lib, tmp, pattern):
    """{symbol: [(address, mnemonic, branch target or None)]} of the kernels whose
    symbol holds `pattern`."""
    so = shutil.copy(lib, tmp)
    subprocess.run([OBJDUMP, "--offloading", so], cwd=tmp, check=True, stdout=subprocess.DEVNULL)
    out = {}
    for f in sorted(os.listdir(tmp)):
        if "amdgcn" not in f:
            continue
        text = subprocess.run([OBJDUMP, "-d", "--no-show-raw-insn", os.path.join(tmp, f)], check=True,
                              stdout=subprocess.PIPE, text=True).stdout
        code = None
        for line in text.splitlines():
            head = re.match(r"^([0-9a-f]+) <(.*)>:$", line)
            if head:
                code = out.setdefault(head[2], []) if pattern in head[2] else None
                base = int(head[1], 16)
                continue
            ins = re.match(r"^\s+(\S+).*// ([0-9A-F]+):", line) if code is not None else None
            if ins:
                to = re.search(r"<[^>]*?(?:\+0x([0-9a-f]+))?>$", line) if "branch" in ins[1] else None
                code.append((int(ins[2], 16), ins[1], base + int(to[1] or "0", 16) if to else None))
    return out


def _faults(code):
    """Walks every path up to its second barrier, as (instruction, barriers
    passed, LDS read since); returns the rules it finds broken."""
    at = {a: k for k, (a, _, _) in enumerate(code)}
    seen, todo, bad = set(), [(0, 0, False)], set()
    while todo:
        s = todo.pop()
        if s in seen or s[0] >= len(code):
            continue
        seen.add(s)
        k, bars, read = s
        _, op, to = code[k]
        if bars == 0 and STORE.match(op):
            bad.add("store ahead of the first barrier")
        if op == "s_barrier":
            if bars == 1:
                continue
            bars, read = 1, False
        elif op.startswith("ds_read") and bars == 1:
            read = True
        elif op == "s_endpgm":
            if read:
                bad.add("leaves by a flag read from LDS behind the first barrier")
            continue
        if to is not None:
            todo.append((at[to], bars, read))
        if op != "s_branch":
            todo.append((k + 1, bars, read))
    return bad


def test_flags_are_held_before_any_is_written(fmd, tmp_path):
    if not os.path.exists(OBJDUMP):
        pytest.skip("no llvm-objdump")
    kernels = _kernels(os.path.join(ROOT, "fastmd_amd", "libfastmd.so"), str(tmp_path), "10k_boundary")
    assert len([k for k in kernels if not k.endswith(".kd")]) == 2, list(kernels)
    for name, code in kernels.items():
        assert any(op == "s_barrier" for _, op, _ in code), name
        assert not _faults(code), (name, _faults(code))
