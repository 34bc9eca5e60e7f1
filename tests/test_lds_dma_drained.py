"""No kernel of the built library may end with a load to LDS in flight: on every
path of a kernel's control flow from a `buffer_load ... lds` to s_endpgm there is
an s_waitcnt vmcnt(0).  Read off the gfx950 code of libacfun_amd.so.  k_gemm32 is
left out: its wait is chosen by the number of chunks still to come, and the
paths that skip vmcnt(0) after the last chunk cannot be taken.  CPU only."""
import os
import re
import subprocess

import pytest

from acfun_amd import capi

OBJDUMP = "/opt/rocm/llvm/bin/llvm-objdump"
LINE = re.compile(r"^\s+(\S.*?)\s*// ([0-9A-F]+): .*?(?:<(\S+?)(?:\+0x([0-9a-f]+))?>)?$")
HEAD = re.compile(r"^([0-9a-f]+) <(\S+)>:$")


def _kernels(tmp_path):
    """(name, [(address, instruction, branch target or None)]) of every kernel."""
    lib = tmp_path / "lib.so"
    os.symlink(capi.LIB_PATH, lib)
    subprocess.run([OBJDUMP, "--offloading", str(lib)], check=True, capture_output=True, cwd=tmp_path)
    for f in sorted(tmp_path.glob("lib.so.*gfx950")):
        text = subprocess.run([OBJDUMP, "-d", str(f)], check=True, capture_output=True, text=True).stdout
        name, base, code = None, 0, []
        for line in text.split("\n"):
            h = HEAD.match(line)
            if h:
                if name:
                    yield name, code
                name, base, code = h.group(2), int(h.group(1), 16), []
                continue
            m = LINE.match(line)
            if m and name:
                target = None
                if m.group(1).startswith(("s_branch", "s_cbranch")):
                    assert m.group(3) == name, line
                    target = base + int(m.group(4) or "0", 16)
                code.append((int(m.group(2), 16), m.group(1), target))
        if name:
            yield name, code


def _ends_in_flight(code):
    at = {a: i for i, (a, _, _) in enumerate(code)}

    def after(i):
        _, ins, target = code[i]
        if ins.startswith("s_branch"):
            return [at[target]]
        return [i + 1] + ([at[target]] if target is not None else [])

    todo = [j for i, (_, ins, _) in enumerate(code)
            if ins.startswith("buffer_load") and ins.endswith(" lds") for j in after(i)]
    seen = set()
    while todo:
        i = todo.pop()
        if i in seen:
            continue
        seen.add(i)
        ins = code[i][1]
        if ins.startswith("s_endpgm"):
            return True
        if not (ins.startswith("s_waitcnt") and "vmcnt(0)" in ins):
            todo += after(i)
    return False


def test_no_kernel_ends_with_lds_loads_in_flight(tmp_path):
    if not os.path.exists(OBJDUMP):
        pytest.skip("no llvm-objdump")
    left, with_dma = [], 0
    for name, code in _kernels(tmp_path):
        if any(ins.startswith("buffer_load") and ins.endswith(" lds") for _, ins, _ in code):
            with_dma += 1
            if re.search(r"\d+k_gemm32I", name) is None and _ends_in_flight(code):
                left.append(name)
    assert with_dma >= 50        # the disassembly was understood
    assert not left, left
