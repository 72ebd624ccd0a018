"""CPU: the waits of w4a16_gemm_reg_kernel and w4a16_gemm_lds_kernel as compiled
into libllmik_hip.so.

The kernels copy activations straight into LDS and wait once a stage, with a
bare count, for the wave's own copies of an earlier stage. The wait is right
for every order of the loads inside a stage exactly if it leaves at most as
many vector memory instructions pending as the last stage issued: then
everything older is complete. Read from the disassembly, whose order the
source alone does not fix."""
from __future__ import annotations

import re
import struct
import subprocess
from pathlib import Path

import pytest

PKG = Path(__file__).resolve().parents[1] / "llm-inference-kernels_amd"
LIB = PKG / "llmik_cuda" / "libllmik_hip.so"
OBJDUMP = Path("/opt/rocm/llvm/bin/llvm-objdump")
MAGIC = b"__CLANG_OFFLOAD_BUNDLE__"
KERNELS = {**{g: rb"_ZN5llmik21w4a16_gemm_reg_kernelILi%dE" % g for g in (32, 64, 128)},
           "lds": rb"_ZN5llmik21w4a16_gemm_lds_kernelE"}


def _device_objects(path):
    data, i = path.read_bytes(), -1
    while (i := data.find(MAGIC, i + 1)) >= 0:
        count, = struct.unpack_from("<Q", data, i + len(MAGIC))
        p = i + len(MAGIC) + 8
        for _ in range(count):
            off, size, n = struct.unpack_from("<QQQ", data, p)
            ident = data[p + 24:p + 24 + n]
            p += 24 + n
            if b"gfx950" in ident and size:
                yield data[i + off:i + off + size]


@pytest.fixture(scope="module")
def listings(tmp_path_factory):
    """Address, text and branch target of each instruction of the kernels."""
    if not LIB.exists() or not OBJDUMP.exists():
        pytest.skip("no built library or no llvm-objdump")
    out, d = {}, tmp_path_factory.mktemp("co")
    for k, obj in enumerate(_device_objects(LIB)):
        names = {g: m.group(0) for g, pat in KERNELS.items() if (m := re.search(pat + rb"\w+(?=\0)", obj))}
        if not names:
            continue
        f = d / f"{k}.o"
        f.write_bytes(obj)
        for g, name in names.items():
            text = subprocess.run([str(OBJDUMP), "-d", "--no-show-raw-insn", f"--disassemble-symbols={name.decode()}",
                                   str(f)], capture_output=True, text=True, check=True).stdout
            base = int(re.search(r"^([0-9a-f]+) <" + name.decode(), text, re.M).group(1), 16)
            ins = []   # (address, instruction, branch target)
            for ln in text.splitlines():
                if m := re.match(r"\t(.*?)\s*// ([0-9A-F]+):", ln):
                    to = re.search(r"\+0x([0-9a-f]+)>$", ln) if "branch" in m.group(1) else None
                    ins.append((int(m.group(2), 16), m.group(1), base + int(to.group(1), 16) if to else None))
            out[g] = ins
    assert len(out) == len(KERNELS)
    return out


# The prologue's first block: copies, words and scales of the first stage.
FIRST = {32: 4 + 2 + 2, 64: 4 + 2 + 1, 128: 4 + 2, "lds": 4 + 2 + 2}
# Unrolled stages and tail; the LDS-staged kernel waits once before its first.
STAGES = {32: 7, 64: 7, 128: 6, "lds": 4}


@pytest.mark.parametrize("group", list(KERNELS))
def test_waits_leave_at_most_the_last_stage_pending(listings, group):
    ins = listings[group]
    at = {a: i for i, (a, _, _) in enumerate(ins)}
    # Fewest vector memory instructions issued since the last barrier, over all
    # paths; before the first barrier, since the prologue's first block.
    since = {0: -FIRST[group]}
    todo = [0]
    waits = {}
    while todo:
        i = todo.pop()
        n = since[i]
        _, s, to = ins[i]
        if re.match(r"(buffer|global|flat|scratch)_", s):
            n += 1
        if s.startswith("s_barrier"):
            near = [m for k in range(max(i - 4, 0), i) if (m := re.search(r"vmcnt\((\d+)\)", ins[k][1]))]
            waits[i] = (int(near[-1].group(1)) if near else 0, n)   # 0: the split hand-off's
            n = 0
        nxt = [] if s.startswith(("s_endpgm", "s_branch")) else [i + 1]
        if to is not None:
            nxt.append(at[to])
        for k in nxt:
            if k < len(ins) and n < since.get(k, 1 << 30):
                since[k] = n
                todo.append(k)
    stages = [w for w in waits.values() if w[0] > 0]
    assert len(stages) == STAGES[group]
    assert all(left <= issued for left, issued in stages), stages
