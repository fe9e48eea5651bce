"""Matrix results in the built device code are touched only after their wait states, on every path.

The hardware does not hold back an instruction that reads or overwrites the result of a matrix
instruction still in the pipe; the compiler places wait states, and within a block it always places
enough.  Where several paths of different length lead to the first touch it has counted one or two too
few (the model and Gram kernels), so this walks every path of the disassembly of the library's kernels
from each matrix instruction to the first touch of its result."""
import glob
import os
import re
import struct
import subprocess

import pytest

from conftest import ROOT

OBJDUMP = "/opt/rocm/llvm/bin/llvm-objdump"
# wait states before a vector instruction (or a store) may read the result, as the compiler keeps them
# within a block, and before one may overwrite it
READ = {"v_mfma_f32_16x16x32_bf16": 8, "v_mfma_f32_16x16x4_f32": 10, "v_mfma_f64_16x16x4_f64": 18}
WRITE = {"v_mfma_f32_16x16x32_bf16": 8, "v_mfma_f32_16x16x4_f32": 10, "v_mfma_f64_16x16x4_f64": 0}
LONG = 64  # clocks of a sleep, and at least of a wait for a load issued since


def device_code(path):
    """the gfx950 code objects in an object file"""
    data, at = open(path, "rb").read(), 0
    while (at := data.find(b"__CLANG_OFFLOAD_BUNDLE__", at)) >= 0:
        p = at + 32
        for _ in range(struct.unpack_from("<Q", data, at + 24)[0]):
            offset, size, length = struct.unpack_from("<QQQ", data, p)
            if b"gfx950" in data[p + 24:p + 24 + length] and size:
                yield data[at + offset:at + offset + size]
            p += 24 + length
        at += 24


def registers(operand):
    out = set()
    for kind, lo, hi, one in re.findall(r"\b([av])(?:\[(\d+):(\d+)\]|(\d+)\b)", operand):
        out.update((kind, i) for i in (range(int(lo), int(hi) + 1) if lo else [int(one)]))
    return frozenset(out)


def functions(code):
    """name -> list of (mnemonic, operands' registers, first operand, branch target's index)"""
    text = subprocess.run([OBJDUMP, "-d", code], capture_output=True, text=True, check=True).stdout
    for part in re.split(r"\n(?=[0-9a-f]+ <)", text):
        head = re.match(r"([0-9a-f]+) <(\w+)>:", part)
        if not head or "v_mfma" not in part:
            continue
        base, lines, index = int(head.group(1), 16), [], {}
        for line in part.splitlines()[1:]:
            m = re.match(r"\t(\w+)(.*?)// ([0-9A-F]+): [0-9A-F ]+(?:<\w+\+0x([0-9a-f]+)>)?", line)
            if m:
                index[int(m.group(3), 16)] = len(lines)
                lines.append((m.group(1), m.group(2).strip(), m.group(4)))
        out = []
        for name, ops, target in lines:
            ops = re.split(r",\s*(?![^\[]*\])", ops)
            to = index.get(base + int(target, 16)) if target else None
            if name == "s_branch" and to is None:
                to = index.get(base)  # (a branch to the function's start has no offset)
            out.append((name, [registers(o) for o in ops], ops[0], to))
        yield head.group(2), out


def too_early(ins):
    bad = []
    for i, (name, regs, _, _) in enumerate(ins):
        if not name.startswith(("v_mfma", "v_smfma")):
            continue
        need = max(READ[name], WRITE[name])
        stack, seen = [(i + 1, 0, regs[0], False, False)], {}
        while stack:
            j, states, live, lds, mem = stack.pop()
            if states >= need or j >= len(ins) or not live or seen.get((j, live, lds, mem), need) <= states:
                continue
            seen[(j, live, lds, mem)] = states
            n, r, first, to = ins[j]
            if n in ("s_endpgm", "s_setpc_b64"):
                continue
            if n == "s_nop":
                stack.append((j + 1, states + int(first, 0) + 1, live, lds, mem))
                continue
            if n == "s_sleep":
                stack.append((j + 1, states + LONG * int(first, 0), live, lds, mem))
                continue
            if n == "s_waitcnt":
                done = lds and "lgkmcnt(0)" in first or mem and "vmcnt(0)" in first
                stack.append((j + 1, states + (LONG if done else 1), live, lds, mem))
                continue
            if to is not None:
                stack.append((to, states + 1, live, lds, mem))
                if n == "s_branch":
                    continue
            read, write = frozenset().union(*r[1:]) if len(r) > 1 else frozenset(), r[0]
            if n.startswith(("ds_write", "ds_store", "global_store", "buffer_store", "flat_store")):
                read, write = read | write, frozenset()
            if n.startswith("v_mfma"):  # (a result as the next addend has its own rule, which is forwarding)
                read = r[1] | r[2]
                live, write = live - write if len(r) > 3 and r[3] & live else live, frozenset()
            if read & live and states < READ[name] or write & live and states < WRITE[name]:
                bad.append((name, i, n, j, states))
            live = live - read - write
            stack.append((j + 1, states + 1, live, lds or n.startswith("ds_read"), mem or n.startswith("global_load")))
    return bad


def test_results_wait(tmp_path):
    objects = sorted(glob.glob(os.path.join(ROOT, "first-project_amd", "_build", "*.o")))
    if not objects or not os.path.exists(OBJDUMP):
        pytest.skip("the library's objects are not built")
    count, bad = 0, []
    for path in objects:
        for k, code in enumerate(device_code(path)):
            file = tmp_path / f"{os.path.basename(path)}.{k}"
            file.write_bytes(code)
            for name, ins in functions(str(file)):
                count += 1
                bad += [(name, *b) for b in too_early(ins)]
    assert count > 0
    assert not bad, bad[:8]


def test_the_walk_finds_an_early_touch():
    mfma = ("v_mfma_f32_16x16x4_f32", [registers(o) for o in ("v[0:3]", "v8", "v9", "v[0:3]")], "v[0:3]", None)
    other = ("v_mov_b32_e32", [registers("v20"), registers("v21")], "v20", None)
    touch = ("v_mov_b32_e32", [registers("v20"), registers("v2")], "v20", None)
    nop = lambda n: ("s_nop", [frozenset()], str(n), None)
    end = ("s_endpgm", [frozenset()], "", None)
    assert too_early([mfma, nop(8), touch, end]) and not too_early([mfma, nop(9), touch, end])
    assert not too_early([mfma] + 10 * [other] + [touch, end])
    # the path around the block with the wait
    branch = ("s_cbranch_vccnz", [frozenset()], "", 4)
    assert too_early([mfma, nop(7), branch, nop(9), touch, end])
