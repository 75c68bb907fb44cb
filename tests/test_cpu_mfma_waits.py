"""Every MFMA of the built library has its wait before the next use of its result's registers.

The matrix cores write a result some issue slots after the instruction, and the hardware does not
hold back an instruction that reads (or overwrites) those registers earlier: the compiler puts
waits there. It has left some out where a result's use was moved behind a uniform branch, so
this walks the disassembly of the library's own code objects: from each MFMA along every path,
counting issue slots until the result is complete."""
import os
import re
import shutil
import struct
import subprocess

import pytest

from w4a8_fp8_wmma import _lib

OBJDUMP = shutil.which("llvm-objdump") or "/opt/rocm/llvm/bin/llvm-objdump"
MAGIC = b"__CLANG_OFFLOAD_BUNDLE__"

# Issue slots from an MFMA to the first other use of its result, as the compiler counts them for
# gfx950: the instruction's passes (8 with an 8-bit operand, 4 for 16-bit ones) + WAIT.
WAIT = 4
PASSES = {"v_mfma_f32_16x16x128_f8f6f4": 8, "v_mfma_scale_f32_16x16x128_f8f6f4": 8,
          "v_mfma_f32_16x16x32_bf16": 4}


def code_objects(path):
    """The gfx950 code objects bundled in a host library."""
    blob = open(path, "rb").read()
    at = blob.find(MAGIC)
    while at >= 0:
        (n,) = struct.unpack_from("<Q", blob, at + len(MAGIC))
        p = at + len(MAGIC) + 8
        for _ in range(n):
            off, size, idlen = struct.unpack_from("<QQQ", blob, p)
            name = blob[p + 24:p + 24 + idlen].decode()
            p += 24 + idlen
            if "gfx950" in name and size:
                yield blob[at + off:at + off + size]
        at = blob.find(MAGIC, at + 1)


REG = re.compile(r"\b([av])(?:\[(\d+):(\d+)\]|(\d+)\b)")


def registers(text):
    out = set()
    for kind, lo, hi, one in REG.findall(text):
        out.update((kind, i) for i in (range(int(lo), int(hi) + 1) if lo else (int(one),)))
    return out


def parse(lines):
    """[(function, [(address, mnemonic, operands)])] of llvm-objdump -d."""
    functions, code = [], []
    for line in lines:
        if line.startswith("\t"):
            text, _, comment = line.partition("//")
            if not comment:
                continue                      # "...": padding
            op, _, args = text.strip().partition(" ")
            code.append((int(comment.split(":")[0], 16), op, args.strip()))
        elif line.endswith(">:"):
            code = []
            functions.append((line[line.index("<") + 1:-2], code))
    return functions


def too_early(code):
    """[(MFMA, early use, issue slots between them)] of one function."""
    index = {addr: i for i, (addr, _, _) in enumerate(code)}

    def after(i):
        """Indexes that may run after instruction i."""
        addr, op, args = code[i]
        nxt = []
        if op == "s_branch" or op.startswith("s_cbranch"):
            off = int(args.split()[0])
            nxt.append(index[addr + 4 + 4 * (off - 65536 if off >= 32768 else off)])
        if op not in ("s_branch", "s_endpgm") and i + 1 < len(code):
            nxt.append(i + 1)
        return nxt

    found = []
    for i, (_, op, args) in enumerate(code):
        if not op.startswith("v_mfma"):
            continue
        passes = PASSES[op]
        dst = args.split(",")[0]
        result = registers(dst)
        best, todo = {}, [(j, 0) for j in after(i)]
        while todo:
            j, slots = todo.pop()
            if slots >= passes + WAIT or best.get(j, 99) <= slots:
                continue
            best[j] = slots
            _, o, a = code[j]
            used = registers(a) & result if o[0] != "s" else set()
            if o.startswith("v_mfma"):
                # among themselves the matrix cores keep the order of results and addends;
                # an operand they do not
                used = registers(" ".join(a.split(", ")[1:3])) & result
                if not used:
                    slots = max(slots, passes)   # it is taken when the passes are through
            if used:
                found.append((f"{op} {args}", f"{o} {a}", slots))
                continue
            slots += int(a) + 1 if o == "s_nop" else 1
            todo.extend((k, slots) for k in after(j))
    return found


LATE = ["\tv_mfma_f32_16x16x128_f8f6f4 v[4:7], v[8:15], v[16:23], 0 // 000000000100: 0 0",
        "\ts_cbranch_scc1 1 // 000000000108: 0", "\tv_mov_b32_e32 v5, 0 // 00000000010C: 0",
        "\ts_nop 9 // 000000000110: 0", "\tv_mov_b32_e32 v4, 0 // 000000000114: 0",
        "\ts_endpgm // 000000000118: 0"]


def test_walk_follows_both_sides_of_a_branch():
    (_, code), = parse(["0000 <f>:"] + LATE)
    assert sorted((slots, use) for _, use, slots in too_early(code)) == [
        (1, "v_mov_b32_e32 v5, 0"), (11, "v_mov_b32_e32 v4, 0")]


@pytest.mark.skipif(not os.path.exists(OBJDUMP), reason="needs the ROCm toolchain's llvm-objdump")
def test_every_mfma_result_is_waited_for(tmp_path):
    mfmas, found = 0, []
    for n, obj in enumerate(code_objects(_lib.LIB_PATH)):
        path = tmp_path / f"{n}.o"
        path.write_bytes(obj)
        text = subprocess.run([OBJDUMP, "-d", str(path)], capture_output=True, text=True, check=True).stdout
        for name, code in parse(text.splitlines()):
            mfmas += sum(op.startswith("v_mfma") for _, op, _ in code)
            found += [(name, *f) for f in too_early(code)]
    assert mfmas > 1000 and not found, found[:8]
