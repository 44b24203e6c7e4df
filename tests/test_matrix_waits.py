"""The results of matrix instructions in the built library are never read, or overwritten, before they are there.

The hardware does not hold such a reader back; the compiler puts the wait in.  It has been seen to leave it out on one of two
paths that meet again (`settle` in csrc/common.h), which no run shows reliably, so the compiled kernels of this library are
walked here: from every matrix instruction along every path, counting a state per instruction and as many as an s_nop names."""
import os
import re
import shutil
import struct
import subprocess

import pytest

OBJDUMP = next((p for p in ("/opt/rocm/llvm/bin/llvm-objdump", shutil.which("llvm-objdump")) if p and os.path.exists(p)), None)
# states from an instruction to a reader of its result: what this compiler keeps where no branch lies between
STATES = {"16x16x4_f32": 10, "16x16x32_bf16": 8, "32x32x16_bf16": 12}
REGISTER = re.compile(r"\b([va])(?:\[(\d+):(\d+)\]|(\d+)\b)")
STORES = ("global_store", "global_atomic", "ds_write", "ds_add", "buffer_store", "scratch_store", "flat_store")


def registers(text):
    found = set()
    for kind, first, last, one in REGISTER.findall(text):
        found.update((kind, i) for i in (range(int(first), int(last) + 1) if first else (int(one),)))
    return found


def operands(text):
    return re.split(r",\s*(?![^\[]*\])", text) if text else []


def kernels(listing):
    """(name, [(address, instruction, operands, rest of the line)]) of an llvm-objdump listing."""
    name, body = None, []
    for line in listing.splitlines():
        head = re.match(r"^[0-9a-f]{16} <(.+)>:", line)
        if head:
            if name:
                yield name, body
            name, body = head.group(1), []
        elif name and line.startswith("\t"):
            code, _, rest = line.partition("//")
            at = re.match(r"\s*([0-9A-F]+):", rest)
            if at:
                parts = code.split(None, 1)
                body.append((int(at.group(1), 16), parts[0], parts[1].strip() if len(parts) > 1 else "", rest))
    if name:
        yield name, body


def read_too_early(body):
    """The places (address of the matrix instruction, states that lie between, states wanted, what comes too early)."""
    place, start, met, found = {line[0]: i for i, line in enumerate(body)}, body[0][0], {}, []

    def after(i):
        _, name, _, rest = body[i]
        if name == "s_endpgm":
            return []
        assert name not in ("s_setpc_b64", "s_swappc_b64"), "a call: its target is not followed"
        if name.startswith(("s_branch", "s_cbranch")):
            target = place[start + int(re.search(r"<[^>]*?(?:\+0x([0-9a-f]+))?>\s*$", rest).group(1) or "0", 16)]
            return [target] if name == "s_branch" else [target, i + 1]
        return [i + 1]

    def touches(i):
        """The registers that instruction i reads too early or overwrites if a result is on its way to them.  (A matrix
        instruction may continue another one's sums at once.)"""
        if i not in met:
            _, name, text, _ = body[i]
            parts = operands(text)
            if name.startswith("v_mfma"):
                met[i] = registers(parts[1]) | registers(parts[2])
            elif name.startswith("s_") or not parts:
                met[i] = set().union(*(registers(part) for part in parts[1:])) if len(parts) > 1 else set()
            else:
                met[i] = registers(text)
        return met[i]

    for i, (address, name, text, _) in enumerate(body):
        if not name.startswith("v_mfma"):
            continue
        wanted = next(states for kind, states in STATES.items() if kind in name)
        result, least, ways = registers(operands(text)[0]), {}, [(j, 0) for j in after(i)]
        while ways:
            j, states = ways.pop()
            if states >= wanted or least.get(j, wanted) <= states:
                continue
            least[j] = states
            if touches(j) & result:
                found.append((hex(address), states, wanted, " ".join(body[j][1:3])))
                continue
            step = int(body[j][2], 0) + 1 if body[j][1] == "s_nop" else 1
            ways += [(k, states + step) for k in after(j)]
    return found


def code_objects(path):
    """The GPU's code objects inside a library that hipcc made."""
    data, at = open(path, "rb").read(), 0
    while (at := data.find(b"__CLANG_OFFLOAD_BUNDLE__", at)) >= 0:
        count, cursor = struct.unpack_from("<Q", data, at + 24)[0], at + 32
        for _ in range(count):
            offset, size, length = struct.unpack_from("<QQQ", data, cursor)
            target = data[cursor + 24:cursor + 24 + length]
            cursor += 24 + length
            if b"gfx950" in target and size:
                yield data[at + offset:at + offset + size]
        at += 24


def test_the_walk_finds_a_wait_that_only_one_path_has():
    """What the compiler has been seen to make: a long arm without a branch of its own, a short one that goes straight on."""
    lines = ["v_mfma_f32_16x16x4_f32 v[2:5], v7, v1, v[2:5]", "s_cbranch_scc1 13"] + ["v_fma_f32 v6, v7, v6, v1"] * 13 + [
        "s_add_i32 s0, s0, 1", "v_mul_f32_e32 v2, v2, v6", "s_endpgm"]

    def listing(lines):
        text = "0000000000001000 <kernel>:\n"
        for i, line in enumerate(lines):
            target = " <kernel+0x%x>" % (4 * (i + 14)) if "branch" in line else ""
            text += "\t%s // %012X: 00000000%s\n" % (line, 0x1000 + 4 * i, target)
        return list(kernels(text))[0][1]
    assert [(states, wanted) for _, states, wanted, _ in read_too_early(listing(lines))] == [(2, 10)]
    waited = lines[:16] + ["s_nop 15"] + lines[16:]
    assert read_too_early(listing(waited)) == []


@pytest.mark.skipif(OBJDUMP is None, reason="no disassembler here")
def test_no_kernel_reads_a_matrix_result_before_it_is_there(tmp_path):
    from tlie_amd.csrc import build
    if not build.is_current():
        build.build(verbose=False)
    walked = 0
    for number, content in enumerate(code_objects(build.library_path())):
        path = tmp_path / f"{number}.elf"
        path.write_bytes(content)
        listing = subprocess.run([OBJDUMP, "-d", "--no-show-raw-insn", str(path)], capture_output=True, text=True, check=True).stdout
        for name, body in kernels(listing):
            if any(line[1].startswith("v_mfma") for line in body):
                walked += 1
                assert read_too_early(body) == [], name
    assert walked > 100
