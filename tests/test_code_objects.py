"""What the compiled gfx950 code itself has to hold where the sources reach past the compiler: the hardware
needs five wait states between a vector instruction that writes a scalar register and a memory instruction that
addresses through it, and the compiler does not look into inline assembly for the latter."""
import os
import re
import struct
import subprocess

import pytest

from camelid_amd import build

OBJDUMP = "/opt/rocm/llvm/bin/llvm-objdump"
LINE = re.compile(r"^\t(\S+)\s*(.*?)\s*// ([0-9A-F]+): [0-9A-F ]+(?:<(.+)\+0x([0-9a-f]+)>)?$")
SGPR = re.compile(r"\bs\[(\d+):(\d+)\]|\bs(\d+)\b|\b(vcc)\b")
WAIT_STATES = 5


def code_objects():
    """The gfx950 code objects of the library (uncompressed offload bundles, one per source file)."""
    data = open(build.LIB, "rb").read()
    at = 0
    while (at := data.find(b"__CLANG_OFFLOAD_BUNDLE__", at)) >= 0:
        (n,), p = struct.unpack_from("<Q", data, at + 24), at + 32
        for _ in range(n):
            offset, size, length = struct.unpack_from("<QQQ", data, p)
            if b"gfx950" in data[p + 24:p + 24 + length] and size:
                yield data[at + offset:at + offset + size]
            p += 24 + length
        at += 24


def sgprs(text):
    out = set()
    for lo, hi, one, vcc in SGPR.findall(text):
        out |= {"vcc"} if vcc else set(range(int(lo or one), int(hi or one) + 1))
    return out


def written_by_vector(op, operands):
    if not op.startswith("v_"):
        return set()
    parts = operands.split(", ")
    carry = "_co_" in op or op.startswith(("v_div_scale", "v_mad_u64", "v_mad_i64"))
    return sgprs(", ".join(parts[:2 if carry else 1]))


def hazards(listing):
    """[(function, address of the write, address of the load)] in an llvm-objdump listing."""
    found, code, name, start = [], [], "", {}
    for line in listing.splitlines():
        head = re.match(r"^([0-9a-f]{16}) <(.+)>:$", line)
        if head:
            name = head.group(2)
            start[name] = int(head.group(1), 16)
            continue
        m = LINE.match(line)
        if m:
            op, operands, at, target, plus = m.groups()
            code.append((name, op, operands, int(at, 16), (target, int(plus, 16)) if target and op.startswith(("s_cbranch", "s_branch")) else None))
    index = {c[3]: i for i, c in enumerate(code)}
    for i, (name, op, operands, at, _) in enumerate(code):
        regs = written_by_vector(op, operands)
        if not regs:
            continue
        todo, seen = [(i + 1, 0, frozenset(regs))], set()
        while todo:
            k, waited, live = state = todo.pop()
            if state in seen or k >= len(code) or waited >= WAIT_STATES or not live or code[k][0] != name:
                continue
            seen.add(state)
            _, kop, kops, kat, target = code[k]
            if kop.startswith(("global_", "buffer_", "flat_", "scratch_")) and sgprs(kops) & live:
                found.append((name, hex(at), hex(kat)))
            if kop.startswith("s_") and not kop.startswith(("s_cmp", "s_cbranch", "s_branch", "s_waitcnt", "s_nop", "s_barrier", "s_bitcmp")):
                live = live - sgprs(kops.split(", ")[0])  # (a scalar write waits for the vector one, and no memory instruction has to wait for it)
            waited += int(kops, 0) + 1 if kop == "s_nop" else 1
            if target:
                todo.append((index[start[target[0]] + target[1]], waited, live))
            if kop not in ("s_branch", "s_endpgm", "s_setpc_b64"):
                todo.append((k + 1, waited, live))
    return found


def test_the_check_finds_a_base_read_too_early():
    text = "0000000000000100 <f>:\n" + "".join(
        f"\t{ins} // {0x100 + 4 * i:012X}: 00000000\n"
        for i, ins in enumerate(["v_readlane_b32 s2, v1, 0", "v_readlane_b32 s3, v1, 1", "s_mov_b32 m0, s9", "s_nop 0", "global_load_lds_dword v4, s[2:3]", "s_endpgm"]))
    assert hazards(text) == [("f", "0x100", "0x110"), ("f", "0x104", "0x110")]
    assert not hazards(text.replace("s_nop 0", "s_nop 3"))
    assert not hazards(text.replace("s_nop 0", "s_mov_b64 s[4:5], s[2:3]").replace("v4, s[2:3]", "v4, s[4:5]"))


@pytest.mark.skipif(not os.path.exists(OBJDUMP), reason="no llvm-objdump")
def test_no_memory_instruction_addresses_through_a_register_just_written(tmp_path):
    n, loads = 0, 0
    for i, blob in enumerate(code_objects()):
        path = tmp_path / f"{i}.co"
        path.write_bytes(blob)
        listing = subprocess.run([OBJDUMP, "-d", path], capture_output=True, text=True, check=True).stdout
        n, loads = n + 1, loads + listing.count("\tglobal_load_lds_")
        assert hazards(listing) == []
    assert n == sum(s.endswith(".hip") for s in build.SOURCES)
    assert loads > 1000  # (the wide kernels' inline assembly was looked at)
