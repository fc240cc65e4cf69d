"""Wait states the hardware leaves to software, looked for in the library's own machine code.

The compiler puts them between instructions that it makes itself.  It does not look inside inline assembly, so
a store, load or wait written that way can stand too close to what the compiler puts around it, and nothing at run
time says so.  The rules checked are those that the memory instructions used here fall under (CDNA3 instruction set
guide, "Manually Inserted Wait States"; in wait states: one per instruction, N + 1 for s_nop N):

- a flat, global or scratch store of more than 64 bits, or a buffer store of that size without a scalar offset, then a
  vector instruction that writes one of the registers holding its data: 2
- a vector instruction that writes a scalar register, then a vector memory instruction that reads it: 5
- a scalar write of M0, then a load straight into LDS: 1
"""
import os
import re
import struct
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
LIB = os.path.join(ROOT, "grad.cpp_amd", "lib", "libgradhip.so")
OBJDUMP = "/opt/rocm/llvm/bin/llvm-objdump"

_REG = re.compile(r"\b([vsa])(?:(\d+)\b|\[(\d+):(\d+)\])|\b(vcc|m0)\b")
_LINE = re.compile(r"^\t(\S+)(?: (.*?))?\s*// ([0-9A-F]+):")
_TARGET = re.compile(r"<([^>+]+)(?:\+0x([0-9a-f]+))?>\s*$")


def code_objects(path):
    """The gfx950 code objects bundled into a library."""
    data, at = open(path, "rb").read(), 0
    magic = b"__CLANG_OFFLOAD_BUNDLE__"
    while (at := data.find(magic, at)) >= 0:
        count, = struct.unpack_from("<Q", data, at + 24)
        entry = at + 32
        for _ in range(count):
            offset, size, length = struct.unpack_from("<QQQ", data, entry)
            triple = data[entry + 24:entry + 24 + length].decode()
            entry += 24 + length
            if "gfx950" in triple:
                yield data[at + offset:at + offset + size]
        at = entry


def registers(text):
    """The registers an operand names, as a set of ('v', 3), ('s', 106), ('m0', 0) ..."""
    found = set()
    for kind, one, lo, hi, name in _REG.findall(text):
        if name:
            found |= {("s", 106), ("s", 107)} if name == "vcc" else {("m0", 0)}
        else:
            found |= {(kind, i) for i in range(int(one or lo), int(one or hi) + 1)}
    return found


def written(op, operands):
    """Registers a vector arithmetic or scalar instruction writes."""
    if op.startswith(("v_cmpx", "v_nop")) or not operands:
        return set()
    if op.startswith("v_cmp") and op.endswith("_e32"):
        return {("s", 106), ("s", 107)}
    out = registers(operands[0])
    if len(operands) > 1 and (re.match(r"v_(add|sub|subrev|addc|subb|subbrev)_co|v_div_scale|v_mad_[ui]64", op) or "swap" in op):
        out |= registers(operands[1])
    return out


def stored_data(op, operands):
    """Registers whose contents a store of more than 64 bits reads late."""
    if not re.search(r"_store_dwordx[34]$", op):
        return set()
    if op.startswith("buffer_"):
        return set() if re.match(r"s\d", operands[3].split()[0]) else registers(operands[0])
    return registers(operands[1])


def parse(listing):
    code, labels = [], {}
    for line in listing.splitlines():
        m = _LINE.match(line)
        if m:
            op, rest = m.group(1), m.group(2) or ""
            target = _TARGET.search(line) if op.startswith(("s_cbranch", "s_branch")) else None
            code.append((int(m.group(3), 16), op, [o.strip() for o in rest.split(",")] if rest else [],
                         (target.group(1), int(target.group(2) or "0", 16)) if target else None))
        elif line.endswith(">:"):
            labels[line.split("<")[-1][:-2]] = len(code)
    return code, labels


def behind(code, at_address, labels, i, states):
    """(wait states in between, instruction) for everything reachable within so many wait states of i."""
    todo = [(i + 1, 0)]
    while todo:
        j, waited = todo.pop()
        while waited < states and j < len(code):
            _, op, operands, target = code[j]
            yield waited, j
            if op in ("s_endpgm", "s_setpc_b64", "s_swappc_b64"):
                break
            waited += int(operands[0]) + 1 if op == "s_nop" else 1
            if target and target[0] in labels:
                goal = at_address.get(code[labels[target[0]]][0] + target[1])
                if goal is not None:
                    todo.append((goal, waited))
                if op == "s_branch":
                    break
            j += 1


def violations(listing):
    code, labels = parse(listing)
    at_address = {c[0]: i for i, c in enumerate(code)}
    bad = []
    for i, (address, op, operands, _) in enumerate(code):
        if data := stored_data(op, operands):
            for _, j in behind(code, at_address, labels, i, 2):
                if code[j][1].startswith("v_") and written(*code[j][1:3]) & data:
                    bad.append(("data of a wide store written", address, op, code[j][1:3]))
        scalars = {r for r in written(op, operands) if r[0] == "s"} if op.startswith("v_") else set()
        if scalars:
            for _, j in behind(code, at_address, labels, i, 5):
                name, args = code[j][1:3]
                if name.startswith(("global_", "buffer_", "flat_", "scratch_")) and registers(",".join(args)) & scalars:
                    bad.append(("scalar written by a vector instruction read", address, op, code[j][1:3]))
        if op.startswith("s_") and operands and operands[0] == "m0" and not op.startswith(("s_cmp", "s_bitcmp")):
            for _, j in behind(code, at_address, labels, i, 1):
                name, args = code[j][1:3]
                if "_lds_" in name or (name.startswith("buffer_load") and " lds" in ",".join(args)):
                    bad.append(("M0 read", address, op, code[j][1:3]))
    return code, bad


def test_the_rules_are_seen():
    """Each rule on the shortest listing that breaks it, and on one that keeps it."""
    def listing(*lines):
        rows = [(*line.split(" -> "), "")[:2] for line in lines]
        return "<k>:\n" + "".join(f"\t{text} // {4 * i:012X}: 00000000 {goal}\n" for i, (text, goal) in enumerate(rows))

    store = "global_store_dwordx4 v[0:1], v[4:7], off sc1"
    assert violations(listing(store, "v_mov_b32_e32 v5, v9"))[1]
    assert violations(listing(store, "s_nop 0", "v_mov_b32_e32 v5, v9"))[1]
    assert not violations(listing(store, "s_nop 1", "v_mov_b32_e32 v5, v9"))[1]
    assert not violations(listing(store, "v_mov_b32_e32 v8, v5"))[1]
    assert not violations(listing(store, "ds_read_b32 v5, v9"))[1]
    assert not violations(listing("global_store_dwordx2 v[0:1], v[4:5], off", "v_mov_b32_e32 v5, v9"))[1]
    assert violations(listing(store, "s_cbranch_execz 1 -> <k+0xc>", "s_endpgm",
                              "v_mov_b32_e32 v5, v9"))[1]
    assert violations(listing("buffer_store_dwordx4 v[4:7], v0, s[8:11], 0 offen", "v_mov_b32_e32 v5, v9"))[1]
    assert not violations(listing("buffer_store_dwordx4 v[4:7], v0, s[8:11], s3 offen", "v_mov_b32_e32 v5, v9"))[1]
    load = "global_load_lds_dwordx4 v0, s[6:7]"
    assert violations(listing("v_readfirstlane_b32 s6, v1", "s_mov_b32 m0, s2", "s_nop 0", load))[1]
    assert not violations(listing("v_readfirstlane_b32 s6, v1", "s_mov_b32 m0, s2", "s_nop 3", load))[1]
    assert violations(listing("s_mov_b32 m0, s2", load))[1]
    assert violations(listing("v_cmp_eq_u32_e64 s[6:7], v1, v2", "s_nop 3", load))[1]


@pytest.mark.skipif(not os.path.exists(OBJDUMP), reason="no disassembler")
def test_wait_states_of_the_library(tmp_path):
    assert os.path.exists(LIB), "not built"
    objects = list(code_objects(LIB))
    assert len(objects) >= 5  # a code object per HIP source
    wide_stores = 0
    for i, content in enumerate(objects):
        path = tmp_path / f"{i}.co"
        path.write_bytes(content)
        listing = subprocess.run([OBJDUMP, "-d", "--no-show-raw-insn", "--no-leading-addr", str(path)], check=True,
                                 capture_output=True, text=True).stdout
        code, bad = violations(listing)
        assert not bad, f"{len(bad)} places, the first ones: " + "; ".join(f"{w} at {a:#x}: {op} then {b}" for w, a, op, b in bad[:8])
        wide_stores += sum(1 for c in code if re.search(r"_store_dwordx4$", c[1]))
    assert wide_stores > 100  # (the listing is read at all)
