"""Wait states that gfx950 leaves to software, in the library as it was compiled.  The compiler keeps them for the instructions that it
knows; what is written as inline assembly it takes for neither a vector nor a memory instruction, so the waits have to be in the text."""
import collections
import glob
import os
import re
import shutil
import struct
import subprocess

import pytest

OBJDUMP = shutil.which("llvm-objdump") or "/opt/rocm/llvm/bin/llvm-objdump"
REGS = re.compile(r"\b([vsa])\[(\d+):(\d+)\]|\b([vsa])(\d+)\b")
NO_RESULT = re.compile(r"(global|flat|buffer|scratch)_(store|load_lds)|ds_write|s_cbranch|s_branch|s_waitcnt|s_nop|s_barrier|s_endpgm|s_cmp|s_bitcmp|s_setprio|s_sleep")
Ins = collections.namedtuple("Ins", "op text operands written read waits")


def _regs(text):
    return {(m[1] or m[4], n) for m in REGS.finditer(text) for n in (range(int(m[2]), int(m[3]) + 1) if m[1] else (int(m[5]),))}


def _parse(text):
    op, _, rest = text.partition(" ")
    operands = re.split(r",(?![^\[]*\])", rest)
    written = set() if NO_RESULT.match(op) else _regs(operands[0])
    if "swap" in op:
        written |= _regs(operands[1])
    reads_first = not written or "swap" in op or op.startswith(("v_fmac", "v_dot2c"))
    return Ins(op, text, operands, written, _regs(rest if reads_first else ",".join(operands[1:])), int(operands[0], 0) + 1 if op == "s_nop" else 1)


def _code_objects(library):
    """The gfx950 code objects of the offload bundles in a library."""
    data, at = open(library, "rb").read(), 0
    magic = b"__CLANG_OFFLOAD_BUNDLE__"
    while (at := data.find(magic, at)) >= 0:
        entry = at + len(magic) + 8
        for _ in range(struct.unpack_from("<Q", data, entry - 8)[0]):
            offset, size, length = struct.unpack_from("<QQQ", data, entry)
            if b"gfx950" in data[entry + 24: entry + 24 + length]:
                yield data[at + offset: at + offset + size]
            entry += 24 + length
        at += len(magic)


@pytest.fixture(scope="module")
def functions(tmp_path_factory):
    """[(name, instructions, predecessors of each)]"""
    from loongforge_amd import _lib

    if not os.path.exists(OBJDUMP):
        pytest.skip("no llvm-objdump")
    found, parsed = [], {}
    for n, code in enumerate(_code_objects(_lib.LIB_PATH)):
        path = tmp_path_factory.mktemp("code") / ("%d.o" % n)
        path.write_bytes(code)
        out = subprocess.run([OBJDUMP, "-d", "--no-show-raw-insn", str(path)], capture_output=True, text=True, check=True).stdout
        name, ins, places, jumps = None, [], {}, []
        for line in out.splitlines() + ["0 <end>:"]:
            if m := re.match(r"[0-9a-f]+ <(.*)>:", line):
                before = collections.defaultdict(list)
                for k, to in jumps:
                    before[places[to]].append(k)
                for k in range(1, len(ins)):
                    if ins[k - 1].op not in ("s_branch", "s_endpgm", "s_setpc_b64"):
                        before[k].append(k - 1)
                if ins:
                    found.append((name, ins, before))
                name, ins, places, jumps, start = m[1], [], {}, [], None
            elif m := re.match(r"\s+(\S.*?)\s*// ([0-9A-F]+):(?:.*<.*?(?:\+0x([0-9a-f]+))?>)?", line):
                start = int(m[2], 16) if start is None else start
                places[int(m[2], 16) - start] = len(ins)
                if m[1].startswith(("s_branch", "s_cbranch")):
                    jumps.append((len(ins), int(m[3] or "0", 16)))
                if m[1] not in parsed:
                    parsed[m[1]] = _parse(m[1])
                ins.append(parsed[m[1]])
    assert len(found) > 100
    return found


def _memory(i):
    return i.op.startswith(("global_", "flat_", "buffer_", "scratch_"))


def _vector(i):
    return i.op.startswith("v_") and not i.op.startswith(("v_mfma", "v_smfma"))


# wait states, the second instruction, the first, and the registers that they share
RULES = {
    "a matrix instruction reads what a vector instruction wrote":
        (2, lambda i: i.op.startswith("v_mfma"), _vector, lambda first, second: first.written & second.read),
    "a memory instruction reads a scalar register that a vector instruction wrote":
        (5, _memory, _vector, lambda first, second: {r for r in first.written if r[0] == "s"} & second.read),
    "a vector instruction writes the data of a store of more than 8 bytes":
        (2, lambda i: i.op.startswith("v_"), lambda i: re.match(r"(global|flat|scratch)_store_dwordx[34]", i.op),
         lambda first, second: _regs(first.operands[1]) & second.written),
}


@pytest.mark.parametrize("rule", RULES)
def test_wait_states(functions, rule):
    need, is_second, is_first, shared = RULES[rule]
    short = []
    for name, ins, before in functions:
        for k, second in enumerate(ins):
            if not is_second(second):
                continue
            ways, seen = [(p, 0) for p in before[k]], {}
            while ways:
                j, waits = ways.pop()
                if waits >= need or seen.get(j, need) <= waits:
                    continue
                seen[j] = waits
                if is_first(ins[j]) and shared(ins[j], second):
                    short.append("%s: %s | %d | %s" % (name, ins[j].text, waits, second.text))
                ways += [(p, waits + ins[j].waits) for p in before[j]]
    assert not short, "\n".join(short)


def test_wide_stores_in_assembly_bring_their_wait():
    """Whatever the compiler puts behind them today."""
    from loongforge_amd.csrc import build

    found = 0
    for path in sorted(glob.glob(os.path.join(build.HERE, "**", "*.h*"), recursive=True)):
        for text in re.findall(r'\basm\b[^;"]*((?:"(?:[^"\\]|\\.)*"\s*)+)', open(path).read()):
            behind = re.split(r"_store_dwordx[34]\b", text)
            found += len(behind) - 1
            assert len(behind) == 1 or re.search(r"s_nop [1-9]", behind[-1]), (path, text)
    assert found
