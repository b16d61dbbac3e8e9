"""The built library's own code: between a matrix instruction and the first instruction that touches what it writes lie the wait states
that the hardware wants there, on every way through branches.  The compiler pads this distance, but where a branch leaves right behind
a product and joins again it has been seen to count one of the two ways only (the accumulator then lacks the product's last step)."""
import re
import shutil
import struct
import subprocess

import pytest

from speed3r_amd import build

OBJDUMP = shutil.which("llvm-objdump") or shutil.which("llvm-objdump", path="/opt/rocm/llvm/bin")
MAGIC = b"__CLANG_OFFLOAD_BUNDLE__"


def wait_states(op):
    """Behind a product of 4, 8 or 16 passes of the 16-bit unit, or the fp32 product of 8: to a vector or memory instruction that
    reads or writes the result, or a product that reads it as a factor."""
    m, _, k = map(int, re.match(r"v_mfma_f32_(\d+)x(\d+)x(\d+)", op).groups())
    if (m, k) == (16, 4):
        return 10
    return {(16, 16): 8, (16, 32): 8, (32, 16): 12, (32, 8): 20}[m, k]


def registers(operand):
    m = re.fullmatch(r"-?\|?([va])(?:\[(\d+):(\d+)\]|(\d+))\|?", operand)
    if not m:
        return set()
    lo = int(m[2] or m[4])
    return {m[1] + str(i) for i in range(lo, int(m[3] or lo) + 1)}


def code_objects(path):
    data, at = path.read_bytes(), 0
    while (at := data.find(MAGIC, at)) >= 0:
        entry = at + len(MAGIC) + 8
        for _ in range(struct.unpack_from("<Q", data, at + len(MAGIC))[0]):
            offset, size, length = struct.unpack_from("<QQQ", data, entry)
            if b"gfx950" in data[entry + 24:entry + 24 + length] and size:
                yield data[at + offset:at + offset + size]
            entry += 24 + length
        at += len(MAGIC)


def kernels(listing):
    """name -> instructions (mnemonic, operands, index of a branch's target or None)"""
    name, found = None, {}
    for line in listing.splitlines():
        if m := re.match(r"([0-9a-f]+) <(\S+)>:", line):
            name, start = m[2], int(m[1], 16)
            found[name] = ([], {}, start)
        elif name and (m := re.match(r"\s+([a-z]\w*)\s*(.*?)\s*// ([0-9A-F]+):(?:.*<\S+?\+0x([0-9a-f]+)>)?", line)):
            code, where, start = found[name]
            where[int(m[3], 16)] = len(code)
            code.append((m[1], [o.strip() for o in re.split(r",(?![^\[]*\])", m[2])], m[4] and start + int(m[4], 16)))
    return {n: [(op, args, where.get(to)) for op, args, to in code] for n, (code, where, _) in found.items()}


def too_close(code, first):
    """The instruction that touches the result of the product at ``first`` too early, or None."""
    result, need = registers(code[first][1][0]), wait_states(code[first][0])
    ways, seen = [(first + 1, 0)], {}
    while ways:
        i, states = ways.pop()
        while i < len(code) and states < need and seen.get(i, need) > states:
            seen[i] = states
            op, args, to = code[i]
            if op == "s_endpgm":
                break
            if op == "s_nop":
                states += int(args[0], 0)
            elif op == "s_branch":
                i = to - 1
            elif op.startswith("s_cbranch"):
                ways.append((to, states + 1))
            elif op.startswith("v_mfma"):
                if (registers(args[1]) | registers(args[2])) & result:
                    return f"{op} {args}: {states} of {need}"
                if registers(args[0]) & result:   # (another product into the same accumulator goes on from there)
                    break
            elif op[0] != "s":
                if any(registers(a.split()[0]) & result for a in args if a):
                    return f"{op} {args}: {states} of {need}"
            i, states = i + 1, states + 1
    return None


@pytest.mark.skipif(OBJDUMP is None, reason="no disassembler")
def test_products_are_finished_before_their_results_are_touched(tmp_path):
    if not build.library_path().exists():
        pytest.skip("the library is not built")
    products, short = 0, []
    for i, blob in enumerate(code_objects(build.library_path())):
        obj = tmp_path / f"{i}.o"
        obj.write_bytes(blob)
        text = subprocess.run([OBJDUMP, "-d", "--no-show-raw-insn", str(obj)], check=True, capture_output=True, text=True).stdout
        for name, code in kernels(text).items():
            at = [j for j, ins in enumerate(code) if ins[0].startswith("v_mfma")]
            products += len(at)
            short += [f"{name} {code[j][0]} {code[j][1]} -> {bad}" for j in at if (bad := too_close(code, j))]
    assert products > 1000
    assert not short, "\n".join(short)


def test_the_walk_sees_both_ways_of_a_branch():
    product = ("v_mfma_f32_16x16x4_f32", ["v[0:3]", "v8", "v9", "v[0:3]"], None)
    nop, read = ("s_nop", ["9"], None), ("v_max3_f32", ["v10", "v0", "s1", "v1"], None)
    rest = [("s_cbranch_scc1", ["2"], 3), nop, read, ("s_endpgm", [""], None)]
    assert too_close([product, *rest], 0)                                                     # the branch goes round the wait
    assert too_close([product, nop, ("s_cbranch_scc1", ["1"], 4), nop, read, rest[-1]], 0) is None
    assert too_close([product, ("s_nop", ["8"], None), read, rest[-1]], 0)                    # one state short
    assert too_close([product, ("s_nop", ["0x9"], None), read, rest[-1]], 0) is None
