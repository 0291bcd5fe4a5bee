"""The built library's instructions (no GPU): between a matrix instruction and a vector instruction that
touches its registers lie the wait states that gfx950 asks for. The compiler keeps them for its own
instructions, but not around inline asm, which the trellis decode is written in; a violation gives wrong
weights now and then."""
import os
import re
import subprocess

import pytest

from eva_amd import _lib

OBJDUMP = "/opt/rocm/llvm/bin/llvm-objdump"
# passes of a matrix instruction -> wait states before its sums' old registers may be written, and
# before its results' registers may be read or written
WAITS = {"v_mfma_f32_4x4x4_16b_f16": (1, 5), "v_mfma_f32_16x16x32_f16": (3, 7)}


def _regs(operand):
    m = re.fullmatch(r"-?\|?v(?:(\d+)|\[(\d+):(\d+)\])\|?", operand.split()[0] if operand.split() else "")
    if not m:
        return frozenset()
    lo, hi = (m[1], m[1]) if m[1] else (m[2], m[3])
    return frozenset(range(int(lo), int(hi) + 1))


def _violations(code):
    """code: [(address, instruction, branch target or None)] of one function, addresses ascending."""
    at = {a: i for i, (a, _, _) in enumerate(code)}
    bad = []
    for i, (_, text, _) in enumerate(code):
        if not text.startswith("v_mfma"):
            continue
        name, rest = text.split(None, 1)
        old_wait, new_wait = WAITS[name]
        new, _, _, old = ([_regs(o) for o in rest.split(",")] + [frozenset()])[:4]
        paths, seen = [(i + 1, 0)], set()
        while paths:
            j, waited = paths.pop()
            if j >= len(code) or waited >= new_wait or (j, waited) in seen:
                continue
            seen.add((j, waited))
            _, other, target = code[j]
            op, _, args = other.partition(" ")
            if op == "s_nop":
                paths.append((j + 1, waited + int(args) + 1))
                continue
            if op == "s_endpgm":
                continue
            if op.startswith(("v_", "ds_", "buffer_", "global_", "flat_", "scratch_")) and not op.startswith("v_mfma"):
                ops = [_regs(o) for o in args.split(",")]
                written = (ops[0] if op.startswith("v_") else frozenset()) | (ops[1] if "swap" in op else frozenset())
                read = frozenset().union(*(ops[1:] if op.startswith("v_") else ops))
                if (written | read) & new or (waited < old_wait and written & (old - new)):
                    bad.append((text, other, waited))
            if target in at:
                paths.append((at[target], waited + 1))
            if op != "s_branch":
                paths.append((j + 1, waited + 1))
    return bad


def _functions(code_object):
    out = subprocess.run([OBJDUMP, "-d", "--no-show-raw-insn", code_object], capture_output=True, text=True, check=True).stdout
    name, code, start = None, [], 0
    for line in out.splitlines():
        m = re.match(r"^([0-9a-f]+) <(.+)>:", line)
        if m:
            if code:
                yield name, code
            name, code, start = m[2], [], int(m[1], 16)
        elif line.startswith("\t") and name:
            text, _, note = line.partition("//")
            target = re.search(r"<.*\+0x([0-9a-f]+)>", note)
            if ":" not in note:
                continue
            code.append((int(note.split(":")[0], 16), text.strip(), start + int(target[1], 16) if target else None))
    if code:
        yield name, code


def test_violations_are_found():
    mfma = "v_mfma_f32_16x16x32_f16 v[4:7], v[8:11], v[12:15], v[0:3]"

    def run(*texts):
        return len(_violations([(4 * i, t, None) for i, t in enumerate((mfma,) + texts)]))

    assert run("v_mad_u32_u16 v2, v20, v21, v22") == 1                                  # still read as the old sums
    assert run("s_nop 1", "v_mad_u32_u16 v2, v20, v21, v22") == 1
    assert run("s_nop 2", "v_mad_u32_u16 v2, v20, v21, v22") == 0
    assert run("s_nop 5", "v_mul_lo_u16_sdwa v5, v20, v21 dst_sel:WORD_1") == 1         # yet to be written
    assert run("s_nop 5", "v_add_f32_e32 v20, v5, v21") == 1                            # not yet there
    assert run("s_nop 6", "v_add_f32_e32 v5, v5, v21") == 0
    assert run("v_mad_u32_u16 v8, v20, v21, v12") == 0                                  # its factors may change
    back = [(0, "v_mad_u32_u16 v2, v20, v21, v22", None), (4, mfma, None), (8, "s_cbranch_scc0 65533", 0), (12, "s_endpgm", None)]
    assert len(_violations(back)) == 1                                                  # across a loop's end


def test_built_library_keeps_the_wait_states(tmp_path):
    if not os.path.exists(OBJDUMP):
        pytest.skip("no llvm-objdump")
    _lib.lib()
    lib = tmp_path / "lib.so"
    lib.write_bytes(open(os.path.join(os.path.dirname(_lib.__file__), "libevamx.so"), "rb").read())
    subprocess.run([OBJDUMP, "--offloading", "lib.so"], cwd=tmp_path, capture_output=True, check=True)
    objects = sorted(p for p in os.listdir(tmp_path) if p.endswith("gfx950"))
    assert len(objects) >= 10
    count, bad = 0, []
    for o in objects:
        for name, code in _functions(tmp_path / o):
            count += sum(t.startswith("v_mfma") for _, t, _ in code)
            bad += [(name,) + v for v in _violations(code)]
    assert count > 10000 and not bad, (len(bad), bad[:8])
