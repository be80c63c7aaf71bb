"""The device code of the built library: lane-crossing operands (DPP) wait as the hardware asks.

A DPP operand needs two wait states behind the vector instruction that wrote its register, and five behind one that
wrote EXEC.  The compiler keeps both where it sees the instructions; the scan's inline assembly keeps the first by `s_nop`
statements of its own, which hold only while no copy of an operand lands between them and the read."""
import os
import re
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
LIBRARY = os.path.join(ROOT, "snntc-2023_amd", "csrc", "libsnntc_hip.so")
OBJDUMP = "/opt/rocm/llvm/bin/llvm-objdump"
DPP = re.compile(r"row_newbcast|quad_perm|row_shr|row_shl|row_ror|row_bcast|row_mirror|row_half_mirror|wave_sh|wave_ro")


def _registers(operand):
    """The vector registers an operand names."""
    m = re.fullmatch(r"-?\|?v(\d+)\|?", operand) or re.fullmatch(r"v\[(\d+):(\d+)\]", operand)
    if not m:
        return range(0)
    return range(int(m.group(1)), int(m.groups()[-1]) + 1)


def _parse(text):
    """[(address, mnemonic, operands, rest of the line)] and {address: addresses that come before}, function by function."""
    code, before, starts = [], {}, {}
    name = None
    branches = []
    for line in text.splitlines():
        m = re.match(r"([0-9a-f]+) <(.+)>:$", line)
        if m:
            name = m.group(2)
            starts[name] = int(m.group(1), 16)
            code.append(None)
            continue
        m = re.match(r"\s+(\S+)\s*(.*?)\s*// ([0-9A-F]+): [0-9A-F ]+(?:<(.+?)(?:\+0x([0-9a-f]+))?>)?$", line)
        if not m:
            continue
        mnemonic, rest, address = m.group(1), m.group(2), int(m.group(3), 16)
        operands = [o.strip() for o in re.split(r",\s*(?![^\[]*\])", rest.split(" row_")[0].split(" quad_perm")[0])] if rest else []
        if code and code[-1] and code[-1][1] not in ("s_branch", "s_endpgm", "s_setpc_b64"):
            before.setdefault(address, []).append(len(code) - 1)
        if mnemonic.startswith(("s_cbranch", "s_branch")) and m.group(4):
            branches.append((len(code), m.group(4), int(m.group(5) or "0", 16)))
        code.append((address, mnemonic, operands, rest))
    for index, target, offset in branches:
        if target in starts:
            before.setdefault(starts[target] + offset, []).append(index)
    return code, before


def short_waits(text):
    """(DPP reads seen, lines that come too soon behind a write of their operand or of EXEC)."""
    code, before = _parse(text)
    seen, bad = 0, []
    for entry in code:
        if not entry or not entry[1].startswith("v_") or not DPP.search(entry[3]):
            continue
        seen += 1
        sources = [o for o in entry[2][1:] if _registers(o.split(" ")[0])]
        crossed = set(_registers(sources[0].split(" ")[0])) if sources else set()
        todo = [(i, 0) for i in before.get(entry[0], [])]
        while todo:
            index, waited = todo.pop()
            address, mnemonic, operands, rest = code[index]
            if mnemonic.startswith("v_"):
                written = set(_registers(operands[0].split(" ")[0])) if operands else set()
                if mnemonic.startswith("v_swap"):
                    written |= set(_registers(operands[1]))
                if (waited < 2 and written & crossed) or mnemonic.startswith("v_cmpx"):
                    bad.append(f"{address:x} {mnemonic} {rest} -> {entry[0]:x} {entry[1]} {entry[3]}")
                    break
            waited += int(rest) + 1 if mnemonic == "s_nop" else 1
            if waited < 5:
                todo += [(i, waited) for i in before.get(address, [])]
    return seen, bad


def _listing(*instructions):
    return "0000000000000100 <f>:\n" + "".join(f"\t{text} // {0x100 + 4 * i:012X}: 7E040280{extra}\n"
                                               for i, (text, extra) in enumerate((t if isinstance(t, tuple) else (t, "")) for t in instructions))


READ = "v_add_u32_dpp v2, v5, v34 row_newbcast:0 row_mask:0xf bank_mask:0xf bound_ctrl:1"


@pytest.mark.parametrize("between,ok", [([], False), (["s_nop 0"], False), (["s_nop 1"], True), (["v_mov_b32_e32 v6, 0", "s_waitcnt lgkmcnt(0)"], True)])
def test_the_check_counts_wait_states(between, ok):
    assert short_waits(_listing("v_mov_b32_e32 v5, v1", *between, READ)) == (1, []) if ok else short_waits(_listing("v_mov_b32_e32 v5, v1", *between, READ))[1]
    assert short_waits(_listing("v_mov_b32_e32 v34, v1", *between, READ)) == (1, [])               # the other operand may follow at once


def test_the_check_follows_branches_and_exec():
    loop = _listing(READ, "s_nop 4", "v_mov_b32_e32 v[4:5], v1", ("s_cbranch_scc1 65532", " <f>"), "s_endpgm")
    assert short_waits(loop)[1]
    assert short_waits(_listing("v_cmpx_gt_f32_e32 vcc, v58, v70", "s_nop 3", READ)) [1]
    assert short_waits(_listing("v_cmpx_gt_f32_e32 vcc, v58, v70", "s_nop 4", READ)) == (1, [])


def test_dpp_operands_of_the_library_wait(tmp_path):
    if not os.path.exists(LIBRARY) or not os.path.exists(OBJDUMP):
        pytest.skip("needs the built library and llvm-objdump")
    shutil.copy(LIBRARY, tmp_path / "lib.so")
    subprocess.run([OBJDUMP, "--offloading", "lib.so"], cwd=tmp_path, check=True, stdout=subprocess.DEVNULL)
    seen, bad = 0, []
    for part in sorted(p for p in os.listdir(tmp_path) if "gfx950" in p):
        text = subprocess.run([OBJDUMP, "-d", part], cwd=tmp_path, check=True, capture_output=True, text=True).stdout
        n, b = short_waits(text)
        seen += n
        bad += b
    assert seen > 10000
    assert not bad, "\n".join(bad[:20])
