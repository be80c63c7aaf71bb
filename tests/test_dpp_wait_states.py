"""The device code of the built library: lane-crossing operands (DPP) and lane masks wait as the hardware asks.

A DPP operand needs two wait states behind the vector instruction that wrote its register, and five behind one that
wrote EXEC.  The compiler keeps both where it sees the instructions; the scan's inline assembly keeps the first by `s_nop`
statements of its own, which hold only while no copy of an operand lands between them and the read.

A scalar register (a lane mask, vcc) that a vector instruction wrote needs two wait states before another reads it."""
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


# vector instructions with a second result, the carry
CARRIES = re.compile(r"v_(add|sub|subrev|addc|subb|subbrev)_co_|v_div_scale|v_mad_[ui]64")


def _scalars(operand):
    """The scalar registers an operand names."""
    operand = operand.strip("-|")
    if operand.startswith("vcc"):
        return {"vcc"}
    m = re.fullmatch(r"s(\d+)", operand) or re.fullmatch(r"s\[(\d+):(\d+)\]", operand)
    return set(range(int(m.group(1)), int(m.groups()[-1]) + 1)) if m else set()


def short_mask_waits(text):
    """(reads of scalar registers by vector instructions seen, lines that come too soon behind a vector instruction's write)."""
    code, before = _parse(text)
    seen, bad = 0, []

    def registers(entry):
        operands = [_scalars(o.split(" ")[0]) for o in entry[2]]
        results = 2 if CARRIES.match(entry[1]) else 1
        return set().union(*operands[:results]), set().union(*operands[results:])

    for entry in code:
        if not entry or not entry[1].startswith("v_"):
            continue
        read = registers(entry)[1]
        if not read:
            continue
        seen += 1
        todo = [(i, 0) for i in before.get(entry[0], [])]
        while todo:
            index, waited = todo.pop()
            address, mnemonic, operands, rest = code[index]
            if mnemonic.startswith("v_") and registers(code[index])[0] & read:
                bad.append(f"{address:x} {mnemonic} {rest} -> {entry[0]:x} {entry[1]} {entry[3]}")
                break
            waited += int(rest) + 1 if mnemonic == "s_nop" else 1
            if waited < 2:
                todo += [(i, waited) for i in before.get(address, [])]
    return seen, bad


@pytest.mark.parametrize("write,read,other", [
    ("v_cmp_gt_f32_e32 vcc, 0, v59", "v_cndmask_b32_e64 v56, v55, -v55, vcc", "v_cndmask_b32_e64 v56, v55, -v55, s[2:3]"),
    ("v_cmp_gt_f32_e64 s[4:5], 0, v59", "v_cndmask_b32_e64 v56, v55, v54, s[4:5]", "v_cndmask_b32_e32 v56, v55, v54, vcc"),
    ("v_addc_co_u32_e64 v1, vcc, 0, v1, s[6:7]", "v_cndmask_b32_e32 v56, v55, v54, vcc", "v_mul_f32_e32 v2, s9, v2"),
    ("v_readfirstlane_b32 s9, v3", "v_mul_f32_e32 v2, s9, v2", "v_mul_f32_e32 v2, s8, v2"),
])
def test_the_check_sees_masks(write, read, other):
    for between, ok in [([], False), (["s_nop 0"], False), (["s_nop 1"], True), (["v_mov_b32_e32 v6, 0", "s_waitcnt lgkmcnt(0)"], True)]:
        assert bool(short_mask_waits(_listing(write, *between, read))[1]) != ok
    assert not short_mask_waits(_listing(write, other))[1]


def test_lane_masks_of_the_library_wait(tmp_path):
    if not os.path.exists(LIBRARY) or not os.path.exists(OBJDUMP):
        pytest.skip("needs the built library and llvm-objdump")
    shutil.copy(LIBRARY, tmp_path / "lib.so")
    subprocess.run([OBJDUMP, "--offloading", "lib.so"], cwd=tmp_path, check=True, stdout=subprocess.DEVNULL)
    seen, bad = 0, []
    for part in sorted(p for p in os.listdir(tmp_path) if "gfx950" in p):
        text = subprocess.run([OBJDUMP, "-d", part], cwd=tmp_path, check=True, capture_output=True, text=True).stdout
        n, b = short_mask_waits(text)
        seen += n
        bad += b
    assert seen > 10000
    assert not bad, "\n".join(bad[:20])
