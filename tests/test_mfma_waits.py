"""Every use of an MFMA's result waits for it, in the built library's code.

The hardware does not hold back a vector or memory instruction that reads (or
overwrites) an MFMA's result before it is there; the compiler keeps them
apart.  A kernel variant whose result was first used past a branch once read it
too early, so uses on either side of a branch are compared: none past one comes
after fewer instructions (an s_nop counts its own number) than the nearest in
straight code, per MFMA instruction.
"""
import re
import shutil
import subprocess
from pathlib import Path

import pytest

from ztensor_amd import build

OBJDUMP = Path("/opt/rocm/llvm/bin/llvm-objdump")
REG = re.compile(r"\bv(?:\[(\d+):(\d+)\]|(\d+)\b)")
FURTHEST = 24  # wait states past which no use needs a look (16 passes need 19)


def registers(text):
    found = set()
    for a, b, one in REG.findall(text):
        found.update(range(int(a), int(b) + 1) if a else (int(one),))
    return found


def functions(listing):
    """[(address, mnemonic, operands, branch target or None)] of each function."""
    out = []
    for line in listing.splitlines():
        if re.match(r"[0-9a-f]+ <.*>:$", line):
            out.append([])
        elif out and "//" in line:
            code, note = line.split("//", 1)
            mnemonic, _, operands = code.strip().partition(" ")
            target = re.search(r"<[^>]*?(?:\+0x([0-9a-f]+))?>", note)
            base = out[-1][0][0] if out[-1] else int(note.split(":")[0], 16)
            out[-1].append((int(note.split(":")[0], 16), mnemonic, operands.strip(),
                            base + int(target.group(1) or "0", 16) if target else None))
    return [f for f in out if f]


def uses(code):
    """(MFMA, wait states before the first use of its result, whether past a branch), along every path."""
    at = {c[0]: i for i, c in enumerate(code)}
    for i, (_, mfma, operands, _) in enumerate(code):
        if not mfma.startswith("v_mfma"):
            continue
        result = registers(operands.split(",")[0])
        seen, todo = {}, [(i + 1, 0, False)]
        while todo:
            j, waits, branched = todo.pop()
            if j >= len(code) or waits > FURTHEST or seen.get((j, branched), FURTHEST + 1) <= waits:
                continue
            seen[j, branched] = waits
            _, op, args, target = code[j]
            if op.startswith("v_mfma"):
                if registers(args.split(",")[0]) & result:
                    continue  # the sum goes on
            elif registers(args) & result:
                yield mfma, waits, branched
                continue
            if op == "s_endpgm":
                continue
            jump = op.startswith(("s_branch", "s_cbranch"))
            if jump and target in at:
                todo.append((at[target], waits + 1, True))
            if op != "s_branch":
                todo.append((j + 1, waits + (int(args, 0) + 1 if op == "s_nop" else 1), branched or jump))


def closest(listing):
    best = {}
    for code in functions(listing):
        for mfma, waits, branched in uses(code):
            best[mfma, branched] = min(waits, best.get((mfma, branched), FURTHEST))
    return best


def test_the_check_sees_an_early_use():
    text = """0000000000000000 <f>:
	v_mfma_f32_16x16x32_f16 v[0:3], v[4:7], v[8:11], 0         // 000000000000: D3D40000 02021104
	s_nop 7                                                    // 000000000008: BF800007
	v_add_f32_e32 v0, v1, v2                                   // 00000000000C: 02000501
	v_mfma_f32_16x16x32_f16 v[0:3], v[4:7], v[8:11], 0         // 000000000010: D3D40000 02021104
	s_cbranch_scc1 1                                           // 000000000018: BF850001 <f+0x20>
	s_nop 7                                                    // 00000000001C: BF800007
	v_mov_b32_e32 v5, v3                                       // 000000000020: 7E0A0303
	s_endpgm                                                   // 000000000024: BF810000
"""
    assert closest(text) == {("v_mfma_f32_16x16x32_f16", False): 8, ("v_mfma_f32_16x16x32_f16", True): 1}


def test_uses_past_a_branch_wait_as_long(tmp_path):
    if not OBJDUMP.exists():
        pytest.skip("no llvm-objdump")
    if not build.LIB.exists():
        build.build()
    lib = shutil.copy(build.LIB, tmp_path / "lib.so")
    subprocess.run([OBJDUMP, "--offloading", lib], check=True, capture_output=True, cwd=tmp_path)
    best = {}
    for obj in tmp_path.glob(f"lib.so.*{build.ARCH}"):
        listing = subprocess.run([OBJDUMP, "-d", obj], check=True, capture_output=True, text=True).stdout
        for key, waits in closest(listing).items():
            best[key] = min(waits, best.get(key, FURTHEST))
    assert ("v_mfma_f32_16x16x32_f16", True) in best  # there are such uses
    for (mfma, branched), waits in best.items():
        assert not branched or waits >= best[mfma, False], (mfma, waits, best)
