"""Wait states around the LDS copies written in inline assembly, read from the built library.

The compiler's hazard pass does not look into an asm string, so what gfx950 wants before a
buffer_load .. lds has to be there by construction: one wait state after a scalar write of M0 (the
copy's LDS address), five after a VALU write of a scalar register that the copy reads (its
descriptor or its offset; a spilled one comes back by v_readlane)."""
from __future__ import annotations

import os
import re
import shutil
import subprocess

import pytest

from tinyserve_amd import _lib

OBJDUMP = next((p for p in (shutil.which("llvm-objdump"), "/opt/rocm/lib/llvm/bin/llvm-objdump") if p and os.path.exists(p)),
               None)
INS = re.compile(r"^\t(\S+)\s*(.*?)\s*// ([0-9A-F]+):(.*)$")
FUNC = re.compile(r"^[0-9a-f]+ <(.*)>:$")


def _sregs(text: str) -> set[int]:
    out = {int(x) for x in re.findall(r"\bs(\d+)\b", text)}
    for a, b in re.findall(r"\bs\[(\d+):(\d+)\]", text):
        out |= set(range(int(a), int(b) + 1))
    return out


def _valu_sdst(op: str, args: list[str]) -> set[int]:
    """Scalar registers a vector instruction writes."""
    if op.startswith(("v_readfirstlane", "v_readlane", "v_cmp")):
        return _sregs(args[0])
    if re.match(r"v_(add|sub|subrev|addc|subb|subbrev)_co|v_div_scale|v_mad_[ui]64", op):
        return _sregs(args[1])
    return set()


def find_hazards(asm: str) -> tuple[int, list[str]]:
    """(copies seen, the copies with too few wait states) of a disassembly, every path of up to five
    instructions before each copy followed."""
    funcs: list[tuple[str, list]] = []
    for line in asm.splitlines():
        if m := FUNC.match(line):
            funcs.append((m[1], []))
        elif funcs and (m := INS.match(line)):
            funcs[-1][1].append((int(m[3], 16), m[1], m[2].split(","), m[4]))
    copies, bad = 0, []
    for name, ins in funcs:
        at = {i[0]: n for n, i in enumerate(ins)}
        before: list[list[int]] = [[] for _ in ins]
        for n, (_, op, _, tail) in enumerate(ins):
            if op not in ("s_branch", "s_endpgm", "s_setpc_b64") and n + 1 < len(ins):
                before[n + 1].append(n)
            if op.startswith(("s_branch", "s_cbranch")) and (m := re.search(r"<.*\+0x([0-9a-f]+)>", tail)):
                before[at[ins[0][0] + int(m[1], 16)]].append(n)
        for n, (_, op, args, _) in enumerate(ins):
            if not op.startswith("buffer_load") or not re.search(r"\blds\b", args[-1]):
                continue
            copies += 1
            reads, todo, seen = _sregs(",".join(args)), [(p, 0) for p in before[n]], set()
            while todo:
                p, waited = todo.pop()
                if waited >= 5 or (p, waited) in seen:
                    continue
                seen.add((p, waited))
                _, pop, pargs, _ = ins[p]
                if waited < 1 and pop.startswith("s_") and pargs[0].strip() == "m0":
                    bad.append(f"{name}: M0 written by {pop} right before {op}")
                if pop.startswith("v_") and _valu_sdst(pop, pargs) & reads:
                    bad.append(f"{name}: {pop} {','.join(pargs)} {waited} wait states before {op} {','.join(args)}")
                states = int(pargs[0], 0) + 1 if pop == "s_nop" else 1
                todo += [(q, waited + states) for q in before[p]]
    return copies, bad


def _dis(*body: str) -> str:
    return "0000000000001000 <f>:\n" + "".join(f"\t{l:<60}// {0x1000 + 4 * i:012X}: 00000000\n" for i, l in enumerate(body))


COPY = "buffer_load_dwordx4 v1, s[8:11], s5 offen lds"


@pytest.mark.parametrize("body,ok", [
    (("s_mov_b32 m0, s3", COPY), False),
    (("s_mov_b32 m0, s3", "s_nop 0", COPY), True),
    (("v_readlane_b32 s5, v2, 1", "s_add_u32 m0, s3, s4", "s_nop 0", COPY), False),
    (("v_readlane_b32 s5, v2, 1", "s_add_u32 m0, s3, s4", "s_nop 3", COPY), True),
    (("v_readfirstlane_b32 s9, v2", "s_mov_b32 m0, s3", "s_nop 2", COPY), False),
    (("v_readlane_b32 s6, v2, 1", "s_add_u32 m0, s3, s4", "s_nop 0", COPY), True),
])
def test_finder(body, ok):
    copies, bad = find_hazards(_dis(*body))
    assert copies == 1 and (not bad) == ok


def test_lds_copies_wait(tmp_path):
    if OBJDUMP is None or not os.path.exists(_lib.LIB_PATH):
        pytest.skip("needs llvm-objdump and the built library")
    lib = shutil.copy(_lib.LIB_PATH, tmp_path / "lib.so")
    subprocess.run([OBJDUMP, "--offloading", "lib.so"], cwd=tmp_path, check=True, capture_output=True)
    objs = sorted(p for p in os.listdir(tmp_path) if "gfx950" in p)
    assert objs, f"no gfx950 code in {lib}"
    copies, bad = 0, []
    for o in objs:
        asm = subprocess.run([OBJDUMP, "-d", o], cwd=tmp_path, check=True, capture_output=True, text=True).stdout
        n, b = find_hazards(asm)
        copies, bad = copies + n, bad + b
    assert copies > 0 and not bad, f"{len(bad)} of {copies} copies: " + "; ".join(sorted(set(bad))[:8])
