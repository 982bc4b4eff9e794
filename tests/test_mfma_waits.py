"""CPU: the asm MFMAs of gemm_quad.hip, as compiled into the built library.

The compiler does not see the latency of an MFMA written as inline asm: it may place a copy of an
accumulator (its own register moves, at loop exits for instance) right behind one.  A 16x16x32 bf16
MFMA needs 8 wait states before a VALU instruction or a store may read its result; here every such
read, on every path through every kernel, has to be preceded by 8 wait states that the source
guarantees -- s_nop and further MFMAs, whatever scalar code happens to stand in between.  The other
way round an MFMA reads an accumulator two wait states after a VALU instruction wrote it."""

import os
import re
import subprocess

import pytest

from helpers import ROOT

OBJDUMP = "/opt/rocm/llvm/bin/llvm-objdump"
WAITS, WRITE_WAITS = 8, 2
INSN = re.compile(r"^\t(\S+)\s*(.*?)\s*// ([0-9A-F]+):(.*)$")
SYMBOL = re.compile(r"^[0-9a-f]+ <(.+)>:$")
TARGET = re.compile(r"<[^>]*?(?:\+0x([0-9a-f]+))?>\s*$")
AREG = re.compile(r"\ba\[(\d+):(\d+)\]|\ba(\d+)\b")


def _acc(text):
    regs = []
    for lo, hi, one in AREG.findall(text):
        regs.extend(range(int(lo), int(hi) + 1) if lo else (int(one),))
    return regs


def kernels(library, tmp):
    """{kernel: [(address, mnemonic, operands, branch target or None)]} of the library's gfx950 code."""
    link = os.path.join(tmp, "lib.so")
    os.symlink(library, link)
    subprocess.run([OBJDUMP, "--offloading", link], check=True, capture_output=True, cwd=tmp)
    found = {}
    for f in sorted(os.listdir(tmp)):
        if "gfx950" not in f:
            continue
        p = subprocess.Popen([OBJDUMP, "-d", os.path.join(tmp, f)], stdout=subprocess.PIPE, text=True)
        name, code = None, []
        for line in p.stdout:
            m = SYMBOL.match(line)
            if m:
                name, code = m.group(1), []
                if "gemm_quad_kernel" in name:
                    found[name] = code
                continue
            m = INSN.match(line)
            if m and name in found:
                op, args, addr, tail = m.groups()
                t = TARGET.search(tail) if "branch" in op else None
                code.append((int(addr, 16), op, args, int(t.group(1) or "0", 16) if t else None))
        assert p.wait() == 0
    return found


def early_uses(code):
    """Reads of an accumulator less than WAITS guaranteed wait states behind the MFMA that wrote it,
    and MFMAs less than WRITE_WAITS instructions behind a register move into their accumulator: a
    forward pass over basic blocks, keeping per register the fewest of either."""
    base = code[0][0]
    index = {a - base: i for i, (a, *_) in enumerate(code)}
    leaders = {0}
    for i, (_, op, _, target) in enumerate(code):
        if target is not None:
            leaders.update((index[target], i + 1))
    entry, work, bad = {0: ({}, {})}, [0], set()

    def age(state, n, limit):
        return {r: w + n for r, w in state.items() if w + n < limit}

    while work:
        i = work.pop()
        mfma, moved = (dict(s) for s in entry[i])    # register -> wait states since
        while i < len(code):
            addr, op, args, target = code[i]
            n = int(args, 0) + 1 if op == "s_nop" else 1
            dst, _, src = args.partition(",")
            if op.startswith("v_mfma"):
                acc = _acc(src)                      # as its third source
                bad.update((hex(addr), op, args, moved[r]) for r in acc if r in moved)
                mfma, moved = age(mfma, 1, WAITS), age(moved, 1, WRITE_WAITS)
                for r in _acc(dst):
                    mfma[r] = 0
                    moved.pop(r, None)
            else:
                to_acc = op.startswith(("v_accvgpr_write", "v_accvgpr_mov"))
                loaded = op.startswith(("global_load", "ds_read"))
                reads = () if loaded else _acc(src if op.startswith("v_accvgpr") else args)
                bad.update((hex(addr), op, args, mfma[r]) for r in reads if r in mfma)
                if op == "s_nop":
                    mfma = age(mfma, n, WAITS)
                moved = age(moved, n, WRITE_WAITS)
                if to_acc or loaded:
                    for r in _acc(dst):
                        mfma.pop(r, None)
                        if to_acc:
                            moved[r] = 0
            ends = op in ("s_branch", "s_endpgm")
            nxt = [index[target]] if target is not None else []
            if i + 1 in leaders and not ends:
                nxt.append(i + 1)
            for j in nxt:
                old = entry.get(j, ({}, {}))
                new = tuple({r: min(a.get(r, WAITS), b.get(r, WAITS)) for r in a.keys() | b.keys()}
                            for a, b in zip(old, (mfma, moved)))
                if j not in entry or new != old:
                    entry[j] = new
                    work.append(j)
            if nxt or ends:
                break
            i += 1
    return sorted(bad)


@pytest.mark.skipif(not os.path.exists(OBJDUMP), reason="needs the ROCm binary utilities")
def test_accumulators_are_read_after_their_wait_states(tmp_path):
    from qdecode import _lib
    found = kernels(_lib.LIB_PATH, str(tmp_path))
    assert len(found) > 40, sorted(found)
    assert all(any(op.startswith("v_mfma") for _, op, _, _ in code) for code in found.values())
    bad = {name: b for name, code in found.items() if (b := early_uses(code))}
    assert not bad, {name: b[:3] for name, b in bad.items()}
