#!/usr/bin/env python3
"""Static check of matrix products written in inline asm: nothing may touch a product's sums before they are there.

hipcc puts the wait states between its own matrix instructions and whatever reads or overwrites their sums, but it does not see
that a statement of inline asm is one: a copy of the sums to other registers, which it may place anywhere behind the statement,
reads them too early, and a fence further down does not hold it back. This scans the device assembly of every kernel:

  * a register that an inline-asm v_mfma writes is pending for the wait states of an eight-pass product (the 16 x 16 x 32 bf16 form,
    the longest in use); an instruction is one, s_nop N is N + 1;
  * any instruction but another product's accumulation that reads or writes a pending register is a finding;
  * control flow: the state at a label joins the fall-through and every branch to it (back-edges from a first pass).

Usage: python tools/check_mfma_waits.py file.s   (exit status 1 if there is a finding)
"""
import re
import sys

WAIT_STATES = 11
_REGS = re.compile(r"\b([av])(?:\[(\d+):(\d+)\]|(\d+)\b)")


def regs(text):
    out = set()
    for kind, lo, hi, one in _REGS.findall(text):
        out |= {f"{kind}{one}"} if one else {f"{kind}{i}" for i in range(int(lo), int(hi) + 1)}
    return out


def scan(body):
    """Findings (line number, instruction, wait states missing) of one kernel's lines."""
    at_label, found = {}, {}

    def join(into, state):
        for r, n in state.items():
            into[r] = max(into.get(r, 0), n)

    def passed(state, n):
        return {r: left - n for r, left in state.items() if left > n}

    for _ in range(2):
        state, in_asm = {}, False
        for i, line in enumerate(body):
            s = line.strip()
            if s.startswith(";;#ASMSTART") or s.startswith(";;#ASMEND"):
                in_asm = s.startswith(";;#ASMSTART")
                continue
            s = s.split(";")[0].strip()
            if s.endswith(":"):
                join(state, at_label.get(s[:-1], {}))
                continue
            if not s or s.startswith("."):
                continue
            op, _, args = s.partition(" ")
            if op.startswith("v_mfma"):
                dst, a, b = [x.strip() for x in re.split(r",\s*(?![^\[]*\])", args)][:3]
                touched = regs(a) | regs(b)
            else:
                touched = regs(args)
            missing = max((state.get(r, 0) for r in touched), default=0)
            if missing:
                found[i] = (i, s, missing)
            state = passed(state, int(args, 0) + 1 if op == "s_nop" else 1)
            if op.startswith("v_mfma") and in_asm:
                state.update(dict.fromkeys(regs(dst), WAIT_STATES))
            elif op.startswith("s_cbranch") or op == "s_branch":
                join(at_label.setdefault(args.strip(), {}), state)
            if op in ("s_branch", "s_endpgm"):
                state = {}
    return [found[i] for i in sorted(found)]


def check(text):
    """(kernel, line, instruction, missing wait states) of every finding in a device assembly file."""
    out = []
    for km in re.finditer(r"^(_Z\S+):", text, re.M):
        end = text.find(".Lfunc_end", km.end())
        if end >= 0:
            out += [(km.group(1), *f) for f in scan(text[km.end():end].split("\n"))]
    return out


if __name__ == "__main__":
    n = 0
    for path in sys.argv[1:]:
        for name, i, s, missing in check(open(path).read()):
            n += 1
            print(f"{name[:90]}: line {i}: '{s}' {missing} wait states before a product's sums are there")
    print(f"{n} finding(s)")
    sys.exit(1 if n else 0)
