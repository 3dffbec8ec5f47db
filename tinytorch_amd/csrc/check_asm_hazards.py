#!/usr/bin/env python3
"""Scans the compiler's assembly listing of a kernel source for hazards that its asm statements can create.

    python3 check_asm_hazards.py file.s [file.s ...]      (exit status 1 if anything is found)

On gfx9-family chips a scalar register written by a vector instruction (v_readlane of a spilled scalar register,
v_readfirstlane, a compare with a scalar destination) may be read as the address of a vector-memory instruction only
five wait states later.  The compiler inserts the wait states itself for its own instructions, but its hazard pass does
not look into asm statements: a `global_load ... , s[n:n+1]` at the start of a statement, right behind the restore of
s[n:n+1], reads the old value.  The direct global->LDS loads and the Q loads of the kernels here are such statements;
they carry `s_nop`s of their own, and this check holds every listing to it.

Two passes over a listing:
  1. forward from every vector instruction that writes scalar registers: a vector-memory instruction (asm-issued or
     not) that reads one of them within five wait states is reported;
  2. every instruction between the compiler's `;;#ASMSTART` / `;;#ASMEND` markers is classified.  A vector-memory
     instruction with a scalar base must have five wait states of instructions behind it that provably do not write its
     base (a label, a branch or the start of the function inside that window ends the proof: reported).  A scalar-memory
     instruction, or a mnemonic this script does not know, is reported as unclassified: nothing asm-issued passes
     because a pattern failed to match it.

The instruction streams also leave LDS reads in flight behind a statement's end: the next statement's first operands.  The compiler takes their
registers for written; whatever it puts between the statements (a tile's requests, spills, copies) must leave them alone until a wait
has covered them.  The third pass follows every path through a function with the asm-issued LDS reads that may still be in flight, each with the
number of LDS operations issued after it at least: `s_waitcnt lgkmcnt(n)` ends those with n or more (the LDS answers in order; scalar loads, which
do not, are not counted).  Any instruction, the compiler's or a statement's own, that names a register in flight is reported.  In such
functions, whose barriers do not wait for the LDS, so is a barrier that a read of the compiler's own may still be on the way at: behind it other
wavefronts send for what takes that place.
"""
import re
import sys

VMEM = ("global_", "buffer_", "flat_", "scratch_", "tbuffer_")
# what an asm statement may hold besides vector-memory instructions: vector ALU / matrix, LDS, scalar ALU and control
PLAIN = ("v_", "ds_", "s_")
SMEM = ("s_load", "s_buffer_load", "s_store", "s_buffer_store", "s_scratch_", "s_atomic", "s_buffer_atomic", "s_dcache")
WAIT_STATES = 5


def sregs(text):
    out = set()
    for m in re.finditer(r"\bs(\d+)\b|\bs\[(\d+):(\d+)\]", text):
        if m.group(1):
            out.add(int(m.group(1)))
        else:
            out.update(range(int(m.group(2)), int(m.group(3)) + 1))
    return out


def operands(ins):
    return ins.split(None, 1)[1] if " " in ins else ""


def scalar_dests(ins):
    """Scalar registers a vector instruction writes (none for anything else)."""
    if not ins.startswith("v_"):
        return set()
    ops = [o.strip() for o in operands(ins).split(",")]
    dst = sregs(ops[0]) if ops else set()
    if "_co_" in ins and len(ops) > 1:  # carry-out in the second operand
        dst |= sregs(ops[1])
    return dst


def cost(ins):
    return int(ins.split()[1]) + 1 if ins.startswith("s_nop") else 1


def parse(path):
    """-> list of (line number, text, issued by an asm statement); labels are kept as text ending in ':'."""
    ins, in_asm = [], False
    for i, line in enumerate(open(path).read().split("\n")):
        if "#ASMSTART" in line:
            in_asm = True
            continue
        if "#ASMEND" in line:
            in_asm = False
            continue
        t = line.split(";")[0].strip()
        if not t or t.startswith(".") and not t.endswith(":"):
            continue
        ins.append((i + 1, t, in_asm))
    return ins


def scan(path):
    ins = parse(path)
    found = []
    # pass 1: forward from scalar writes by vector instructions
    for k, (i, t, _) in enumerate(ins):
        dst = scalar_dests(t)
        if not dst:
            continue
        waited = 0
        for j, u, _ in ins[k + 1:k + 12]:
            if u.endswith(":"):
                continue
            if u.startswith(VMEM) and waited < WAIT_STATES and sregs(operands(u)) & dst:
                found.append("%s:%d: %s  ->  line %d: %s  (%d wait states)" % (path, i, t, j, u, waited))
            waited += cost(u)
            if waited >= WAIT_STATES:
                break
    # pass 2: everything an asm statement issues
    for k, (i, t, in_asm) in enumerate(ins):
        if not in_asm or t.endswith(":"):
            continue
        if t.startswith(SMEM):
            found.append("%s:%d: %s  (asm-issued scalar-memory instruction: unclassified)" % (path, i, t))
            continue
        if t.startswith(VMEM):
            base = sregs(operands(t))
            if not base:
                continue
            waited, proven = 0, False
            for j, u, _ in reversed(ins[max(0, k - 16):k]):
                if u.endswith(":") or u.startswith(("s_cbranch", "s_branch", "s_setpc", "s_swappc", "s_endpgm")):
                    break  # other paths may lead here: nothing is known about what ran before
                if scalar_dests(u) & base:
                    break
                waited += cost(u)
                if waited >= WAIT_STATES:
                    proven = True
                    break
            if not proven:
                found.append("%s:%d: %s  (scalar base %s: only %d wait states provably free of a vector write)"
                             % (path, i, t, sorted(base), waited))
            continue
        if not t.startswith(PLAIN):
            found.append("%s:%d: %s  (asm-issued instruction this check cannot classify)" % (path, i, t))
    return found


def vregs(text):
    out = set()
    for m in re.finditer(r"\b([va])(\d+)\b|\b([va])\[(\d+):(\d+)\]", text):
        if m.group(1):
            out.add(m.group(1) + m.group(2))
        else:
            out.update(m.group(3) + str(r) for r in range(int(m.group(4)), int(m.group(5)) + 1))
    return out


ENDS = ("s_endpgm", "s_setpc", "s_trap")


class Block:
    def __init__(self):
        self.ins, self.next, self.state = [], [], None


def function_blocks(lines):
    """Basic blocks of one function: lines of (number, text, issued by an asm statement), `.subsection` directives among them.  Code of
    subsection 1 is out of line: what stands before it goes on behind it."""
    main, aside, at = [], [], None
    for ln in lines:
        if ln[1].startswith(".subsection"):
            at = ln[1].split()[1] != "0"
        else:
            (aside if at else main).append(ln)
    blocks, labels = [], {}
    for part in (main, aside):
        cur = Block()
        blocks.append(cur)
        for n, t, a in part:
            if t.endswith(":"):
                new = Block()
                cur.next.append(new)
                cur = new
                blocks.append(cur)
                labels.setdefault(t[:-1], []).append((n, cur))
                continue
            cur.ins.append((n, t, a))
            if t.startswith(("s_cbranch", "s_branch")):
                cur.target = (n, t.split()[-1])
                new = Block()
                if t.startswith("s_cbranch"):
                    cur.next.append(new)
                cur = new
                blocks.append(cur)
            elif t.startswith(ENDS):
                cur = Block()
                blocks.append(cur)
    for b in blocks:
        if hasattr(b, "target"):
            n, name = b.target
            if re.fullmatch(r"\d+[fb]", name):  # a local label: the nearest one that way
                at = [x for x in labels[name[:-1]] if (x[0] > n) == (name[-1] == "f")]
                b.next.append(min(at, key=lambda x: abs(x[0] - n))[1])
            else:
                b.next.append(labels[name][0][1])
    return blocks


def step(state, n, t, asm, report):
    """state: register -> (LDS operations behind its read at least, read issued by an asm statement)."""
    name = t.split(None, 1)[0]
    if report is not None and state:
        touched = sorted(r for r in vregs(operands(t)) & state.keys() if state[r][1])
        if touched:
            report[n] = "%s  (%s may still be on the way from the LDS)" % (t, ", ".join(touched))
        if name == "s_barrier" and not all(by_asm for _, by_asm in state.values()):
            report[n] = "s_barrier  (reads of the compiler's may still be on the way from the LDS)"
    if name == "s_waitcnt":
        m = re.search(r"lgkmcnt\((\d+)\)", t)
        if m:
            state = {r: v for r, v in state.items() if v[0] < int(m.group(1))}
    elif name.startswith("ds_"):
        state = {r: (min(k + 1, 63), by_asm) for r, (k, by_asm) in state.items()}
        if name.startswith("ds_read"):
            state.update((r, (0, asm)) for r in vregs(operands(t).split(",")[0]))
    return state


def scan_in_flight(path):
    """Pass 3."""
    functions, cur, in_asm = [], [], False
    for i, line in enumerate(open(path).read().split("\n")):
        if "#ASMSTART" in line:
            in_asm = True
        elif "#ASMEND" in line:
            in_asm = False
        else:
            t = line.split(";")[0].strip()
            if t.startswith(".Lfunc_end"):
                functions.append(cur)
                cur = []
            elif t and (t.endswith(":") or not t.startswith(".") or t.startswith(".subsection")):
                cur.append((i + 1, t, in_asm))
    functions.append(cur)
    found = []
    for lines in functions:
        if not any(a and t.startswith("ds_read") for _, t, a in lines):
            continue
        blocks = function_blocks(lines)
        for b in blocks:
            b.state = {}
        todo = list(blocks)
        while todo:
            b = todo.pop()
            state = dict(b.state)
            for n, t, a in b.ins:
                state = step(state, n, t, a, None)
            for x in b.next:
                merged = dict(x.state)
                for r, (k, by_asm) in state.items():  # the worst of both ways here
                    other = merged.get(r, (64, by_asm))
                    merged[r] = (min(k, other[0]), by_asm or other[1])
                if merged != x.state:
                    x.state = merged
                    todo.append(x)
        report, streams = {}, False
        for b in blocks:
            state = dict(b.state)
            for n, t, a in b.ins:
                streams |= not a and any(by_asm for _, by_asm in state.values())
                state = step(state, n, t, a, report)
        if not streams:
            report = {n: r for n, r in report.items() if not r.startswith("s_barrier")}
        found += ["%s:%d: %s" % (path, n, r) for n, r in sorted(report.items())]
    return found


def main():
    found = []
    for path in sys.argv[1:]:
        found += scan(path) + scan_in_flight(path)
    for f in found:
        print(f)
    print("%d finding(s)" % len(found))
    return 1 if found else 0


if __name__ == "__main__":
    sys.exit(main())
