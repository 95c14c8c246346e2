#!/usr/bin/env python3
"""Checks the gfx950 assembly of the kernels for what the compiler cannot check: two hazards of the inline-assembly dot
products, and the counted waits of the tile kernels.

The DPP dot products (v_dot2c_f32_f16_dpp ... row_newbcast) are written as inline assembly, so the compiler's hazard
recognizer does not know what they are.  Two rules of the target then rest on the source code alone:

  1. a VGPR written by a vector-ALU instruction may be read through DPP only two issue slots later;
  2. the result of a dot instruction may feed the accumulator of the same dot opcode at once, but any other
     instruction that reads it has to stay three issue slots behind.

The ring loop of the tile kernels (tile_gemm.hpp) copies activations straight into LDS and waits for them with counted
waits, which are right for one order of the vector-memory requests only:

  3. at the barrier in front of a stage's first read, every copy of that stage must have landed: a wait vmcnt(N) after the
     copy counts only if at least N requests were issued between the two.  The copies behind a barrier belong to the stage
     R - 1 ahead (R = stages of the ring, from the kernel's template arguments), so they are due R - 2 barriers later.
     Every barrier interval must hold the same number of copies: one that slipped over a barrier overwrites a stage in use.
  4. copies outside that loop (the first stages, the group sums) must be followed by vmcnt(0) before the next barrier;
  5. no register is spilled inside the loop: a reload from scratch stands behind a wait for every request in flight.

This script reads the device assembly the build keeps (one .s per source file) and fails on any of these patterns,
whichever way it came about (instruction scheduling, a register copy the allocator put in).  s_nop N counts as N + 1 slots.
Usage: lint_isa.py file.s [...]
"""
import re
import sys

DPP = re.compile(r"^(v_\w+_dpp)\s+(v\d+|v\[\d+:\d+\]),\s*(v\d+)")
DOT = re.compile(r"^(v_dot\w+)\s+(v\d+),")
VALU_DST = re.compile(r"^v_\w+\s+(v\d+|v\[(\d+):(\d+)\])")
REG = re.compile(r"\bv(\d+)\b|\bv\[(\d+):(\d+)\]")


def regs_of(text):
    out = set()
    for m in REG.finditer(text):
        if m.group(1) is not None:
            out.add(int(m.group(1)))
        else:
            out.update(range(int(m.group(2)), int(m.group(3)) + 1))
    return out


def written(line):
    m = VALU_DST.match(line)
    if not m or line.startswith("v_cmp") or line.startswith("v_readlane") or line.startswith("v_readfirstlane"):
        return set()
    return regs_of(m.group(1))


def lint(path):
    errors = []
    kernel = "?"
    window = []  # (slots_ago_base, line) of recent instructions, newest last
    for raw in open(path):
        line = raw.split(";")[0].strip()
        if line.endswith(":") and line.startswith("_Z"):
            kernel = line.rstrip(":")
            window = []
            continue
        if not line or line.startswith((".", "//")) or line.endswith(":"):
            continue
        nop = re.match(r"^s_nop\s+(\d+)", line)
        slots = int(nop.group(1)) + 1 if nop else 1
        # rule 1: the DPP source of this instruction against vector-ALU writes in the two slots before it
        m = DPP.match(line)
        if m:
            src = int(m.group(3)[1:])
            dist = 0
            for s_, prev in reversed(window):
                if dist >= 2:
                    break
                if src in written(prev):
                    errors.append(f"{path}: {kernel}: DPP source v{src} written {dist} slot(s) before: '{prev}' -> '{line}'")
                dist += s_
        # rule 2: readers of a dot result within three slots (the same opcode accumulating into it is exempt)
        dist = 0
        for s_, prev in reversed(window):
            if dist >= 3:
                break
            d = DOT.match(prev)
            if d:
                dst = int(d.group(2)[1:])
                mine = DOT.match(line)
                same_acc = mine and mine.group(1).replace("_dpp", "") == d.group(1).replace("_dpp", "") and int(mine.group(2)[1:]) == dst
                operands = line.split(None, 1)[1] if " " in line else ""
                reads = regs_of(operands.split(",", 1)[1]) if "," in operands and line.startswith("v_") else regs_of(operands)
                if same_acc:
                    reads = regs_of(",".join(operands.split(",")[1:])) - {dst} if dst not in regs_of(",".join(operands.split(",")[1:3])) else {dst}
                    if dst in reads:
                        errors.append(f"{path}: {kernel}: dot result v{dst} read as a source {dist} slot(s) later: '{prev}' -> '{line}'")
                elif dst in reads and not line.startswith("s_"):
                    errors.append(f"{path}: {kernel}: dot result v{dst} read {dist} slot(s) later: '{prev}' -> '{line}'")
            dist += s_
        window.append((slots, line))
        if len(window) > 8:
            window.pop(0)
    return errors


# ring stages R of a tile kernel: nint_tile_kernel<U, NW, MT, NB, R, GLU>, row_tile_kernel<KIND, NW, MT, NB, R>;
# moe_tile_kernel<GLU> and moe_tile_few_kernel<GLU> hold a ring loop for every size of chunk and profile, all of kMoeRing stages
TILE = re.compile(r"^_ZN3mfq1[569](?:nint_tile_kernelI.*ELi\d+ELi\d+ELi\d+ELi(\d+)ELb[01]E|row_tile_kernelILi\d+ELi\d+ELi\d+ELi\d+ELi(\d+)E"
                  r"|moe_tile_(?:few_)?kernelILb[01]E)E")
MOE_RING = 4
VMEM = re.compile(r"^(buffer|global|flat|scratch)_")
VMCNT = re.compile(r"^s_waitcnt\b.*\bvmcnt\((\d+)\)")
BRANCH = re.compile(r"^s_c?branch\w*\s+(\.LBB\w+)")


def tile_events(body):
    """(kind, value) of the instructions rules 3 and 4 are about: 'copy', 'req', ('wait', N), 'barrier', and 'mfma'."""
    out = []
    for line in body:
        w = VMCNT.match(line)
        if w:
            out.append(("wait", int(w.group(1))))
        elif VMEM.match(line):
            out.append(("copy" if line.endswith(" lds") else "req", 0))
        elif line.startswith("s_barrier"):
            out.append(("barrier", 0))
        elif line.startswith("v_mfma"):
            out.append(("mfma", 0))
    return out


def landed(events, copy, barrier):
    """Whether the copy at index `copy` is known to have landed at index `barrier`."""
    younger = 0
    for kind, n in events[copy + 1:barrier]:
        if kind in ("copy", "req"):
            younger += 1
        elif kind == "wait" and n <= younger:
            return True
    return False


def lint_ring(events, R):
    """Rule 3 on the events of one pass through the ring loop."""
    once = [i for i, e in enumerate(events) if e[0] == "barrier"]
    per = [sum(e[0] == "copy" for e in (events + events)[a:b])
           for a, b in zip(once, once[1:] + [len(events) + once[0]])]
    if len(set(per)) != 1 or per[0] == 0:
        return [f"copies per barrier interval {per}"]
    passes = -(-(R - 2) // len(once)) + 1
    ev = events * passes
    bar = [i for i, e in enumerate(ev) if e[0] == "barrier"]
    errors = []
    for k in range(len(bar) - len(once), len(bar)):
        lo, hi = bar[k - (R - 2)], bar[k - (R - 2) + 1]
        late = sum(ev[i][0] == "copy" and not landed(ev, i, bar[k]) for i in range(lo, hi))
        if late:
            errors.append(f"barrier {k - len(bar) + len(once) + 1} of {len(once)} of the ring loop: {late} of {per[0]} copies of the next stage may be in flight")
    return errors


def lint_tile(name, lines, R):
    at = {line[:-1]: i for i, line in enumerate(lines) if line.endswith(":")}
    loops = []
    for i, line in enumerate(lines):
        b = BRANCH.match(line)
        if b and at.get(b.group(1), len(lines)) < i:
            lo = at[b.group(1)]
            ev = tile_events(lines[lo:i])
            if any(e[0] == "copy" for e in ev) and any(e[0] == "barrier" for e in ev):
                loops.append((sum(e[0] == "mfma" for e in ev), lo, i, ev))
    if not loops:
        return ["no ring loop found"]
    # innermost ones: a block moved out of line jumps back over whatever lies in between
    inner = [a for a in loops if not any(a[1] <= b[1] and b[2] <= a[2] and a is not b for b in loops)]
    # the loops over group sums wait for their copies on the spot; what does not is a ring
    rings = [a for a in inner if lint_outside(a[3])]
    if not rings:
        return ["no ring loop found"]
    errors, rest, at = [], [], 0
    for _, lo, hi, ev in sorted(rings, key=lambda a: a[1]):
        errors += lint_ring(ev, R)
        spilled = sum(line.startswith("scratch_") for line in lines[lo:hi])
        if spilled:
            errors.append(f"{spilled} scratch accesses in a ring loop")  # rule 5
        rest += tile_events(lines[at:lo]) + [("barrier", 0)]
        at = hi
    return errors + lint_outside(rest + tile_events(lines[at:]))


def lint_outside(events):
    """Rule 4: a copy outside a ring loop and the next barrier (of the next pass, at the end of a loop)."""
    errors = []
    for i, e in enumerate(events):
        if e[0] == "copy":
            nxt = next((j for j in range(i, len(events)) if events[j][0] == "barrier"), len(events))
            if ("wait", 0) not in events[i:nxt]:
                errors.append("a copy outside the ring loop reaches a barrier without vmcnt(0)")
    return errors


def lint_tiles(path):
    """(errors, tile kernels seen)"""
    errors, seen, name, R, lines = [], 0, None, 0, []
    for raw in open(path):
        line = raw.split(";")[0].strip()
        if line.startswith("_Z") and line.endswith(":"):
            m = TILE.match(line)
            if not m and any(k in line for k in ("nint_tile_kernelI", "row_tile_kernelI", "moe_tile_kernelI", "moe_tile_few_kernelI")):
                errors.append(f"{path}: {line} is a tile kernel of unknown template arguments")
            name, lines = (line[:-1], []) if m else (None, [])
            if m:
                R = int(m.group(1) or m.group(2) or MOE_RING)
        elif name and line.startswith(".Lfunc_end"):
            errors += [f"{path}: {name}: {e}" for e in lint_tile(name, lines, R)]
            seen, name = seen + 1, None
        elif name and line and (not line.startswith(".") or line.endswith(":")):
            lines.append(line)
    return errors, seen


def main():
    bad, tiles = [], 0
    for p in sys.argv[1:]:
        bad += lint(p)
        errors, seen = lint_tiles(p)
        bad += errors
        tiles += seen
    for e in bad[:40]:
        print(e)
    if bad:
        print(f"lint_isa: {len(bad)} hazard(s)")
        return 1
    print(f"lint_isa: {len(sys.argv) - 1} file(s) clean, {tiles} tile kernel(s) among them")
    return 0


if __name__ == "__main__":
    sys.exit(main())
