"""Hazard check of the generated gfx950 assembly for the hazards the compiler cannot resolve inside inline assembly.

The hand-written kernels issue memory instructions from inline assembly.  LLVM inserts the wait states the hardware
needs between dependent instructions for the instructions it generates itself, but it does not look inside an
assembly statement.  Two of those rules can be broken by code the compiler places *in front of* such a statement:

* a scalar register written by the vector ALU (``v_readlane_b32`` / ``v_readfirstlane_b32``: this is how spilled
  scalar registers come back) needs five wait states before a vector-memory instruction reads it as descriptor or
  offset -- otherwise the load goes out with the register's old value, i.e. to a wild address;
* ``M0`` written by the scalar ALU needs one wait state before a direct-to-LDS load uses it.

And the compiler does not know that such a load writes LDS, so it waits for none:

* no path through a kernel may end with a direct-to-LDS load that was never waited for: its data would land in LDS that by then
  holds something else, this workgroup's results or another workgroup's tiles.

``lint(path)`` returns the violations found in an assembly file (``hipcc -S --cuda-device-only``); the build fails
on any.
"""

from __future__ import annotations

import re
import sys

_VMEM = ("buffer_", "global_", "scratch_", "flat_", "tbuffer_")


def _instructions(path: str):
    out = []
    with open(path) as f:
        for n, line in enumerate(f, 1):
            t = line.strip()
            if not t or t[0] in ";." or t.endswith(":") or t.startswith(";;#"):
                continue
            out.append((n, t))
    return out


def _sregs(operands: str) -> set[int]:
    regs: set[int] = set()
    for m in re.finditer(r"\bs\[(\d+):(\d+)\]", operands):
        regs.update(range(int(m.group(1)), int(m.group(2)) + 1))
    for m in re.finditer(r"\bs(\d+)\b", operands):
        regs.add(int(m.group(1)))
    return regs


def _wait_states(text: str) -> int:
    m = re.match(r"s_nop (\d+)", text)
    return int(m.group(1)) + 1 if m else 1


def _blocks(path: str):
    """The kernels of an assembly file as basic blocks: per kernel {label: ([(line, text)], successors)}, the first block the entry."""
    kernels, label, nxt = [], None, 0
    with open(path) as f:
        for n, line in enumerate(f, 1):
            t = line.split(";", 1)[0].strip()
            m = re.match(r"([.\w$]+):$", t)
            if m and not m.group(1).startswith("."):
                kernels.append({})
                label = m.group(1)
                kernels[-1][label] = ([], [])
            elif not kernels or label is None:
                continue
            elif m:
                if not m.group(1).startswith(".LBB"):
                    label = None   # (.Lfunc_end and what follows: no code)
                    continue
                kernels[-1][label][1].append(m.group(1))
                label = m.group(1)
                kernels[-1][label] = ([], [])
            elif t and t[0] != ".":
                code, succ = kernels[-1][label]
                code.append((n, t))
                b = re.match(r"s_(c?)branch\w* +([.\w$]+)", t)
                if b:
                    succ.append(b.group(2))
                if b or t.startswith("s_endpgm"):
                    nxt += 1
                    here, label = kernels[-1], f"+{nxt}"
                    here[label] = ([], [])
                    if b and b.group(1):
                        succ.append(label)
    return kernels


def _open_loads(kernel) -> list[tuple[int, int]]:
    """(line of the s_endpgm, line of the load) of every end of a kernel that a direct-to-LDS load may still be open at.  Vector-memory
    operations complete in order, so a load with k of them behind it is over once at most k may be outstanding."""
    entry = next(iter(kernel))
    state = {entry: None}   # block -> (operations behind the last open direct-to-LDS load, its line); None: no such load
    work, ends = [entry], {}
    while work:
        name = work.pop()
        code, succ = kernel[name]
        open_ = state[name]
        for n, t in code:
            if t.startswith(_VMEM) and not t.startswith(("buffer_inv", "buffer_wb")):
                if t.endswith(" lds"):
                    open_ = (0, n)
                elif open_ is not None:
                    open_ = (min(open_[0] + 1, 64), open_[1])
            elif t.startswith("s_waitcnt"):
                m = re.search(r"vmcnt\((\d+)\)", t)
                if m and open_ is not None and int(m.group(1)) <= open_[0]:
                    open_ = None
            elif t.startswith("s_endpgm") and open_ is not None:
                ends[n] = open_[1]
        for to in succ:
            if to not in kernel:
                continue
            old = state.get(to, ())
            new = open_ if old == () or old is None else old if open_ is None else min(old, open_)
            if old == () or new != old:
                state[to] = new
                work.append(to)
    return sorted(ends.items())


def lint(path: str) -> list[str]:
    ins = _instructions(path)
    found = [f"{path}:{end}: the kernel ends with the direct-to-LDS load of line {load} never waited for"
             for kernel in _blocks(path) for end, load in _open_loads(kernel)]
    for idx, (n, t) in enumerate(ins):
        if not t.startswith(_VMEM):
            continue
        used = _sregs(t.split(None, 1)[1] if " " in t else "")
        waited = 0
        for k in range(idx - 1, max(idx - 8, -1), -1):
            pn, pt = ins[k]
            if waited >= 5:
                break
            d = re.match(r"v_read(?:first)?lane_b32 s(\d+)", pt)
            if d and int(d.group(1)) in used:
                found.append(f"{path}:{n}: `{t}` reads s{d.group(1)} {waited} wait states after `{pt}` (line {pn}); needs 5")
            waited += _wait_states(pt)
        if t.endswith(" lds") and idx > 0 and re.match(r"s_\w+ m0\b", ins[idx - 1][1]):
            found.append(f"{path}:{n}: `{t}` directly behind `{ins[idx - 1][1]}`; M0 needs one wait state")
    return found


if __name__ == "__main__":
    bad = [v for p in sys.argv[1:] for v in lint(p)]
    print("\n".join(bad) if bad else "no hazards found")
    sys.exit(1 if bad else 0)
