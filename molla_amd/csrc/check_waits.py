"""Checks the gfx950 assembly of prefill.hip: every direct load to LDS
(global_load_lds, issued by inline assembly that the compiler does not count)
has landed before the barrier after which other waves read it.

    python3 check_waits.py FILE.s

Loads return in order, so an LDS load has landed at an `s_waitcnt vmcnt(N)` if
at most N loads were issued after it.  Between an LDS load and the next
s_barrier there has to be a wait whose N is at most the number of loads that
lie between the two, counted in the order of the emitted code: a compiler that
moves a load ahead of the LDS load, or merges two into one, ends up with too few
and the check fails.  Only global and buffer loads count as younger ones.  A
label or a branch in between fails too: the order of the lines is then not the
order of execution.

m0 holds an LDS load's address, and the compiler does not know that the assembly
writes it: it may appear only where a load sets it, with nothing but an s_nop
before the load.
"""

import re
import sys

LDS_LOAD = re.compile(r"(global|buffer)_load_lds_|(global|buffer)_load_\S+\s.*\blds\b")
LOAD = re.compile(r"(global|buffer)_load_")
M0 = re.compile(r"\bm0\b")
VMCNT = re.compile(r"vmcnt\((\d+)\)")


def check(lines):
    """(LDS loads seen, messages about what is wrong)."""
    m0 = None  # the line that set m0 for the next LDS load
    pending = []  # [line number, younger loads] of LDS loads not known to have landed
    seen, bad = 0, []

    def fail(at, why):
        bad.extend(f"line {at}: {why} before the LDS load of line {line} has landed" for line, _ in pending)
        pending.clear()

    for at, raw in enumerate(lines, 1):
        text = raw.split(";")[0].strip()
        if not text or text.startswith("."):
            if re.match(r"\.L\w+:", text):  # (a label that is jumped to)
                fail(at, "a label")
            continue
        if M0.search(text):
            if not text.startswith("s_mov_b32 m0,") or m0 is not None:
                bad.append(f"line {at}: m0 used by other code")
            m0 = at
            continue
        if m0 is not None and not text.startswith("s_nop"):
            if not LDS_LOAD.match(text):
                bad.append(f"line {m0}: m0 set, and no LDS load after it")
            m0 = None
        elif LDS_LOAD.match(text):
            bad.append(f"line {at}: an LDS load whose m0 was not set")
        if LDS_LOAD.match(text):
            for p in pending:
                p[1] += 1
            pending.append([at, 0])
            seen += 1
        elif LOAD.match(text):
            for p in pending:
                p[1] += 1
        elif text.startswith("s_waitcnt"):
            found = VMCNT.search(text)
            if found:
                pending[:] = [p for p in pending if p[1] < int(found.group(1))]
            elif "lgkmcnt" not in text and "expcnt" not in text:  # (a bare count)
                fail(at, "a wait that is not understood")
        elif text.startswith("s_barrier"):
            fail(at, "a barrier")
        elif text.startswith(("s_cbranch", "s_branch", "s_setpc", "s_endpgm")):
            fail(at, "a branch")
    fail(len(lines), "the end")
    return seen, bad


def main(path):
    with open(path) as f:
        seen, bad = check(f.read().splitlines())
    for b in bad:
        print(f"{path}: {b}", file=sys.stderr)
    if not seen:
        print(f"{path}: no LDS load found", file=sys.stderr)
    return 1 if bad or not seen else 0


if __name__ == "__main__":
    sys.exit(main(sys.argv[1]))
