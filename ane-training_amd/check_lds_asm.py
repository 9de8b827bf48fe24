"""Build check of k_gemm.hip's inline LDS reads (run by `make check`).

The tiled GEMM issues its fragment reads (ds_read_b128) as inline assembly and
waits for them with a separate `s_waitcnt lgkmcnt(0)` statement that names the
destination registers as in/out operands.  The compiler cannot see that a read
is still in flight between the two statements; this script scans the device
assembly of every k_gemm_tile instantiation and fails if any instruction
reads or writes the destination register of an LDS read that no wait has
retired yet: lgkmcnt(0) retires every read, and the compiler's own
lgkmcnt(n) retires all but the n youngest LDS operations when no scalar load
is in flight (LDS operations complete in order).  Reads in flight are followed
along the branches, not in text order: the compiler places blocks of the
epilogue between blocks of the main loop.

    python3 check_lds_asm.py k_gemm.s
"""
import re
import sys


def regset(tok):
    m = re.match(r"([va])\[(\d+):(\d+)\]", tok)
    if m:
        return {f"{m.group(1)}{i}" for i in range(int(m.group(2)), int(m.group(3)) + 1)}
    m = re.match(r"([va])(\d+)$", tok)
    return {tok} if m else set()


YOUNGEST = 64      # operations whose order is kept: a wait names at most 63 of them
NOTHING = ((frozenset(), False), ())

def blocks_of(body):
    """Basic blocks [(label, [instructions])] in text order."""
    out = [(None, [])]
    for ln in body.split("\n"):
        t = ln.split(";")[0].strip()
        m = re.match(r"(\.LBB\w+):", t)
        if m:
            out.append((m.group(1), []))
            continue
        if not t or t.startswith(".") or t.endswith(":"):
            continue
        out[-1][1].append(t)
        if re.match(r"s_c?branch|s_endpgm|s_setpc", t):
            out.append((None, []))
    return out


def run_block(instrs, state, report):
    """The lgkm operations in flight after the block: ((destination registers of
    the older ones, whether a scalar load is among them), the youngest ones in
    order, oldest first, each (destination registers, is scalar memory)).  LDS
    operations complete in order, so a wait lgkmcnt(n) retires all but the n
    youngest: the order of those older than any n is not needed, only what they
    still have to write.  Scalar loads complete out of order, so with one in
    flight only lgkmcnt(0) retires anything."""
    (old, old_scalar), young = state
    young = list(young)
    for t in instrs:
        ops = [x for x in re.split(r"[ ,]+", t) if x]
        lds, scalar = ops[0].startswith("ds_"), ops[0].startswith(("s_load", "s_buffer_load"))
        returns = ops[0].startswith(("ds_read", "ds_bpermute", "ds_permute", "ds_swizzle"))
        pending = old.union(*(d for d, _ in young))
        if pending:
            used = set()
            for o in ops[2 if returns else 1:]:   # (a later read of the same register lands later)
                used |= regset(o)
            if used & pending:
                report(t)
        if lds or scalar:
            dst = regset(ops[1]) if returns else set()
            young.append((frozenset(dst), scalar))
            if len(young) > YOUNGEST:
                d, sc = young.pop(0)
                old, old_scalar = old | d, old_scalar or sc
            continue
        if ops[0] == "s_waitcnt":
            m = re.search(r"lgkmcnt\((\d+)\)", t)
            n = int(m.group(1)) if m else YOUNGEST
            if n == 0:
                old, old_scalar, young = frozenset(), False, []
            elif n < YOUNGEST and not old_scalar and not any(sc for _, sc in young):
                old = frozenset()
                young = young[-n:]
    return (old, old_scalar), tuple(young)


def check(asm_text):
    bad = []
    names = re.findall(r"^(_Z11k_gemm_tile\S*):", asm_text, re.M)
    for name in names:
        a = asm_text.index(name + ":") + len(name) + 1
        b = asm_text.index(".Lfunc_end", a)
        blocks = blocks_of(asm_text[a:b])
        at = {lab: i for i, (lab, _) in enumerate(blocks) if lab}
        seen = [set() for _ in blocks]
        found = set()
        work = [(0, NOTHING)]
        while work:
            i, state = work.pop()
            if state in seen[i]:
                continue
            seen[i].add(state)
            instrs = blocks[i][1]
            after = run_block(instrs, state, lambda t, i=i: found.add((i, t)))
            last = instrs[-1] if instrs else ""
            m = re.match(r"s_c?branch\w*\s+(\.LBB\w+)", last)
            if m:
                work.append((at[m.group(1)], after))
            if not re.match(r"s_branch|s_endpgm|s_setpc", last) and i + 1 < len(blocks):
                work.append((i + 1, after))
        bad += [(name, t) for _, t in sorted(found)]
    return names, bad


def main():
    names, bad = check(open(sys.argv[1]).read())
    if not names:
        print("check_lds_asm: no k_gemm_tile functions found", file=sys.stderr)
        return 1
    for name, t in bad:
        print(f"check_lds_asm: {name}: pending LDS read register used by: {t}", file=sys.stderr)
    if bad:
        return 1
    print(f"check_lds_asm: {len(names)} tile kernels, no use of a pending LDS read")
    return 0


if __name__ == "__main__":
    sys.exit(main())
