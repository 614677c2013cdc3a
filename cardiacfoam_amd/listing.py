"""Check of the compiler's device listings for register copies under the wrong lanes.

Where divergent lanes join, the kernel restores its execution mask (``s_or_b64 exec, exec,
..``).  With many scalar spills at such a place this compiler (ROCm 7.2, gfx950) can put a
vector register's spill or copy ahead of the restore: the lanes that skipped the branch do
not write the register, and a later read finds what an earlier kernel left in it.  Results
then depend on what ran before.  Seen in the FP64 ionic kernels: ORd's four-wave batch
kernel (release gates that stayed at 0, different from run to run), the RKF45 kernels of
Gaur (not finite) and the RKF45 batch kernels of TNNP, Courtemanche,
PerisYague, Grandi and ToRORd.  The flags in build.py leave none; the build looks every
listing over, so that another compiler or source cannot bring them back unseen.  A register
that some other write reaches is not reported, so the check finds reads of what an earlier
kernel left, not every misplaced copy.

masked_reads(path): per kernel the reads of a vector register that no other write reaches
than such copies.
"""
import re

_REG = re.compile(r"\b([va])(\d+)\b|\b([va])\[(\d+):(\d+)\]")
_RESTORE = re.compile(r"s_or_b64 exec, exec, ")
_LABEL = re.compile(r"^(\.LBB\w+):")
_BLOCK = re.compile(r"^; %bb\.\d+:")
_COPY = ("v_accvgpr", "v_mov_b", "scratch_load")
_ENDS = ("s_cbranch", "s_branch", "s_endpgm", "s_setpc")
_FAR = re.compile(r"\((\.LBB\w+)-\.Lpost_getpc")       # a branch beyond the offset's range
_NO_RESULT = ("s_", "ds_write", "ds_add", "global_store", "scratch_store", "flat_store",
              "buffer_store")
_SCALAR_RESULT = ("v_cmp", "v_readlane", "v_readfirstlane")


def _regs(text):
    out = []
    for m in _REG.finditer(text):
        if m.group(1):
            out.append(m.group(1) + m.group(2))
        else:
            out += [m.group(3) + str(k) for k in range(int(m.group(4)), int(m.group(5)) + 1)]
    return out


def _writes_reads(inst):
    op, _, rest = inst.partition(" ")
    ops = rest.split(",")
    if op.startswith("v_writelane"):        # a scalar's spill: one lane, whatever the mask
        return [], []
    if op.startswith(_NO_RESULT):
        return [], _regs(rest)
    if op.startswith(_SCALAR_RESULT):
        return [], _regs(",".join(ops[1:]))
    w, r = _regs(ops[0]), _regs(",".join(ops[1:]))
    if op.startswith(("v_fmac", "v_mac")):
        r = r + w
    if op.startswith("v_swap"):
        w = w + _regs(ops[1])
    return w, r


def _blocks(lines):
    blocks, labels, cur = [], {}, []
    for no, line in lines:
        m = _LABEL.match(line)
        if m or _BLOCK.match(line):
            if cur:
                blocks.append(cur)
                cur = []
            if m:
                labels[m.group(1)] = len(blocks)
            continue
        inst = " ".join(line.split(";")[0].split())
        if not inst or inst.startswith("."):
            continue
        cur.append((no, inst))
        if inst.startswith(_ENDS):
            blocks.append(cur)
            cur = []
    if cur:
        blocks.append(cur)
    succ = []
    for b, insts in enumerate(blocks):
        last, to = insts[-1][1], []
        m = re.match(r"s_c?branch\w* (\.LBB\w+)", last)
        if last.startswith("s_setpc"):
            m = next(filter(None, (_FAR.search(t) for _, t in reversed(insts))), None)
        if m and m.group(1) in labels and labels[m.group(1)] < len(blocks):
            to.append(labels[m.group(1)])
        if not last.startswith(("s_branch", "s_endpgm", "s_setpc")) and b + 1 < len(blocks):
            to.append(b + 1)
        succ.append(to)
    return blocks, succ


def _kernel(lines):
    blocks, succ = _blocks(lines)
    rows, suspects = [], 0
    for b, insts in enumerate(blocks):
        # copies ahead of the mask's restore, unless the block is the branch's own body
        restore = next((j for j, (_, t) in enumerate(insts) if _RESTORE.match(t)), -1)
        if b and blocks[b - 1][-1][1].startswith("s_cbranch_execz"):
            restore = -1
        row = []
        for j, (no, t) in enumerate(insts):
            w, r = _writes_reads(t)
            bad = j < restore and t.startswith(_COPY) and bool(w)
            suspects += bad
            row.append((no, t, w, r, bad))
        rows.append((restore, row))
    if not suspects:
        return []
    last_write = []
    for _, row in rows:
        kept = {}
        for _, _, w, _, bad in row:
            kept.update((q, bad) for q in w)
        last_write.append((frozenset(q for q, x in kept.items() if not x),
                           frozenset(q for q, x in kept.items() if x), frozenset(kept)))
    reach = [None] * len(rows)          # (registers a plain write reaches, a suspect one)
    reach[0], work = (frozenset(), frozenset()), [0]
    while work:
        b = work.pop()
        plain, bad, both = last_write[b]
        out = ((reach[b][0] - both) | plain, (reach[b][1] - both) | bad)
        for s in succ[b]:
            new = out if reach[s] is None else (reach[s][0] | out[0], reach[s][1] | out[1])
            if new != reach[s]:
                reach[s] = new
                work.append(s)
    found = []
    for b, (restore, row) in enumerate(rows):
        if reach[b] is None:
            continue
        plain, bad = set(reach[b][0]), set(reach[b][1])
        for j, (no, t, w, r, is_bad) in enumerate(row):
            found += [(q, no, t) for q in r if q in bad and q not in plain and j > restore]
            for q in w:
                (bad if is_bad else plain).add(q)
                (plain if is_bad else bad).discard(q)
    return found


def masked_reads(path):
    """{kernel: [(register, line, instruction), ...]} of the listing at path."""
    found, name, lines = {}, None, []
    with open(path) as f:
        for no, line in enumerate(f, 1):
            m = re.match(r"^(_Z\w+):", line)
            if m:
                name, lines = m.group(1), []
            elif line.startswith(".Lfunc_end"):
                hits = _kernel(lines) if name else []
                if hits:
                    found[name] = hits
                name = None
            elif name:
                lines.append((no, line))
    return found
