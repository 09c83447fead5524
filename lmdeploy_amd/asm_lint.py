"""Build-time check of the generated GCN assembly of the GEMM kernels.

The kernels issue global loads from inline assembly and wait for them by count (`s_waitcnt
vmcnt(N)`), so the compiler does not know when a load's destination registers become valid.  It
is free to copy or reuse such a register between the load and the wait - which reads a stale value
or, worse, lets the load land on an unrelated value such as an address.  This pass builds the
control-flow graph of every kernel, propagates "VGPR v is the destination of the p-th youngest
load in flight" to a fixed point (a wait for vmcnt(N) retires every load with p > N; where paths
join, the younger position wins), and reports any compiler-generated instruction that touches a
register whose load may still be in flight.

LDS reads issued from inline assembly (`ds_read_*`) are tracked the same way: they return in order, and a wait
for lgkmcnt(N) retires every one with N younger ones behind it.  (Whatever else counts there is not counted here,
which only keeps destinations in flight for longer.  A destination that nothing reads any
more is the dangerous one: the compiler hands the register to another value at once, and the
read lands on it later.)

MFMAs issued from inline assembly hide a third hazard: the hardware does not interlock a matrix
instruction's result against vector instructions, the compiler normally pads with s_nop, and it
cannot see into inline assembly.  Compiler-generated accumulator moves (`v_accvgpr_*`) must
therefore not follow an inline-assembly MFMA that writes the same AGPR within `_MFMA_SETTLE` wait
states, nor write an AGPR that an inline-assembly MFMA reads within the next two.

Lanes that exchange values through LDS need something between the writes and the reads that the compiler moves neither
across, also where they belong to one wave, which LDS serves in order: a barrier of the workgroup or of the wave.  No LDS read that the
compiler generates may follow an LDS write of its own without one.

Assembly that masks its loads and then sets EXEC to all ones, instead of what it found there, may only stand where every
lane is active: elsewhere it would switch lanes on in the middle of a branch that they did not take.  Kernels start with all
lanes (their workgroups are whole waves); from there the pass follows EXEC and the scalar registers that hold a copy of it.
"""
from __future__ import annotations

import re
from typing import Dict, List, Tuple

_LOAD = re.compile(r"^\s*global_load_(?:lds_)?dword(?:x2|x3|x4)?\s+v(?:\[(\d+):(\d+)\]|(\d+))\s*,")
_DSREAD = re.compile(r"^\s*ds_read\w*\s+v(?:\[(\d+):(\d+)\]|(\d+))\s*,")
_STORE = re.compile(r"^\s*global_(?:store|atomic)\w*\s")
_VMCNT = re.compile(r"vmcnt\((\d+)\)")
_LGKMCNT = re.compile(r"lgkmcnt\((\d+)\)")
_VREG = re.compile(r"\bv(?:\[(\d+):(\d+)\]|(\d+)\b)")
_FUNC = re.compile(r"^(_Z\w+):")
_LABEL = re.compile(r"^(\.LBB\w+):")
_BRANCH = re.compile(r"^\s*s_(c?branch)\w*\s+(\.LBB\w+)")


def _regs(m) -> range:
    if m.group(1) is not None:
        return range(int(m.group(1)), int(m.group(2)) + 1)
    return range(int(m.group(3)), int(m.group(3)) + 1)


class _Ins:
    __slots__ = ("kind", "regs", "n", "text", "line")

    def __init__(self, kind, regs, n, text, line):
        self.kind, self.regs, self.n, self.text, self.line = kind, regs, n, text, line


def _parse(lines: List[Tuple[int, str]]):
    """-> blocks: list of (label, [ins], successors-by-label, falls_through)"""
    blocks, cur, label, in_asm = [], [], "<entry>", False

    def close(succ, fall):
        nonlocal cur, label
        blocks.append([label, cur, succ, fall])
        cur, label = [], None

    for ln, raw in lines:
        s = raw.strip()
        if s.startswith(";;#ASMSTART"):
            in_asm = True
            continue
        if s.startswith(";;#ASMEND"):
            in_asm = False
            continue
        m = _LABEL.match(raw)
        if m:
            if label is not None:
                close([], True)
            label = m.group(1)
            continue
        code = raw.split(";")[0].strip()
        if not code or code.startswith("."):
            continue
        if label is None:
            label = "<anon%d>" % ln
        m = _BRANCH.match(code)
        if m:
            close([m.group(2)], m.group(1) == "cbranch")
            continue
        if code.startswith("s_endpgm"):
            close([], False)
            continue
        m = _LOAD.match(code)
        if m:
            regs = [] if "_lds_" in code else list(_regs(m))
            cur.append(_Ins("load", regs, 0, code, ln))
            continue
        if _STORE.match(code):
            cur.append(_Ins("load", [], 0, code, ln))  # stores count in vmcnt too: only makes waits conservative
            continue
        if in_asm:
            m = _DSREAD.match(code)
            if m:
                cur.append(_Ins("ldsread", list(_regs(m)), 0, code, ln))
                continue
        if code.startswith("s_waitcnt"):
            everything = re.match(r"s_waitcnt\s+(0|0x0)\s*$", code) is not None
            v = _VMCNT.search(code)
            if v is not None or everything:
                cur.append(_Ins("wait", [], 0 if everything else int(v.group(1)), code, ln))
            v = _LGKMCNT.search(code)
            if v is not None or everything:
                cur.append(_Ins("ldswait", [], 0 if everything else int(v.group(1)), code, ln))
            continue
        if in_asm:
            continue  # hand-written: assumed to respect the waits it places
        regs = [r for m in _VREG.finditer(code) for r in _regs(m)]
        if regs:
            cur.append(_Ins("use", regs, 0, code, ln))
    if label is not None:
        close([], False)
    return blocks


def _transfer(state: Dict[int, int], ins: List[_Ins], report=None) -> Dict[int, int]:
    """state: register -> position of its load among those in flight (1 = youngest); a register
    with an LDS read in flight is kept under the key -(register + 1), with its position among the LDS reads."""
    st = dict(state)
    for i in ins:
        if i.kind == "load":
            st = {r: (p + 1 if r >= 0 else p) for r, p in st.items()}
            for r in i.regs:
                st[r] = 1
        elif i.kind == "wait":
            st = {r: p for r, p in st.items() if r < 0 or p <= i.n}
        elif i.kind == "ldsread":
            st = {r: (p + 1 if r < 0 else p) for r, p in st.items()}
            for r in i.regs:
                st[-(r + 1)] = 1
        elif i.kind == "ldswait":
            st = {r: p for r, p in st.items() if r >= 0 or p <= i.n}
        elif report is not None:
            for r in i.regs:
                if r in st or -(r + 1) in st:
                    report(i, r)
                    break
    return st


_MFMA_SETTLE = 20  # wait states after which the result of the longest MFMA used here (8 passes) is readable
_MFMA = re.compile(r"^\s*v_mfma\w*\s+a\[(\d+):(\d+)\]\s*,(.*)$")
_AREG = re.compile(r"\ba(?:\[(\d+):(\d+)\]|(\d+)\b)")
_NOP = re.compile(r"^\s*s_nop\s+(\d+)")


def _mfma_hazards(name: str, lines: List[Tuple[int, str]]) -> List[str]:
    """Textual (fall-through order) check of compiler-generated AGPR moves next to inline-assembly MFMAs."""
    seq, in_asm = [], False  # (line, code, in_asm)
    for ln, raw in lines:
        s = raw.strip()
        if s.startswith(";;#ASMSTART"):
            in_asm = True
            continue
        if s.startswith(";;#ASMEND"):
            in_asm = False
            continue
        code = raw.split(";")[0].strip()
        if not code or (code.startswith(".") and not code.endswith(":")):
            continue
        seq.append((ln, code, in_asm))  # (labels stay in the sequence: they delimit loops)
    out = []
    # A loop whose body holds inline-assembly MFMAs must not move accumulators at all: across the
    # back edge the MFMAs at the bottom of the body precede whatever stands at its top.  Blocks and
    # edges of the function; a branch back to a label closes a loop only if the branch can be
    # reached from that label (out-of-line blocks at the end of a function also jump backwards).
    starts = sorted({0} | {k for k, (_, c, _) in enumerate(seq) if c.endswith(":")}
                    | {k + 1 for k, (_, c, _) in enumerate(seq) if _BRANCH.match(c) or c.startswith("s_endpgm")})
    starts = [k for k in starts if k < len(seq)]
    block_of = {}
    for bi, k0 in enumerate(starts):
        for k in range(k0, starts[bi + 1] if bi + 1 < len(starts) else len(seq)):
            block_of[k] = bi
    label_block = {c[:-1]: block_of[k] for k, (_, c, _) in enumerate(seq) if c.endswith(":")}
    succ = [set() for _ in starts]
    for bi, k0 in enumerate(starts):
        k1 = (starts[bi + 1] if bi + 1 < len(starts) else len(seq)) - 1
        last = seq[k1][1]
        m = _BRANCH.match(last)
        if m and m.group(2) in label_block:
            succ[bi].add(label_block[m.group(2)])
        if not last.startswith("s_endpgm") and not (m and m.group(1) == "branch") and bi + 1 < len(starts):
            succ[bi].add(bi + 1)

    def reach(src, edges):
        seen, work = {src}, [src]
        while work:
            for nb in edges[work.pop()]:
                if nb not in seen:
                    seen.add(nb)
                    work.append(nb)
        return seen

    pred = [set() for _ in starts]
    for bi, ss in enumerate(succ):
        for t in ss:
            pred[t].add(bi)
    for bi in range(len(starts)):
        for h in succ[bi]:
            if h > bi or bi not in reach(h, succ):
                continue  # not a back edge of a loop
            body = reach(h, succ) & reach(bi, pred)
            ks = [k for k in range(len(seq)) if block_of[k] in body]
            if any(seq[k][2] and _MFMA.match(seq[k][1]) for k in ks):
                for k in ks:
                    bl, bc, ba = seq[k]
                    if not ba and bc.startswith("v_accvgpr"):
                        out.append("%s: line %d moves an accumulator inside a loop of inline-assembly MFMAs: %s"
                                   % (name, bl, bc))
    for k, (ln, code, asm) in enumerate(seq):
        if asm or not code.startswith("v_accvgpr"):
            continue
        mine = {r for m in _AREG.finditer(code) for r in _regs(m)}
        waited, j = 0, k - 1
        while j >= 0 and waited < _MFMA_SETTLE:
            pl, pc, pasm = seq[j]
            if pc.startswith("s_branch") or pc.startswith("s_endpgm"):
                break  # not reached from the text above
            m = _MFMA.match(pc) if pasm else None
            if m and mine & set(range(int(m.group(1)), int(m.group(2)) + 1)):
                out.append("%s: line %d moves an accumulator %d wait states after the MFMA of line %d wrote it: %s"
                           % (name, ln, waited, pl, code))
                break
            n = _NOP.match(pc)
            if not pc.endswith(":"):
                waited += int(n.group(1)) + 1 if n else 1
            j -= 1
        if code.startswith("v_accvgpr_write") or code.startswith("v_accvgpr_mov"):
            dst = next(iter(_regs(_AREG.search(code))))
            for pl, pc, pasm in [x for x in seq[k + 1:k + 6] if not x[1].endswith(":")][:2]:
                m = _MFMA.match(pc) if pasm else None
                if m and dst in {r for a in _AREG.finditer(m.group(3)) for r in _regs(a)}:
                    out.append("%s: line %d writes a%d right before the MFMA of line %d reads it: %s"
                               % (name, ln, dst, pl, code))
                    break
    return out


_M0_WRITE = re.compile(r"^(?!s_cmp|s_bitcmp)\S+\s+m0\b")


def _m0_hazards(name: str, lines: List[Tuple[int, str]]) -> List[str]:
    """A direct-to-LDS load from inline assembly takes its LDS address from M0.  Where an assembly statement does not set M0
    before such a load, it relies on an earlier statement's value, which the compiler does not know to be in use: then
    no compiler-generated instruction of the function may write M0."""
    borrowed, writes, in_asm, is_set = False, [], False, False
    for ln, raw in lines:
        s = raw.strip()
        if s.startswith(";;#ASMSTART"):
            in_asm, is_set = True, False
            continue
        if s.startswith(";;#ASMEND"):
            in_asm = False
            continue
        code = raw.split(";")[0].strip()
        if in_asm:
            is_set = is_set or _M0_WRITE.match(code) is not None
            borrowed = borrowed or ("_lds_" in code and not is_set)
        elif _M0_WRITE.match(code):
            writes.append((ln, code))
    return ["%s: line %d writes M0, which an assembly statement sets for loads in later ones: %s" % (name, ln, code)
            for ln, code in writes if borrowed]


_LDS_WRITE = re.compile(r"^ds_(?:write|store)")
_LDS_READ = re.compile(r"^ds_(?:read|load)")


def _graph(lines: List[Tuple[int, str]]):
    """-> blocks of a function, each [label, [(line, code, in_asm)], successors by label, falls through].  A barrier of the wave,
    which is a comment in the assembly, is the code `wave_barrier`."""
    blocks, cur, label, in_asm = [], [], "<entry>", False
    for ln, raw in lines:
        s = raw.strip()
        if s.startswith(";;#ASM"):
            in_asm = s.startswith(";;#ASMSTART")
            continue
        m = _LABEL.match(raw)
        if m:
            blocks.append([label, cur, [], True])
            label, cur = m.group(1), []
            continue
        code = "wave_barrier" if s.startswith("; wave barrier") else raw.split(";")[0].strip()
        if not code or code.startswith("."):
            continue
        m = _BRANCH.match(code)
        if m or code.startswith("s_endpgm"):
            blocks.append([label, cur, [m.group(2)] if m else [], bool(m) and m.group(1) == "cbranch"])
            label, cur = "<after %d>" % ln, []
            continue
        cur.append((ln, code, in_asm))
    blocks.append([label, cur, [], False])
    return blocks


def _reaches(blocks, start, transfer, merge):
    """The state at the start of every block that can be reached: `start` at the entry, `transfer(state, instructions)` through
    a block, `merge(state, state, block)` where paths join (blocks count from -1 down; it has to be monotone); None where nothing arrives."""
    index = {b[0]: k for k, b in enumerate(blocks)}
    entry = [None] * len(blocks)
    entry[0] = start
    work = [0]
    while work:
        k = work.pop()
        _, ins, succ, fall = blocks[k]
        st = transfer(entry[k], ins)
        for j in [index[s] for s in succ if s in index] + ([k + 1] if fall and k + 1 < len(blocks) else []):
            new = st if entry[j] is None else merge(entry[j], st, -1 - j)
            if new != entry[j]:
                entry[j] = new
                work.append(j)
    return entry


def _lds_hazards(name: str, lines: List[Tuple[int, str]]) -> List[str]:
    """LDS reads that can follow an LDS write with no barrier between (both the compiler's own)."""
    out = []

    def transfer(written, ins, report=False):
        for ln, code, asm in ins:
            if code == "wave_barrier" or code.startswith("s_barrier"):
                written = False
            elif not asm and _LDS_WRITE.match(code):
                written = True
            elif not asm and written and report and _LDS_READ.match(code):
                out.append("%s: line %d reads LDS after a write with no barrier between: %s" % (name, ln, code))
        return written

    blocks = _graph(lines)
    for b, at in zip(blocks, _reaches(blocks, False, transfer, lambda x, y, _: x or y)):
        if at is not None:
            transfer(at, b[1], report=True)
    return out


_SREGS = re.compile(r"s(?:\[(\d+):(\d+)\]|(\d+))")
_SECOND_RESULT = re.compile(r"v_(?:\w+_co_|div_scale|mad_[ui]64)")
_NO_LANE = ("part", (None,))
_NO_RESULT = ("s_cmp", "s_bitcmp", "s_wait", "s_setprio", "s_barrier", "s_nop", "global_", "buffer_", "flat_", "ds_", "wave_barrier")


def _common(x, y):
    return x[:next((k for k, (p, q) in enumerate(zip(x, y)) if p != q), min(len(x), len(y)))]


def _within(v):
    """The narrowings that lead to a mask which holds what a register holds; None: not known."""
    return None if v is None or v[0] == "rest" else v[1]


def _exec_transfer(state, ins, report=None):
    """What is known of EXEC: the narrowings, by line, that lead from all lanes (none: all of them) to a mask that holds it.
    state: (EXEC's, ((n, what s[n:n+1] or vcc holds), ...)); a register holds ("mask", narrowings), a part of one ("part",
    narrowings), no lane ("part", (None,)), or ("rest", narrowings, wider), what the first lacks of the second as long as EXEC is the first."""
    now, held = state[0], dict(state[1])

    def narrowed(base, ln):
        """A new mask inside `base`; nothing that was said of an earlier one of this line holds any more."""
        for n in [n for n, v in held.items() if ln in v[1]]:
            del held[n]
        return (base[:base.index(ln)] if ln in base else base) + (ln,)

    def joined(v, ln):
        """EXEC and what a register holds, together."""
        if v is None:
            return narrowed((), ln)
        if v[0] == "rest":
            return v[2] if v[1] == now else narrowed((), ln)
        if v == _NO_LANE or v[0] == "mask" and now[:len(v[1])] == v[1]:
            return v[1] if v != _NO_LANE else now
        return narrowed(_common(now, v[1]), ln)

    for ln, code, asm in ins:
        op, _, rest = code.partition(" ")
        if op.startswith(_NO_RESULT):
            continue
        args = [a.strip() for a in rest.split(",")]
        if asm and args[0] == "exec":  # the mask of the statement's loads, which ends it with all ones
            if args[1] == "-1":
                if now and report is not None:
                    report(ln, code)
                now = ()
            continue
        m = [_SREGS.fullmatch(a) for a in args]
        reg = [a if a == "vcc" else int(x.group(1)) if x and x.group(1) else None for a, x in zip(args, m)]
        fixed = {"exec": ("mask", now), "-1": ("mask", ()), "0": _NO_LANE}
        value = [fixed.get(a, held.get(n)) for a, n in zip(args, reg)]
        was, new, also = now, None, None
        if "saveexec" in op:
            new, v = ("mask", now), value[1]
            if op == "s_and_saveexec_b64":
                now = narrowed(now, ln)
            elif op == "s_or_saveexec_b64":
                now = joined(v, ln)
            elif op == "s_andn2_saveexec_b64" and v is not None and v[0] == "rest" and v[1] == now:  # the other side of a branch
                now = narrowed(v[2], ln)
                new = ("rest", now, v[2])
            else:
                now = narrowed((), ln)
            if new[0] == "mask" and ln in new[1]:
                new = None
        elif args[0] == "exec":
            v = value[2] if len(value) > 2 and args[1] == "exec" else None
            if op == "s_mov_b64" and value[1] is not None and value[1][0] == "mask":
                now = value[1][1]
            elif op == "s_or_b64":
                now = joined(v, ln)
            elif op == "s_xor_b64" and v is not None and v[0] == "mask" and v[1][:len(now)] == now and v[1] != now:
                now = narrowed(now, ln)
                also = (reg[2], ("rest", now, was))
            else:
                now = narrowed(now if op in ("s_and_b64", "s_andn2_b64") and args[1] == "exec" else (), ln)
        elif args[0].startswith("exec"):
            now = narrowed((), ln)
        elif op == "s_mov_b64":
            new = value[1]
        elif op == "s_xor_b64" and args[1] == "exec" and value[2] is not None and value[2][0] == "mask" and now[:len(value[2][1])] == value[2][1]:
            new = ("rest", now, value[2][1])
        elif op in ("s_and_b64", "s_andn2_b64", "s_or_b64"):
            x, y = map(_within, value[1:3])
            if op == "s_andn2_b64":
                part = x
            elif op == "s_and_b64":
                part = x if y is None or x is not None and len(x) > len(y) else y
            else:
                part = y if x == _NO_LANE[1] else x if y == _NO_LANE[1] else None if x is None or y is None else _common(x, y)
            new = ("part", part) if part is not None else None
        elif op.startswith("v_cmpx_"):
            now = narrowed(now, ln)
        elif op.startswith("v_cmp_"):
            new = ("part", now)
            if op.endswith("_e32"):
                reg[0] = "vcc"
        written = m[:2] if _SECOND_RESULT.match(op) else m[:1]
        for x in written:
            if x:
                lo, hi = int(x.group(1) or x.group(3)), int(x.group(2) or x.group(3))
                for n in [n for n in held if n != "vcc" and n <= hi and n + 1 >= lo]:
                    del held[n]
        if any(a.startswith("vcc") for a in args[:2]):
            held.pop("vcc", None)
        for n, v in ((reg[0], new), also or (None, None)):
            if n is not None and v is not None and v != ("part", ()):
                held[n] = v
    return now, tuple(sorted(held.items(), key=str))


def _exec_merge(x, y, block):
    now = x[0]
    if x[0] != y[0]:
        now = _common(*(z[0][:z[0].index(block)] if block in z[0] else z[0] for z in (x, y))) + (block,)
    held, other = [], dict(y[1])
    for n, v in x[1]:
        w = other.get(n)
        if w != v:
            p, q = _within(v), _within(w)
            part = q if p == _NO_LANE[1] else p if q == _NO_LANE[1] else None if p is None or q is None else _common(p, q)
            v = ("part", part) if part else None
        if v is not None and block not in v[1]:
            held.append((n, v))
    return now, tuple(held)


def _exec_hazards(name: str, lines: List[Tuple[int, str]]) -> List[str]:
    """Assembly that sets EXEC to all ones where a lane may be switched off."""
    out: List[str] = []
    blocks = _graph(lines)
    if not any(asm and code.replace(" ", "") == "s_mov_b64exec,-1" for b in blocks for _, code, asm in b[1]):
        return out
    states = _reaches(blocks, ((), ()), _exec_transfer, _exec_merge)
    for b, at in zip(blocks, states):
        if at is not None:
            _exec_transfer(at, b[1], lambda ln, code: out.append(
                "%s: line %d switches every lane on where some may be off: %s" % (name, ln, code)))
    return out


def lint(asm_text: str, only_if_name_has: str = "kernel") -> List[str]:
    """Returns one message per violation (empty list: clean)."""
    out: List[str] = []
    funcs, cur, name = [], [], None
    for ln, raw in enumerate(asm_text.split("\n"), 1):
        m = _FUNC.match(raw)
        if m:
            name, cur = m.group(1), []
            continue
        if raw.startswith(".Lfunc_end"):
            if name is not None and only_if_name_has in name:
                funcs.append((name, cur))
            name = None
            continue
        if name is not None:
            cur.append((ln, raw))
    for name, lines in funcs:
        out.extend(_mfma_hazards(name, lines))
        out.extend(_m0_hazards(name, lines))
        out.extend(_lds_hazards(name, lines))
        out.extend(_exec_hazards(name, lines))
        blocks = _parse(lines)
        index = {b[0]: k for k, b in enumerate(blocks)}
        entry: List[Dict[int, int]] = [None] * len(blocks)  # type: ignore
        entry[0] = {}
        work = [0]
        while work:
            k = work.pop()
            label, ins, succ, fall = blocks[k]
            st = _transfer(entry[k], ins)
            nxt = [index[s] for s in succ if s in index]
            if fall and k + 1 < len(blocks):
                nxt.append(k + 1)
            for j in nxt:
                if entry[j] is None:
                    entry[j] = dict(st)
                    work.append(j)
                else:
                    merged, changed = entry[j], False
                    for r, p in st.items():
                        if r not in merged or p < merged[r]:
                            merged[r] = p
                            changed = True
                    if changed:
                        work.append(j)
        for k, (label, ins, succ, fall) in enumerate(blocks):
            if entry[k] is None:
                continue
            _transfer(entry[k], ins, lambda i, r: out.append(
                "%s: line %d touches v%d while a load into it may be in flight: %s" % (name, i.line, r, i.text)))
    return out
