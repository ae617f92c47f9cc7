"""What the compiler does not look after around inline assembly, checked in the assembly it writes.

The hazard recogniser knows the instructions the compiler selected, not those inside an asm statement: it counts no wait
states from or to them.  The kernels that place matrix instructions and direct loads into LDS by hand rely on what stands
between them, which another compiler or an edit elsewhere in the kernel can change without a word.  The build runs
`check` over those files (build.py).

M0, which the loads into LDS take their address from, is a reserved register: an asm statement cannot name it as changed (the
compiler warns of undefined behaviour), so it has to be the asm statements' alone.

Wait states are counted as the compiler counts them, one per instruction and N + 1 for `s_nop N`, along every path that leads
to an instruction, around loops too.
"""
import re

MFMA_RESULT = 19        # a matrix instruction of 16 passes and any other use of its result (the ones here have 8 at most)
VALU_TO_MFMA = 2        # a vector instruction's result and a matrix instruction that reads it
VALU_SGPR_TO_VMEM = 5   # a scalar register written by a vector instruction and a memory instruction that reads it
M0_TO_LOAD_LDS = 1      # M0 written by a scalar instruction and the load into LDS that takes its address from it

_REG = re.compile(r"(?<![\w.$@])(?:([avs])(\d+)|([avs])\[(\d+):(\d+)\]|(m0|vcc))(?!\w)")
_MEMORY = ("global_", "buffer_", "scratch_", "flat_")


def _regs(text):
    out = set()
    for m in _REG.finditer(text):
        if m.group(1):
            out.add((m.group(1), int(m.group(2))))
        elif m.group(3):
            out.update((m.group(3), i) for i in range(int(m.group(4)), int(m.group(5)) + 1))
        else:
            out.add((m.group(6), 0))
    return out


class _Instr:
    __slots__ = ("line", "text", "op", "args", "asm", "before", "_uses", "_defs")

    def __init__(self, line, text, asm):
        self.line, self.text, self.asm, self.before = line, text, asm, []
        parts = text.split(None, 1)
        self.op = parts[0]
        self.args = [a.strip() for a in re.split(r",(?![^\[]*\])", parts[1])] if len(parts) > 1 else []
        self._uses = self._defs = None

    mfma = property(lambda i: i.op.startswith("v_mfma"))
    valu = property(lambda i: i.op.startswith("v_") and not i.mfma)
    waits = property(lambda i: int(i.args[0], 0) + 1 if i.op == "s_nop" else 1)

    def defs(self):
        """Registers written (of vector and scalar arithmetic; a compare's masks among them)."""
        if self._defs is None:
            writes = self.op.startswith(("v_", "s_")) and self.args and not self.op.startswith(("s_cmp", "s_nop", "s_wait"))
            self._defs = _regs(self.args[0]) if writes else set()
            if self.op.startswith(("v_add_co", "v_sub_co", "v_addc_co", "v_subb_co", "v_mad_u64", "v_mad_i64", "v_div_scale")):
                self._defs = self._defs | _regs(self.args[1])
        return self._defs

    def uses(self):
        """Registers read, the result's among them where it is an operand as well."""
        if self._uses is None:
            self._uses = _regs(" , ".join(self.args[1:] if self.op.startswith(("v_", "s_")) else self.args))
        return self._uses


def _function(lines):
    """Instructions of one function, each with those that can stand in front of it."""
    instrs, labels, jumps, pending, asm, falls = [], {}, [], [], False, False
    for nr, raw in lines:
        text = raw.strip()
        if text.startswith(";;#ASM"):
            asm = text.startswith(";;#ASMSTART")
            continue
        text = text.split(";", 1)[0].split("//", 1)[0].strip()
        if not text:
            continue
        if text.endswith(":"):
            pending.append(text[:-1])
            continue
        if text.startswith("."):
            continue
        i = _Instr(nr, text, asm)
        if falls:
            i.before.append(instrs[-1])
        for name in pending:
            labels[name] = i
        pending = []
        instrs.append(i)
        if i.op in ("s_branch",) or i.op.startswith("s_cbranch"):
            jumps.append((i, i.args[0]))
        falls = i.op not in ("s_branch", "s_endpgm", "s_setpc_b64")
    for i, name in jumps:
        if name in labels:
            labels[name].before.append(i)
    return instrs


def _behind(instr, window, wanted):
    """The first instruction that `wanted` holds for with fewer than `window` wait states between it and `instr`, or None."""
    best = {}
    todo = [(b, 0) for b in instr.before]
    while todo:
        b, waits = todo.pop()
        if waits >= window or best.get(id(b), window) <= waits:
            continue
        best[id(b)] = waits
        if wanted(b):
            return b
        todo.extend((p, waits + b.waits) for p in b.before)
    return None


def _check_function(name, instrs, out):
    def fault(i, b, what):
        out.append("%s: line %d: %s: %s ... %s" % (name, i.line, what, b.text, i.text))

    for i in instrs:
        if not i.mfma:
            acc = {r for r in (i.uses() | i.defs()) if r[0] in "av"}
            if any(r[0] == "a" for r in acc) or (acc and not i.asm):
                b = _behind(i, MFMA_RESULT, lambda b: b.mfma and b.asm and b.defs() & acc) if acc else None
                if b:
                    fault(i, b, "a product's result is touched too early")
        elif i.asm:
            b = _behind(i, VALU_TO_MFMA, lambda b: b.valu and b.defs() & i.uses())
            if b:
                fault(i, b, "a product reads a vector result too early")
        if i.asm and i.op.startswith(_MEMORY):
            scalar = {r for r in i.uses() if r[0] in ("s", "vcc")} | ({("m0", 0)} if "lds" in i.op else set())
            b = _behind(i, VALU_SGPR_TO_VMEM, lambda b: b.valu and b.defs() & scalar)
            if b:
                fault(i, b, "a memory instruction reads a scalar register too early")
        if not i.asm and ("m0", 0) in i.uses() | i.defs():
            out.append("%s: line %d: the compiler uses M0 as well: %s" % (name, i.line, i.text))
        if "_load_lds_" in i.op:
            b = _behind(i, M0_TO_LOAD_LDS, lambda b: b.op.startswith("s_") and ("m0", 0) in b.defs())
            if b:
                fault(i, b, "a load into LDS follows its address too early")


def check(text, spills=True, fused=True, registers=()):
    """The faults found in an assembly file, as texts; `spills`, `fused`: also registers kept in memory, and products rounded
    to half in the instruction that forms them (v_fma_mixlo / mixhi: one rounding where the sources have two); `registers`: pairs of
    a pattern and the vector registers, of both files, that a kernel whose name it is found in may have (a CU holds one workgroup of
    four waves less for them otherwise).  A pattern that no kernel has is a fault as well."""
    out, name, lines = [], None, []
    used = re.findall(r"^\s*\.amdhsa_kernel (\S+)$.*?^\s*\.amdhsa_next_free_vgpr (\d+)$", text, re.M | re.S) if registers else []
    for pattern, most in registers:
        seen = [(k, int(n)) for k, n in used if re.search(pattern, k)]
        out += ["%s: %d registers, %d at most" % (k, n, most) for k, n in seen if n > most]
        if not seen:
            out.append("no kernel is named like %s" % pattern)
    for nr, line in enumerate(text.splitlines(), 1):
        m = re.match(r"^([A-Za-z_$][\w$]*):", line)
        if m:
            name, lines = m.group(1), []
            continue
        if line.startswith(".Lfunc_end"):
            if name:
                _check_function(name, _function(lines), out)
            name = None
        elif name:
            lines.append((nr, line))
            if fused and re.match(r"\s*v_fma_mix(lo|hi)_", line):
                out.append("%s: line %d: a product is rounded once: %s" % (name, nr, line.strip()))
        if spills:
            m = re.match(r"^\s*; ScratchSize: ([1-9]\d*)", line)
            if m:
                out.append("line %d: %s bytes of registers in memory" % (nr, m.group(1)))
    return out
