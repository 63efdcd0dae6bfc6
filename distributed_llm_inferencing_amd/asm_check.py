"""Wait states around inline assembly, read off the assembly that hipcc wrote.

hipcc pads the hazards of its own gfx950 instructions and none of an asm statement's. Where a kernel's matrix
instructions are asm statements, copies that hipcc makes of their accumulators (out of the AGPR file where branches
meet, say) may stand too close behind them, and the hardware does not hold such a read back. ``check`` follows the
control flow from every producer and names the consumers that come too early. The counts are those that hipcc itself
pads behind the builtins; an instruction counts for one wait state, ``s_nop n`` for n + 1.
"""
from __future__ import annotations

import re

# wait states from a matrix product to any other reader or writer of its result (4, 8 and 16 passes)
MFMA_RESULT = {"v_mfma_f32_16x16x32_bf16": 8, "v_mfma_f32_32x32x16_bf16": 12}
MFMA_RESULT_MOST = 20
# from a vector instruction to a matrix product that reads its result
MFMA_OPERAND = 2
# from a vector instruction's scalar result to a memory instruction that reads it
SCALAR_TO_MEMORY = 5
_MEMORY = ("buffer_", "global_", "flat_", "scratch_")

_REG = re.compile(r"(?<![\w.])([vas])(?:(\d+)|\[(\d+):(\d+)\])(?!\w)")
_LABEL = re.compile(r"^([.\w$]+):")


def registers(operand: str) -> frozenset:
    out = set()
    for kind, one, first, last in _REG.findall(operand):
        lo, hi = (int(one), int(one)) if one else (int(first), int(last))
        out.update((kind, i) for i in range(lo, hi + 1))
    return frozenset(out)


class Code:
    """A function's instructions: (name, operands, line of the file), and where its labels stand."""

    def __init__(self, name: str):
        self.name, self.code, self.labels = name, [], {}

    def following(self, at: int):
        name, ops, _ = self.code[at]
        if name in ("s_endpgm", "s_setpc_b64"):
            return
        if name.startswith(("s_branch", "s_cbranch")):
            yield self.labels[ops[0]]
        if name != "s_branch" and at + 1 < len(self.code):
            yield at + 1

    def within(self, at: int, states: int):
        """The instructions that can follow ``at`` before ``states`` wait states have passed."""
        left, todo = {}, [(n, states) for n in self.following(at)]
        while todo:
            n, s = todo.pop()
            if s <= left.get(n, 0):
                continue
            left[n] = s
            name, ops, _ = self.code[n]
            s -= int(ops[0], 0) + 1 if name == "s_nop" else 1
            if s > 0:
                todo += [(m, s) for m in self.following(n)]
        return left


def functions(text: str):
    """The functions of an assembly file as hipcc writes it."""
    kinds = set(re.findall(r"^\s*\.type\s+([\w.$]+),@function", text, re.M))
    fn = None
    for i, line in enumerate(text.splitlines(), 1):
        line = line.split(";", 1)[0].rstrip()
        if not line:
            continue
        label = _LABEL.match(line)
        if label:
            if label[1] in kinds:
                fn = Code(label[1])
            elif label[1].startswith(".Lfunc_end"):
                if fn is not None:
                    yield fn
                fn = None
            elif fn is not None:
                fn.labels[label[1]] = len(fn.code)
        elif fn is not None and not line.lstrip().startswith("."):
            name, _, ops = line.strip().partition(" ")
            fn.code.append((name, [o.strip() for o in re.split(r",(?![^\[]*\])", ops.strip())], i))


def _result_touched(result: frozenset, name: str, ops) -> bool:
    if not name.startswith("v_mfma"):
        return any(result & registers(o) for o in ops)
    # (a product's own accumulator goes on in the next one, and is begun anew, without a wait)
    same = lambda o: not result & registers(o) or registers(o) == result
    return bool(result & (registers(ops[1]) | registers(ops[2]))) or not (same(ops[0]) and same(ops[3]))


def _written(name: str, ops) -> frozenset:
    """The registers that a vector instruction other than a matrix product writes."""
    second = "swap" in name or "div_scale" in name or "_co_" in name
    return registers(ops[0]) | (registers(ops[1]) if second else frozenset())


def faults(fn: Code):
    """(line, what) of the consumers in a function that come too early."""
    for at, (name, ops, line) in enumerate(fn.code):
        if name.startswith("v_mfma"):
            result = registers(ops[0])
            for n in fn.within(at, MFMA_RESULT.get(name, MFMA_RESULT_MOST)):
                if _result_touched(result, *fn.code[n][:2]):
                    yield fn.code[n][2], f"{fn.code[n][0]} {fn.code[n][1][0]} too early behind line {line}'s {name} {ops[0]}"
        elif name.startswith("v_"):
            result = _written(name, ops)
            scalars = frozenset(r for r in result if r[0] == "s")
            for n in fn.within(at, SCALAR_TO_MEMORY if scalars else MFMA_OPERAND):
                to, used, where = fn.code[n]
                early = scalars if to.startswith(_MEMORY) else result if to.startswith("v_mfma") and not scalars else ()
                if any(registers(o).intersection(early) for o in used):
                    yield where, f"{to} {used[0]} too early behind line {line}'s {name} {ops[0]}"


def check(text: str, src: str) -> None:
    """Raise where an instruction of the assembly ``text`` comes before its operands' wait states are over."""
    found = [f"{fn.name}, line {line}: {what}" for fn in functions(text) for line, what in sorted(set(faults(fn)))]
    if found:
        raise RuntimeError(f"{src}: {len(found)} hazards that hipcc does not pad, such as\n" + "\n".join(found[:8]))
