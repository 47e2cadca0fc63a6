"""No instruction of a built kernel touches a register that a load may still
write.

The kernels that count their loads by hand (``s_waitcnt`` with a number, loads in
inline assembly) are correct only if every register such a load writes is left
alone from the load to a wait that covers it.  The compiler does not know that
the load is still on its way: to it the register holds its value at once, and
where nothing reads the value any more the register is free.  A load that lands
late then overwrites what was put there since, an address as well as a result.

This happened.  The streaming kernel as it was before ``gemm_bs.hip`` asked for
the weights of four steps past the last one and waited for them behind its loop,
but the compiler had computed the epilogue's first addresses above that wait, in
registers that nobody read any more.  Left after whole trips of its four-step
loop, those registers' loads were the oldest and had landed; left after the first
step of a trip (17 steps: 4096 x 1088 x 4096), they were the youngest, and the
launch ended with an illegal access.

The disassembly of every kernel in the library is followed along all its
branches: per register the least number of younger operations of the counter that
its load is booked on, so that ``s_waitcnt cnt(n)`` frees those with n or more.
Loads of one counter complete in order (scalar loads, which do not, are the
compiler's own and not looked at)."""
import os
import re
import subprocess

import pytest

from test_registers import LIBRARY, _code_objects

OBJDUMP = "/opt/rocm/llvm/bin/llvm-objdump"
_REG = re.compile(r"\b([va])(?:(\d+)\b|\[(\d+):(\d+)\])")
_LINE = re.compile(r"^\t(\S+)\s*(.*?)\s*// ([0-9A-F]{12}): ([0-9A-F]{8})")


def _registers(text):
    found = []
    for kind, one, low, high in _REG.findall(text):
        base = 256 if kind == "a" else 0  # accumulation registers
        found += [base + r for r in (range(int(one), int(one) + 1) if one else range(int(low), int(high) + 1))]
    return found


class Instruction:
    """What of an instruction matters here: where it may go next, what it waits
    for, which registers it touches at once and which it writes later."""

    def __init__(self, op, operands, address, word):
        self.op, self.text, self.address = op, f"{op} {operands}", address
        self.target = None
        if op.startswith(("s_branch", "s_cbranch")):
            offset = word & 0xFFFF
            self.target = address + 4 + 4 * (offset - 0x10000 if offset & 0x8000 else offset)
        first = operands.split(",")[0]
        self.touches, self.later, self.counter = _registers(operands), [], None
        if re.match(r"(buffer|global|flat|scratch)_(load|store|atomic)", op):
            self.counter = 0
            to_lds = "_lds_" in op or re.search(r"\blds\b", operands)
            if ("_load" in op and not to_lds) or ("atomic" in op and "sc0" in operands):
                self.later = _registers(first)
        elif op.startswith("ds_"):
            self.counter = 1
            if re.match(r"ds_(read|bpermute|permute|swizzle)|ds_\w*_rtn", op):
                self.later = _registers(first)
        if self.later:  # (asked for twice: the second load lands last)
            self.touches = _registers(operands[len(first):])
        waits = [re.search(name + r"\((\d+)\)", operands) for name in ("vmcnt", "lgkmcnt")]
        self.waits = [int(w.group(1)) if op == "s_waitcnt" and w else None for w in waits]


def kernels_of(listing):
    """Kernel name -> its instructions, from a disassembly."""
    kernels, body = {}, None
    for line in listing:
        head = re.match(r"^[0-9a-f]{16} <(.*)>:$", line)
        if head:
            body = kernels.setdefault(head.group(1), [])
            continue
        m = _LINE.match(line)
        if m and body is not None:
            body.append(Instruction(m.group(1), m.group(2), int(m.group(3), 16), int(m.group(4), 16)))
    return {name: body for name, body in kernels.items() if body}


def touched_in_flight(body):
    """The instructions that touch a register whose load may be on its way."""
    at = {ins.address: i for i, ins in enumerate(body)}
    leaders = {at[ins.target] for ins in body if ins.target is not None}
    states, work, bad = {0: ({}, {})}, [0], {}

    def reach(i, ages):
        if i not in states:
            states[i] = tuple(dict(a) for a in ages)
            work.append(i)
            return
        changed = False
        for have, new in zip(states[i], ages):
            for r, age in new.items():
                if have.get(r, 1 << 30) > age:
                    have[r], changed = age, True
        if changed:
            work.append(i)

    while work:
        i = work.pop()
        ages = [dict(a) for a in states[i]]
        while True:
            ins = body[i]
            for c, n in enumerate(ins.waits):
                if n is not None:
                    ages[c] = {r: a for r, a in ages[c].items() if a < n}
            if any(r in a for a in ages for r in ins.touches):
                bad[ins.address] = ins.text
            if ins.counter is not None:
                c = ins.counter
                ages[c] = {r: a + 1 for r, a in ages[c].items()}
                ages[c].update((r, 0) for r in ins.later)
            assert ins.op not in ("s_setpc_b64", "s_swappc_b64"), "calls are not followed"
            if ins.target is not None:
                reach(at[ins.target], ages)
            if ins.op in ("s_endpgm", "s_branch"):
                break
            i += 1
            if i in leaders:
                reach(i, ages)
                break
    return bad


@pytest.fixture(scope="module")
def kernels(tmp_path_factory):
    if not os.path.exists(LIBRARY):
        import __graft_entry__
        __graft_entry__.build()
    found, folder = {}, tmp_path_factory.mktemp("code")
    for i, elf in enumerate(_code_objects(open(LIBRARY, "rb").read())):
        path = folder / f"{i}.elf"
        path.write_bytes(elf)
        listing = subprocess.run([OBJDUMP, "-d", "--no-show-raw-insn", "--mcpu=gfx950", str(path)], capture_output=True,
                                 text=True, check=True).stdout
        found.update(kernels_of(listing.splitlines()))
    assert len(found) > 100
    return found


@pytest.mark.parametrize("family", ["gemm_i8_wreg", "gemm_i8_bs", "gemm_i8_dma_bs", r"gemm_i8_dmaI", "gemm_i8_flight",
                                    "gemm_i8_skinny", r"gemm_i8I|gemm_i8_batched|sum_parts|pad_rows|pack_b", "quant|dql|minmax|copy"])
def test_no_register_is_touched_before_its_load_has_landed(kernels, family):
    forms = {n: body for n, body in kernels.items() if re.search("k_(" + family + ")", n)}
    assert forms, sorted(kernels)
    bad = {n: b for n, b in ((n, touched_in_flight(body)) for n, body in forms.items()) if b}
    assert not bad, "\n".join(f"{n}\n    " + "\n    ".join(f"{a:x}: {t}" for a, t in list(b.items())[:5]) for n, b in bad.items())


def test_empty_descriptors_come_with_an_offset_of_zero(kernels):
    """The streaming kernels ask for steps past the last one with a descriptor of
    size 0.  The device drops what lies past (size - scalar offset), unsigned: the
    scalar offset is then 0, so a step's second half must lie in the instruction's
    own offset, for every second load of the weights."""
    forms = {n: body for n, body in kernels.items() if re.search("k_gemm_i8_(dma_)?bsI", n)}
    assert forms
    for name, body in forms.items():
        loads = [ins.text for ins in body if re.match(r"buffer_load_dwordx4 v\[\d+:\d+\], v\d+, s\[\d+:\d+\], s\d+ offen", ins.text)
                 and " lds" not in ins.text]
        assert loads and 2 * sum("offset:1024" in t for t in loads) == len(loads), (name, loads[:4])


def loops_of(body):
    """The loops (strongly connected parts of the branches) as lists of instructions."""
    at = {ins.address: i for i, ins in enumerate(body)}
    nexts = [([at[ins.target]] if ins.target is not None else []) +
             ([i + 1] if ins.op not in ("s_branch", "s_endpgm") and i + 1 < len(body) else []) for i, ins in enumerate(body)]
    order, low, stack, found = {}, {}, [], []
    for root in range(len(body)):
        walk = [] if root in order else [(root, iter(nexts[root]))]
        if walk:
            order[root] = low[root] = len(order)
            stack.append(root)
        while walk:
            i, rest = walk[-1]
            for j in rest:
                if j not in order:
                    order[j] = low[j] = len(order)
                    stack.append(j)
                    walk.append((j, iter(nexts[j])))
                    break
                if j in low:
                    low[i] = min(low[i], order[j])
            else:
                walk.pop()
                if walk:
                    low[walk[-1][0]] = min(low[walk[-1][0]], low[i])
                if low[i] == order[i]:
                    part = sorted(stack[stack.index(i):])
                    del stack[stack.index(i):]
                    for j in part:
                        del low[j]
                    if len(part) > 1:
                        found.append([body[j] for j in part])
    return found


def test_the_k_loop_waits_for_one_set_of_loads(kernels):
    """k_gemm_i8 keeps the operands of two steps on their way: in its loop nothing waits
    for the loads of the step before (with a way out in front of the odd step it did in
    every second step, 109 x 10959 x 224 49 -> 59 us)."""
    forms = {n: body for n, body in kernels.items() if re.search(r"k_gemm_i8ILi\d+ELi128E.*Li[12]ELb[01]EEE", n)}
    assert len(forms) > 20
    for name, body in forms.items():
        loops = [part for part in loops_of(body) if any("mfma" in ins.op for ins in part)]
        assert len(loops) == 2, name  # with and without row sums
        for part in loops:
            loads = sum(ins.op == "global_load_dwordx4" for ins in part)
            waits = [ins.waits[0] for ins in part if ins.waits[0] is not None]
            assert loads == 2 * (3 if "ILi64E" in name else 4) and min(waits) >= loads // 2, (name, loads, waits)


@pytest.mark.parametrize("wait,touch,seen", [
    ("s_waitcnt vmcnt(0)", "v_mov_b32_e32 v4, 0", False),
    ("s_waitcnt vmcnt(1)", "v_mov_b32_e32 v4, 0", False),    # one younger load may stand
    ("s_waitcnt vmcnt(1)", "v_mov_b32_e32 v8, 0", True),     # that one
    ("s_waitcnt lgkmcnt(0)", "v_mov_b32_e32 v4, 0", True),   # the other counter
    ("s_nop 0", "v_add_u32_e32 v1, v7, v2", True),           # read
    ("s_nop 0", "global_load_dword v9, v[6:7], off", True),  # as an address
    ("s_nop 0", "global_load_dword v4, v[10:11], off", False),
])
def test_the_rule_itself(wait, touch, seen):
    """Two loads of four registers, a wait, an instruction."""
    lines = ["buffer_load_dwordx4 v[4:7], v0, s[0:3], 0 offen", "buffer_load_dwordx4 v[8:11], v0, s[0:3], 0 offen offset:1024",
             wait, touch, "s_endpgm "]
    if touch.endswith("v[10:11], off"):  # (not an address that is itself on its way)
        lines[1] = "s_nop 0"
    listing = ["%016x <k>:" % 0] + ["\t%s // %012X: 00000000" % (t, 8 * i) for i, t in enumerate(lines)]
    body, = kernels_of(listing).values()
    assert len(body) == 5 and bool(touched_in_flight(body)) == seen
