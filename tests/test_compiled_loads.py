"""The registers and waits of loads that are written in assembly, in the compiled code (no GPU).

gemm_rows loads W in assembly and waits for it by counts.  The compiler takes the outputs of such a load as there at once: where a launch
shape does not fit the vector registers it copies them away or reuses them while the load is on its way, which gives wrong sums or, where
the register has become an address, a memory fault.  Here the file is compiled as it is built, and every kernel is walked, along every path
that can be taken:

* for each register that a load may still write, the least number of loads issued behind it: a wait for all but N retires what has N
  or more behind it, and nothing but a wait may name the others;
* the same for each copy of x into LDS: none may be on its way at a barrier, which publishes them;
* from one barrier to the next a wave issues the copies of one slice of x at most and reads at most one slice from LDS, and it reads
  none before the first barrier.

Not looked at: which of its two slots a slice is copied to and read from, and the order of LDS reads (the compiler's own)."""
import os
import re
import subprocess

import pytest

from tiny_llm_infer_amd.kernels import build

REGISTERS = re.compile(r"\b([va])(?:\[(\d+):(\d+)\]|(\d+))")
MEMORY = ("global_", "buffer_load", "buffer_store", "buffer_atomic", "scratch_", "flat_")
COPY = ("copy", 0)                               # stands for the LDS bytes of a copy on its way


def registers(text):
    out = set()
    for kind, first, last, one in REGISTERS.findall(text):
        out.update((kind, i) for i in range(int(first or one), int(last or one) + 1))
    return out


def kernels(assembly):
    """name -> basic blocks: lists of instructions, and the numbers of the blocks that may follow (first where a branch leads)."""
    found, name = {}, None
    for line in assembly.split("\n"):
        text = line.split(";")[0].strip()
        if re.match(r"[A-Za-z_]\w*:", line):
            name, blocks, labels = line.split(":")[0], [[]], {}
        elif name and line.startswith(".Lfunc_end"):
            follow = []
            for i, block in enumerate(blocks):
                last = block[-1] if block else ""
                to = [labels[last.split()[-1]]] if last.startswith(("s_branch", "s_cbranch")) else []
                if not last.startswith(("s_branch", "s_endpgm")) and i + 1 < len(blocks):
                    to.append(i + 1)
                follow.append(to)
            found[name], name = (blocks, follow), None
        elif name and text.startswith(".LBB"):
            labels[text.rstrip(":")] = len(blocks)
            blocks.append([])
        elif name and text and not text.startswith("."):
            blocks[-1].append(text)
            if text.startswith(("s_branch", "s_cbranch", "s_endpgm")):
                blocks.append([])
    return found


class Shape:
    """What a kernel's template parameters <RT, WAVES, MT, MH, GATED, KG> make of a slice for one wave."""

    def __init__(self, name):
        rt, waves, mt = (int(n) for n in re.search(r"gemm_rows_kernelILi(\d+)ELi(\d+)ELi(\d+)E", name).groups())
        self.fragments, self.copies, self.reads = 4 * rt, mt * 16 // (4 * waves), 4 * mt


# The two ways of copying a slice of x (whole, and with the columns past K) are arms that the compiler joins by scalar flags: a path that
# takes both or neither does not exist.  A flag is a pair of scalar registers set to -1 or 0, read by "vcc = exec and (not) flag" before a
# branch on vcc; what is known of flags, vcc and exec is part of a path's state, and anything else that names one forgets it.
FLAG_SET = re.compile(r"s_mov_b64 (s\[\d+:\d+\]), (-1|0)$")
FLAG_READ = re.compile(r"s_(andn2|and)_b64 vcc, exec, (s\[\d+:\d+\])$")


def flags_of(blocks):
    return {m.group(2) for block in blocks for m in map(FLAG_READ.match, block) if m}


def named_scalars(text):
    out = set()
    for first, last, one in re.findall(r"\bs(?:\[(\d+):(\d+)\]|(\d+))", text):
        out.update(range(int(first or one), int(last or one) + 1))
    return out


def known_after(known, instruction, flags):
    """``known``: flag, "vcc" or "exec" -> whether it is not zero."""
    changed = {}
    if m := FLAG_SET.match(instruction):
        if m.group(1) in flags:
            changed = {m.group(1): m.group(2) == "-1"}
    elif m := FLAG_READ.match(instruction):
        flag = known.get(m.group(2))
        if flag is not None and known.get("exec"):
            changed = {"vcc": flag == (m.group(1) == "and")}
        known = {k: v for k, v in known.items() if k != "vcc"}
        return {**known, **changed}
    elif instruction.startswith("s_cbranch"):
        return known
    scalars = named_scalars(instruction)
    kept = {}
    for k, v in known.items():
        if k in ("vcc", "exec"):
            lost = k in instruction or (k == "exec" and "v_cmpx" in instruction)
        else:
            lost = bool(scalars & named_scalars(k))
        if not lost:
            kept[k] = v
    return {**kept, **changed}


def taken(block, follow, known):
    """The blocks that may follow, given what is known."""
    last = block[-1] if block else ""
    m = re.match(r"s_cbranch_(vcc|exec)(z|nz)\b", last)
    if not m or m.group(1) not in known or len(follow) < 2:
        return follow
    jumps = known[m.group(1)] == (m.group(2) == "nz")
    return follow[:1] if jumps else follow[1:]


class Path:
    """State of a walk: register (or COPY) of a load that may be on its way -> loads and stores issued behind it; copies and LDS reads
    since the last barrier; what is known of flags."""

    def __init__(self, shape, behind, copies, reads, known):
        self.shape, self.behind, self.copies, self.reads, self.known = shape, behind, copies, reads, known

    def key(self):
        return self.copies, self.reads, tuple(sorted(self.known.items()))

    def step(self, instruction, flags):
        """Goes over an instruction; true where it may not stand here."""
        op = instruction.split()[0]
        wrong = False
        self.known = known_after(self.known, instruction, flags)
        if op == "s_waitcnt":
            if wait := re.search(r"vmcnt\((\d+)\)", instruction):
                self.behind = {r: n for r, n in self.behind.items() if n < int(wait.group(1))}
            return False
        if op == "s_barrier":
            wrong = COPY in self.behind
            self.copies = self.reads = 0
            return wrong
        if not op.startswith("s_"):
            wrong = any(r in self.behind for r in registers(instruction))
        if op.startswith("ds_read"):
            self.reads = min(self.reads + 1, self.shape.reads + 1)
            wrong |= self.reads > self.shape.reads
        if op.startswith(MEMORY):
            self.behind = {r: n + 1 for r, n in self.behind.items()}
            if "_load_lds_" in op:
                self.behind[COPY] = 0
                self.copies = min(self.copies + 1, self.shape.copies + 1)
                wrong |= self.copies > self.shape.copies
            elif "_load_" in op:
                self.behind.update((r, 0) for r in registers(instruction[len(op):].split(",")[0]))
        return wrong


def faults(name, kernel):
    """Instructions that may not stand where they do, on some path."""
    blocks, follow = kernel
    shape, flags = Shape(name), flags_of(blocks)
    start = Path(shape, {}, 0, shape.reads, {"exec": True})
    entry = {(0, start.key()): {}}
    work, found = [(0, start.key())], set()
    while work:
        i, key = place = work.pop()
        path = Path(shape, entry[place], key[0], key[1], dict(key[2]))
        for j, instruction in enumerate(blocks[i]):
            if path.step(instruction, flags):
                found.add((i, j))
        for to in taken(blocks[i], follow[i], path.known):
            place = (to, path.key())
            before = entry.get(place)
            joined = dict(path.behind) if before is None else {**path.behind, **before}
            joined = {r: min(n, path.behind.get(r, 64), 64) for r, n in joined.items()}
            if joined != before:
                entry[place] = joined
                work.append(place)
    return [blocks[i][j] for i, j in sorted(found)]


@pytest.fixture(scope="module")
def rows_kernels(tmp_path_factory):
    out = str(tmp_path_factory.mktemp("gemm_rows") / "gemm_rows.s")
    done = subprocess.run([build._hipcc(), *build.FLAGS, "--cuda-device-only", "-S", os.path.join(build.CSRC, "gemm_rows.hip"), "-o", out],
                          stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True)
    assert done.returncode == 0, done.stdout
    with open(out) as f:
        found = {n: k for n, k in kernels(f.read()).items() if "gemm_rows_kernel" in n}
    assert len(found) == 12                      # six launch shapes, each with a gate and without
    return found


def changed(kernel, change):
    """The kernel with every instruction replaced by the list that ``change(block, place, instruction)`` gives, or left where that is None."""
    blocks, follow = kernel
    out = []
    for i, block in enumerate(blocks):
        out.append([])
        for j, text in enumerate(block):
            new = change(i, j, text)
            out[-1].extend([text] if new is None else new)
    return out, follow


def waits_for_x(kernel):
    """(block, place of the wait, place of the barrier) of the two barriers that publish slices of x: the loop's, the last slice's.  Behind the
    last one LDS is read at once; behind the loop's the copies of the next slice are issued first."""
    blocks, _ = kernel
    loop, last = [], []
    for i, block in enumerate(blocks):
        for j, text in enumerate(block):
            waits = [k for k in range(j) if block[k].startswith("s_waitcnt vmcnt")]
            if text == "s_barrier" and waits:
                (last if any(t.startswith("ds_read") for t in block[j:]) else loop).append((i, waits[-1], j))
    assert len(loop) == len(last) == 1
    return loop[0], last[0]


def test_nothing_is_named_before_its_wait(rows_kernels):
    for name, kernel in rows_kernels.items():
        assert faults(name, kernel) == [], name


def test_no_register_is_moved_out_of_the_way(rows_kernels):
    """No accumulation registers, nothing spilled."""
    for name, (blocks, _) in rows_kernels.items():
        assert not [t for block in blocks for t in block if "accvgpr" in t or t.startswith("scratch_")], name


def test_every_arm_of_copies_is_walked(rows_kernels):
    """A copy issued twice is more than a slice's: found in each arm, so each arm is on some path."""
    for name, kernel in rows_kernels.items():
        blocks, _ = kernel
        copies = [(i, j) for i, block in enumerate(blocks) for j, t in enumerate(block) if t.startswith("global_load_lds_")]
        arms = {i: (i, j) for i, j in copies}
        assert len(arms) == 4 and len(copies) == 4 * Shape(name).copies, name    # before the loop and in it, whole and with columns past K
        for place in arms.values():
            assert faults(name, changed(kernel, lambda i, j, t: [t, t] if (i, j) == place else None)), (name, place)


def later(text, loads):
    return [re.sub(r"vmcnt\((\d+)\)", lambda m: f"vmcnt({int(m.group(1)) + loads})", text)]


MISTAKES = {
    "a register moved behind its load": lambda p, at, text: [text, f"v_accvgpr_write_b32 a0, v{p.register}"] if at == p.load else None,
    "a register reused behind its load": lambda p, at, text: [text, f"v_mov_b32_e32 v{p.register}, 0"] if at == p.load else None,
    "waits for W one load late": lambda p, at, text: later(text, 1) if at in p.w_waits else None,
    "waits for x one copy late": lambda p, at, text: later(text, 1) if at in p.x_waits else None,
    "x waited for eight loads late": lambda p, at, text: later(text, 8) if at in p.x_waits else None,
    "x not waited for": lambda p, at, text: ["s_waitcnt vmcnt(63)"] if at in p.x_waits else None,
    "no wait for x": lambda p, at, text: [] if at in p.x_waits else None,
    "no wait for the last slice of x": lambda p, at, text: [] if at == p.x_waits[1] else None,
    "no barrier in the loop": lambda p, at, text: [] if at == p.barriers[0] else None,
    "no barrier before the last slice": lambda p, at, text: [] if at == p.barriers[1] else None,
    "a read before the first barrier": lambda p, at, text: [text, "ds_read_b128 v[0:3], v0"] if at == (0, 0) else None,
}


class Places:
    def __init__(self, kernel):
        blocks, _ = kernel
        every = [((i, j), t) for i, block in enumerate(blocks) for j, t in enumerate(block)]
        loop, last = waits_for_x(kernel)
        self.x_waits = [at[:2] for at in (loop, last)]
        self.barriers = [(at[0], at[2]) for at in (loop, last)]
        self.w_waits = [at for at, t in every if re.match(r"s_waitcnt vmcnt\([1-9]\d*\)$", t) and at not in self.x_waits]
        self.load, text = [(at, t) for at, t in every if t.startswith("global_load_dwordx4")][-1]
        self.register = text.split("[")[1].split(":")[0]


@pytest.mark.parametrize("mistake", MISTAKES)
def test_the_walk_sees_mistakes(rows_kernels, mistake):
    for name, kernel in rows_kernels.items():
        places = Places(kernel)
        assert len(places.w_waits) == 7, name    # four k-steps of a slice in the loop, three of the last one (its fourth waits for all)
        assert faults(name, changed(kernel, lambda i, j, text: MISTAKES[mistake](places, (i, j), text))), name
