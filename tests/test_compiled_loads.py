"""The registers of loads that are written in assembly, in the compiled code (no GPU).

gemm_rows loads W in assembly and waits for it by counts.  The compiler takes the outputs of such a load as there at once: where a launch
shape does not fit the vector registers it copies them away or reuses them while the load is on its way, which gives wrong sums or, where
the register has become an address, a memory fault.  Here every kernel of the file is compiled and walked: for each register that
a load may still write, the least number of loads issued behind it on any path; a wait for all but N retires what has N or more
behind it, and nothing but a wait may name the others.  This checks the counts of the waits as well."""
import os
import re
import subprocess
from concurrent.futures import ThreadPoolExecutor

import pytest

from tiny_llm_infer_amd.kernels import build

REGISTERS = re.compile(r"\b([va])(?:\[(\d+):(\d+)\]|(\d+))")
MEMORY = ("global_", "buffer_load", "buffer_store", "buffer_atomic", "scratch_", "flat_")
RAGGED = "const bool ragged = (K & 127) != 0;"
LAST_SLICE = "if (ragged && slice == k_steps - 1) {"


def registers(text):
    out = set()
    for kind, first, last, one in REGISTERS.findall(text):
        out.update((kind, i) for i in range(int(first or one), int(last or one) + 1))
    return out


def kernels(assembly):
    """name -> basic blocks: lists of instructions, and the numbers of the blocks that may follow."""
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


def after(behind, instruction):
    """``behind``: register of a load that may be on its way -> loads and stores issued behind it."""
    op = instruction.split()[0]
    if op == "s_waitcnt":
        wait = re.search(r"vmcnt\((\d+)\)", instruction)
        return {r: n for r, n in behind.items() if n < int(wait.group(1))} if wait else behind
    if not op.startswith(MEMORY):
        return behind
    behind = {r: n + 1 for r, n in behind.items()}
    if "_load_" in op and "_lds_" not in op:
        behind.update((r, 0) for r in registers(instruction[len(op):].split(",")[0]))
    return behind


def faults(kernel):
    """Instructions that name a register of a load that may still be on its way."""
    blocks, follow = kernel
    entry = [None] * len(blocks)
    entry[0], work = {}, [0]
    while work:
        i = work.pop()
        behind = entry[i]
        for instruction in blocks[i]:
            behind = after(behind, instruction)
        for j in follow[i]:
            joined = dict(behind) if entry[j] is None else {**behind, **entry[j]}
            joined = {r: min(n, behind.get(r, 64), 64) for r, n in joined.items()}
            if joined != entry[j]:
                entry[j] = joined
                work.append(j)
    found = []
    for i, block in enumerate(blocks):
        behind = entry[i]
        for instruction in block if behind is not None else ():
            if not instruction.startswith("s_") and any(r in behind for r in registers(instruction)):
                found.append(instruction)
            behind = after(behind, instruction)
    return found


def compiled(folder, source, name):
    path = os.path.join(folder, name + ".hip")
    with open(path, "w") as f:
        f.write(source)
    out = path[:-4] + ".s"
    subprocess.run([build._hipcc(), *build.FLAGS, "-I", build.CSRC, "--cuda-device-only", "-S", path, "-o", out], check=True, stdout=subprocess.DEVNULL,
                   stderr=subprocess.DEVNULL)
    with open(out) as f:
        return f.read()


# The two ways of copying a slice of x are compiled apart: both issue as many copies, but in one kernel the walk would also take
# paths with neither or both, which do not exist.
@pytest.fixture(scope="module")
def assembly(tmp_path_factory):
    with open(os.path.join(build.CSRC, "gemm_rows.hip")) as f:
        source = f.read()
    assert RAGGED in source and LAST_SLICE in source
    forms = {"built": source, "whole": source.replace(RAGGED, "const bool ragged = false;"),
             "ragged": source.replace(RAGGED, "const bool ragged = true;").replace(LAST_SLICE, "if (ragged) {")}
    folder = str(tmp_path_factory.mktemp("gemm_rows"))
    with ThreadPoolExecutor(len(forms)) as pool:
        texts = list(pool.map(lambda form: compiled(folder, forms[form], form), forms))
    return dict(zip(forms, texts))


def rows_kernels(assembly):
    found = {n: k for n, k in kernels(assembly).items() if "gemm_rows_kernel" in n}
    assert len(found) == 12                      # six launch shapes, each with a gate and without
    return found


@pytest.mark.parametrize("form", ["whole", "ragged"])
def test_no_register_is_named_before_its_wait(assembly, form):
    for name, kernel in rows_kernels(assembly[form]).items():
        assert faults(kernel) == [], name


def test_no_register_is_moved_out_of_the_way(assembly):
    """The kernels as they are built: no accumulation registers, nothing spilled."""
    for name, (blocks, _) in rows_kernels(assembly["built"]).items():
        assert not [t for block in blocks for t in block if "accvgpr" in t or t.startswith("scratch_")], name


def test_the_walk_sees_mistakes(assembly):
    name, kernel = next(iter(rows_kernels(assembly["whole"]).items()))
    blocks, follow = kernel
    place = [(i, j) for i, block in enumerate(blocks) for j, t in enumerate(block) if t.startswith("global_load_dwordx4")][-1]
    register = blocks[place[0]][place[1]].split("[")[1].split(":")[0]
    moved = [list(b) for b in blocks]
    moved[place[0]].insert(place[1] + 1, f"v_accvgpr_write_b32 a0, v{register}")
    assert faults((moved, follow))               # a register copied while its load is on its way
    longer = [[re.sub(r"vmcnt\((\d+)\)", lambda m: f"vmcnt({int(m.group(1)) + 1})" if m.group(1) != "0" else m.group(0), t) for t in b] for b in blocks]
    assert faults((longer, follow))              # waits for one load less than they should
