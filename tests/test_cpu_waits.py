"""The tiled GEMMs stage token rows by LDS DMA and wait for them by counting the
loads issued after them ("s_waitcnt vmcnt(N)" before the step's barrier). N is
written in the source, the loads are the compiler's: here the built kernels'
own code is read, and at every barrier no DMA may still be in flight."""

import os
import re
import shutil
import subprocess

import pytest

import rpgbarengine_amd as eng

OBJDUMP = "/opt/rocm/llvm/bin/llvm-objdump"
KERNELS = ["Q8GemmKernelILi64E", "Q8GemmKernelILi128E", "TGemmKernelILi12E", "TGemmKernelILi14E"]

VMEM = re.compile(r"^(buffer|global|scratch|flat)_(load|store|atomic)")


def dma_at_barriers(code):
    """Walks the instructions [(address, text, branch target or None)] from the
    first DMA on through the loop around it, twice, with the queue of memory
    operations in flight, oldest first. Loads that a forward branch may skip
    are not counted on. Returns (barriers seen, those with a DMA in flight)."""
    at = {a: i for i, (a, _, _) in enumerate(code)}
    first = next(i for i, (_, t, _) in enumerate(code) if " lds" in t)
    back = next(i for i in range(first, len(code))
                if code[i][2] is not None and code[i][2] < code[i][0]
                and any(" lds" in t for _, t, _ in code[at[code[i][2]]:i]))
    loop = at[code[back][2]]
    queue, seen, bad = [], 0, 0
    for span in (range(first, back), range(loop, back)):
        skip = -1
        for i in span:
            addr, text, target = code[i]
            if target is not None and target > addr and target <= code[back][0]:
                skip = max(skip, target)
            if VMEM.match(text) and (" lds" in text or addr >= skip):
                queue.append(" lds" in text)
            n = re.search(r"vmcnt\((\d+)\)", text)
            if n:
                queue = queue[len(queue) - min(len(queue), int(n.group(1))):]
            if text.startswith("s_barrier"):
                seen += 1
                bad += any(queue)
    return seen, bad


def listing(text):
    out = []
    for line in text.splitlines():
        m = re.match(r"\s+(\S.*?)\s+// ([0-9A-F]+): [0-9A-F ]+(?:<\S+\+0x([0-9a-f]+)>)?", line)
        if m:
            out.append((int(m.group(2), 16), m.group(1), m.group(3)))
    base = out[0][0]
    return [(a, t, base + int(x, 16) if x and t.startswith(("s_cbranch", "s_branch")) else None) for a, t, x in out]


@pytest.fixture(scope="module")
def functions(tmp_path_factory):
    if not os.path.exists(OBJDUMP):
        pytest.skip("no llvm-objdump")
    d = tmp_path_factory.mktemp("code")
    lib = shutil.copy(eng.LIB_PATH, str(d))
    subprocess.run([OBJDUMP, "--offloading", lib], check=True, capture_output=True)
    found = {}
    for f in sorted(os.listdir(d)):
        if "gfx950" not in f:
            continue
        with open(os.path.join(d, f), "rb") as h:
            data = h.read()
            if b"Q8GemmKernel" not in data and b"TGemmKernel" not in data:
                continue
        text = subprocess.run([OBJDUMP, "-d", os.path.join(d, f)], check=True, capture_output=True, text=True).stdout
        for part in re.split(r"\n(?=[0-9a-f]+ <)", text):
            m = re.match(r"[0-9a-f]+ <(\S+)>:", part)
            if m:
                found[m.group(1)] = part
    return found


@pytest.mark.parametrize("kernel", KERNELS)
def test_dma_has_landed_at_every_barrier(functions, kernel):
    (name,) = [n for n in functions if kernel in n]
    seen, bad = dma_at_barriers(listing(functions[name]))
    assert seen >= 8 and bad == 0  # (four steps a super-block, the loop twice)


def test_the_check_sees_a_missing_load():
    """Three loads counted on, two issued: the DMA before them is in flight."""
    dma, load = "buffer_load_dwordx4 v1, s[4:7], s2 offen lds", "global_load_dwordx4 v[2:5], v6, s[8:9]"

    def code(loads):
        body = [dma] + [load] * loads + ["s_waitcnt vmcnt(3)", "s_barrier", "s_cbranch_scc1 1"]
        return [(4 * i, t, 0 if t.startswith("s_cbranch") else None) for i, t in enumerate(body)]

    assert dma_at_barriers(code(3)) == (2, 0)
    assert dma_at_barriers(code(2)) == (2, 2)
