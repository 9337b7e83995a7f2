"""The GEMM path's counted waits, followed through the library's device code (CPU).

sg_mainloop waits with s_waitcnt vmcnt(n) before each step's barrier until only
loads newer than the step's own LDS fill can be outstanding.  The count holds
only if the loads it counts on are there in the compiled code (the compiler
drops loads that nobody reads), so this disassembles the built library and
follows the queue of outstanding vector memory operations along every path.
"""
import os
import re
import subprocess
from pathlib import Path

import pytest

from littlebit_amd.build import LIB_PATH

OBJDUMP = Path(os.environ.get("ROCM_PATH", "/opt/rocm")) / "llvm" / "bin" / "llvm-objdump"
KERNELS = [f"sg_latent_kernelILb{s}ELb{g}ELi{mi}E" for s, g in ((1, 0), (0, 1), (0, 0)) for mi in (1, 2, 4)[:3 - s]] + [
    f"sg_expand_kernelI{y}Lb{s}ELi{mi}ELi{nj}E" for y in "ft" for s in (0, 1) for mi, nj in ((1, 1), (2, 1), (2, 2))]


def listing(asm):
    """{kernel: [(address, mnemonic, operands, branch target)]} of a disassembly."""
    out, code, start = {}, None, 0
    for line in asm.splitlines():
        m = re.match(r"([0-9a-f]+) <(\S+)>:", line)
        if m:
            code = out.setdefault(m[2], [])
            start = int(m[1], 16)
            continue
        m = re.match(r"\s+(\S+)\s*(.*?)\s*// ([0-9A-F]+):.*?(?:<\S+\+0x([0-9a-f]+)>)?$", line)
        if m and code is not None:
            code.append((int(m[3], 16), m[1], m[2], start + int(m[4], 16) if m[4] else None))
    return out


def early_barriers(code, mi, nj, prologue_groups):
    """Addresses of barriers that step k can pass while a fill of a step <= k is in flight.

    Fill f is the DMA instructions mi * f .. of a path, step k its k-th barrier; both are kept
    relative to the current step, which makes the states finite.  The loads of a column's sign
    words are one 16-byte load or, of a matrix under 4 words, 4 of 4 bytes; the compiler tests the
    same condition twice, so only paths with one load per column and group are real.
    """
    index = {c[0]: i for i, c in enumerate(code)}
    succ = []
    for i, (_, op, _, target) in enumerate(code):
        s = [] if op == "s_endpgm" or (op == "s_branch") else [i + 1]
        if op.startswith(("s_branch", "s_cbranch")):
            s.append(index[target])
        succ.append([j for j in s if j < len(code)])
    barriers = [i for i, c in enumerate(code) if c[1] == "s_barrier"]
    pred = [[] for _ in code]
    for i, s in enumerate(succ):
        for j in s:
            pred[j].append(i)
    live, todo = set(barriers), list(barriers)  # a barrier is still ahead
    while todo:
        for j in pred[todo.pop()]:
            if j not in live:
                live.add(j)
                todo.append(j)
    targets = {c[3] for c in code}

    def segment(i, queue, dma):
        """(barrier, queue before it, next DMA, groups of words) of every path from i to the next barrier."""
        seen, ends, todo = set(), set(), [(i, queue, dma, 0, 0)]
        while todo:
            state = todo.pop()
            if state in seen or state[0] not in live:
                continue
            seen.add(state)
            i, queue, dma, groups, run = state
            at, op, args, _ = code[i]
            if at in targets:
                run = 0
            if op == "s_barrier":
                ends.add((i, queue, dma, groups))
                continue
            if op == "s_waitcnt" and "vmcnt" in args:
                n = int(re.search(r"vmcnt\((\d+)\)", args)[1])
                queue = queue[max(0, len(queue) - n):]
            elif op.startswith("global_load_lds"):
                queue, dma = queue + (dma,), dma + 1
            elif op.startswith(("global_", "scratch_", "buffer_", "flat_")):
                queue = queue + (None,)
                run = run + 1 if op == "global_load_dword" else 0
                if op == "global_load_dwordx4" or run == 4:
                    groups, run = groups + 1, 0
            if op.startswith(("s_cbranch", "s_branch")):
                run = 0
            todo += [(j, queue, dma, groups, run) for j in succ[i]]
        return ends

    bad, seen, todo = set(), set(), [(0, (), 0, prologue_groups)]
    while todo:
        state = todo.pop()
        if state in seen:
            continue
        seen.add(state)
        i, queue, dma, want = state
        ends = segment(i, queue, dma)
        for b in {e[0] for e in ends}:
            paths = [e for e in ends if e[0] == b]
            paths = [e for e in paths if e[3] == want] or [e for e in paths if e[3] == 0]
            assert paths, hex(code[b][0])
            for _, q, d, _ in paths:
                if any(f is not None and f < mi for f in q):
                    bad.add(code[b][0])
                todo.append((b + 1, tuple(None if f is None else f - mi for f in q if f is None or f >= mi), d - mi, nj))
    assert len(barriers) >= 7  # four steps of the ring, three of the rest
    return sorted(bad)


@pytest.fixture(scope="module")
def kernels(tmp_path_factory):
    if not OBJDUMP.exists() or not LIB_PATH.exists():
        pytest.skip("llvm-objdump or the built library not found")
    d = tmp_path_factory.mktemp("gemm_waits")
    (d / "lib.so").symlink_to(LIB_PATH)
    subprocess.run([str(OBJDUMP), "--offloading", "lib.so"], cwd=d, check=True, capture_output=True)
    obj = next(d.glob("*gfx950"))
    names = [f"_ZN12_GLOBAL__N_1{len(k.split('I')[0])}{k}EEvNS_8SgParamsE" for k in KERNELS]
    r = subprocess.run([str(OBJDUMP), "-d", "--no-show-raw-insn", f"--disassemble-symbols={','.join(names)}", str(obj)],
                       check=True, capture_output=True, text=True)
    return dict(zip(KERNELS, map(listing(r.stdout).__getitem__, names)))


@pytest.mark.parametrize("name", KERNELS)
def test_every_fill_has_landed_before_its_step(kernels, name):
    split = "Lb1E" in name.split("kernelI")[1][:5]
    tiles = [int(x) for x in re.findall(r"Li(\d)E", name)]
    mi, nj = tiles[0], tiles[1] if len(tiles) > 1 else 1
    bad = early_barriers(kernels[name], mi, nj, nj if split else 2 * nj)
    assert not bad, [hex(b) for b in bad]


def test_a_dropped_load_is_found():
    """Step 1 waits for two fills of one DMA and a load that is not there: step 1's own fill may be in flight."""
    loads = ["global_load_lds_dwordx4 v[0:1], off"] * 3
    step = ["s_waitcnt vmcnt(2) lgkmcnt(0)", "s_barrier"]
    tail = loads[:1] + ["s_waitcnt vmcnt({}) lgkmcnt(0)", "s_barrier"] + (loads[:1] + step) * 5

    def code(count):
        words = ["global_load_dwordx4 v[2:5], v[6:7], off"]
        return [(4 * i, *s.split(" ", 1), None) if " " in s else (4 * i, s, "", None)
                for i, s in enumerate(words + loads + step + [t.format(count) for t in tail] + ["s_endpgm"])]

    assert early_barriers(code(2), 1, 1, 1) == []
    assert early_barriers(code(3), 1, 1, 1) == [4 * 8]
