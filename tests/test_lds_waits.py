"""Barriers that hand LDS data from wave to wave, in the assembly of the tile kernel (tile.hip): at the barrier at the top of its loop over the row tiles, none of
a wave's LDS writes may still be on its way, whichever path led there.  The wait ahead of it leaves the last few LDS accesses in flight, on the
understanding that they are reads."""
import os
import re
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HIPCC = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
FLAGS = ["--offload-arch=gfx950", "-O3", "-std=c++17", "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops"]
DONE = 1 << 20                                       # no write in flight


def _blocks(lines):
    """Basic blocks of one kernel: [(instructions, successors)], by position."""
    blocks, names, far = [[]], {}, None
    for line in lines:
        label = re.match(r"^(\.LBB\d+_\d+):", line)
        if label:
            blocks.append([])
            names[label.group(1)] = len(blocks) - 1
            continue
        text = line.split(";")[0].strip()
        m = re.match(r"s_add_u32 .*\((\.LBB\d+_\d+)-\.Lpost_getpc", text)       # a jump beyond a branch's reach: s_getpc, s_add, s_addc, s_setpc
        far = m.group(1) if m else far
        if not text or text.startswith(".") or text.endswith(":"):
            continue
        blocks[-1].append(text if not text.startswith("s_setpc") else "s_branch " + far)
        if re.match(r"s_(c?branch|setpc|endpgm)", text):
            blocks.append([])
    after = []
    for i, block in enumerate(blocks):
        last = block[-1] if block else ""
        to = [names[last.split()[1]]] if re.match(r"s_c?branch", last) else []
        if not re.match(r"s_(branch|endpgm)", last) and i + 1 < len(blocks):
            to.append(i + 1)
        after.append(to)
    return blocks, after


def _in_cycles(after):
    """Blocks that can reach themselves (Tarjan, without recursion)."""
    index, low, on, stack, found, clock = {}, {}, set(), [], set(), 0
    for root in range(len(after)):
        if root in index:
            continue
        work = [(root, iter(after[root]))]
        index[root] = low[root] = clock = clock + 1
        stack.append(root), on.add(root)
        while work:
            v, rest = work[-1]
            for w in rest:
                if w not in index:
                    index[w] = low[w] = clock = clock + 1
                    stack.append(w), on.add(w)
                    work.append((w, iter(after[w])))
                    break
                if w in on:
                    low[v] = min(low[v], index[w])
            else:
                work.pop()
                if work:
                    low[work[-1][0]] = min(low[work[-1][0]], low[v])
                if low[v] == index[v]:
                    part = set()
                    while v not in part:
                        part.add(stack.pop())
                    on -= part
                    if len(part) > 1 or v in after[v]:
                        found |= part
    return found


def _pending_writes(lines):
    """(barriers in loops, those of them where an LDS write may be in flight).  A wave's LDS accesses complete in order: a write that `d` others have followed is
    done once at most d are to come.  Over all paths the smallest d counts."""
    blocks, after = _blocks(lines)
    cyclic = _in_cycles(after)

    def through(block, d, seen=None):
        for text in block:
            if re.match(r"ds_(write|store)", text):
                d = 0
            elif text.startswith("ds_"):
                d = min(d + 1, DONE)
            elif text.startswith("s_waitcnt"):
                m = re.search(r"lgkmcnt\((\d+)\)", text)
                if m and d >= int(m.group(1)):
                    d = DONE
            elif text.startswith("s_barrier") and seen is not None:
                seen.append(d)
        return d

    start = [DONE] * len(blocks)
    todo = list(range(len(blocks)))
    while todo:
        i = todo.pop()
        d = through(blocks[i], start[i])
        for j in after[i]:
            if d < start[j]:
                start[j] = d
                todo.append(j)
    seen = []
    for i in sorted(cyclic):
        through(blocks[i], start[i], seen)
    return len(seen), sum(d < DONE for d in seen)


def test_the_check_itself():
    loop = [".LBB0_1:", "s_waitcnt lgkmcnt(4)", "s_barrier", "ds_write_b128 v1, v2", "{}", "s_cbranch_scc1 .LBB0_1", "s_endpgm"]
    reads = lambda n: [t for line in loop for t in (["ds_read_b128 v[0:3], v9"] * n if line == "{}" else [line])]
    assert _pending_writes(reads(4)) == (1, 0) and _pending_writes(reads(3)) == (1, 1)
    assert _pending_writes(["ds_write_b32 v1, v2"] + reads(4)) == (1, 1)
    assert _pending_writes(["ds_write_b32 v1, v2", "s_waitcnt vmcnt(1) lgkmcnt(0)"] + reads(4)) == (1, 0)


@pytest.mark.skipif(not os.path.exists(HIPCC), reason="hipcc not available")
def test_no_lds_write_crosses_the_tile_loops_barrier(tmp_path):
    asm = tmp_path / "k.s"
    subprocess.run([HIPCC] + FLAGS + ["-S", "--cuda-device-only", os.path.join(ROOT, "bitstack_amd", "csrc", "tile.hip"), "-o", str(asm)], check=True, capture_output=True)
    kernels, name = {}, None
    for line in asm.read_text().splitlines():
        m = re.match(r"^(_Z\w+):", line)
        name = m.group(1) if m else None if line.startswith(".Lfunc_end") else name
        if name:
            kernels.setdefault(name, []).append(line)
    assert len(kernels) == 5, sorted(kernels)
    counts = {name: _pending_writes(lines) for name, lines in kernels.items()}
    print(counts)
    # one loop per width and number of blocks: 4 + 10 + 16 where everything fits, and with tokens one per width for the waves without columns
    assert max(loops for loops, _ in counts.values()) == 33 and min(loops for loops, _ in counts.values()) >= 16
    assert all(bad == 0 for _, bad in counts.values()), counts
