"""The assembly checks of test_build_resources.py and test_lds_waits.py for the kernels that neither of them builds: no scratch memory, and none of a wave's LDS writes on its way at the barrier
of the tile kernel's loop, in its builds for ranks below 16 too."""
import os
import re
import subprocess

import pytest

from test_build_resources import CSRC, FLAGS, HIPCC
from test_lds_waits import _pending_writes

SOURCES = ["tile.hip", "tile_ranks.hip", "tile_few_ranks.hip", "column.hip", "column_ranks.hip", "gemm_pipe.hip", "prefill_step.hip", "panel.hip", "gemv_sparse.hip"]


@pytest.fixture(scope="module")
def assembly(tmp_path_factory):
    """{source: assembly}, all compiled side by side."""
    if not os.path.exists(HIPCC):
        pytest.skip("hipcc not available")
    to = tmp_path_factory.mktemp("asm")
    runs = [(src, subprocess.Popen([HIPCC] + FLAGS + ["-w", "-S", "--cuda-device-only", os.path.join(CSRC, src), "-o", str(to / src)], stdout=subprocess.DEVNULL, stderr=subprocess.DEVNULL)) for src in SOURCES]
    assert [src for src, run in runs if run.wait() != 0] == []
    return {src: (to / src).read_text() for src in SOURCES}


@pytest.mark.parametrize("src", SOURCES)
def test_no_scratch_memory(src, assembly):
    sizes = [int(v) for v in re.findall(r"\.private_segment_fixed_size:\s+(\d+)", assembly[src])]
    assert sizes and max(sizes) == 0 and not re.search(r"^\s+scratch_(load|store)", assembly[src], re.M)


@pytest.mark.parametrize("src", ["tile_ranks.hip", "tile_few_ranks.hip"])
def test_no_lds_write_crosses_the_tile_loops_barrier(src, assembly):
    kernels, name = {}, None
    for line in assembly[src].splitlines():
        m = re.match(r"^(_Z\w+):", line)
        name = m.group(1) if m else None if line.startswith(".Lfunc_end") else name
        if name:
            kernels.setdefault(name, []).append(line)
    assert len(kernels) == 4, sorted(kernels)        # the rebuild and one to three token tiles
    counts = {name: _pending_writes(lines) for name, lines in kernels.items()}
    assert min(loops for loops, _ in counts.values()) >= 16 and all(bad == 0 for _, bad in counts.values()), counts
