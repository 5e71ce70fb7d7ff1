"""Blocks that hand results to the last block of their launch: a barrier waits
for no memory, so every wavefront has to wait for its own atomics before the
barrier that precedes the counter.  A timing in which one is missing cannot be
forced, so the test reads the assembly that the build's flags give: behind
each count of k_nl_assign there is a wait for all of the wavefront's memory
operations before the next barrier.  Nothing here runs on a GPU."""
import os
import re
import subprocess

import pytest

from molmodel_amd import build as B


def kernel_lines(source, name, out):
    cmd = [B.HIPCC] + B.COMMON + B.EXTRA.get(source, []) + ["--cuda-device-only", "-S", os.path.join(B.CSRC, source), "-o", out]
    p = subprocess.run(cmd, capture_output=True, text=True, timeout=300)
    assert p.returncode == 0, p.stderr
    text = open(out).read()
    body = re.search(rf"^_ZN5mmamd\d+{name}E\w*:[^\n]*\n(.*?)\.Lfunc_end", text, re.M | re.S)
    assert body, name
    return [l.split(";")[0].strip() for l in body.group(1).splitlines()]


def test_counts_are_waited_for(tmp_path):
    if not os.path.exists(B.HIPCC):
        pytest.skip("hipcc not present")
    lines = kernel_lines("nbrlist.hip", "k_nl_assign", str(tmp_path / "nbrlist.s"))
    counts = [i for i, l in enumerate(lines) if l.startswith("global_atomic_add") and "sc0" not in l]
    assert counts
    for i in counts:
        after = lines[i:lines.index("s_barrier", i)]
        assert any(l.startswith("s_waitcnt") and "vmcnt(0)" in l for l in after), after
