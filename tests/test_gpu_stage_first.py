"""The first positions handed to a new engine cost what later ones do: the
pinned buffer has its pages when the engine is made, so the call's own thread
takes no page fault in it (its first write to a fresh buffer of this size
takes one per large page).  The least of three engines, since the runtime may
fault once for its own purposes."""
import resource

import numpy as np
import pytest

from molmodel_amd.engine import Engine
from test_gpu_stage import points

pytestmark = pytest.mark.gpu


def faults():
    return resource.getrusage(resource.RUSAGE_THREAD).ru_minflt


def test_first_positions_fault_no_pages(gpu_lib):
    s, p = points(98304)
    r = np.ascontiguousarray(s.r)
    warm = Engine(s, p)
    warm.set_positions(r)
    n, kept = [], []
    for _ in range(3):
        e = Engine(s, p)
        a = faults()
        e.set_positions(r)
        n.append(faults() - a)
        kept.append(e)   # its buffer is not the next engine's
    print("[stage first] page faults", n)
    assert min(n) == 0
