"""Where handed-in positions land on the device, at the edges of the transfer's
parts (16384 sites) and of the buffer (2^18): reading them back cannot tell,
since the way out undoes the way in.  Here a few Lennard-Jones pairs lie on
either side of each edge, each with a displacement of its own along x, y and
z, among sites that interact with nothing.  The forces are those of a small
engine that holds the pairs alone; the
same FP32 terms, so 1e-5 of the largest force is ample, and every other site's
force is zero."""
import numpy as np
import pytest

from molmodel_amd import waterbox as W
from molmodel_amd.engine import Engine
from test_gpu_stage import points

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [16385, 262145])
def test_planes_at_part_edges(gpu_lib, n):
    s, p = points(n)
    second = np.unique([b for b in (1, 8192, 16384, 16385 + 16384, 131072, 262144, n - 1) if b < n])
    at = np.sort(np.concatenate([second - 1, second]))
    for k, b in enumerate(second):
        s.r[b] = s.r[b - 1] + [1.10 + 0.02 * k, 0.31 - 0.03 * k, -0.17 - 0.04 * k]
    s.site_mask[at] = W.SITE_HAS_LJ
    s.sig, s.eps = s.sig.copy(), s.eps.copy()   # points() shares one array
    s.sig[at], s.eps[at] = 1.1, 0.2
    print("[stage layout] sites", n, "pairs", len(second), flush=True)
    e = Engine(s, p)
    e.set_positions(s.r)
    e.compute()
    f = e.forces()
    i = np.arange(len(at), dtype=np.int32)
    few = W.System(boxl=s.boxl, r=s.r[at], v=s.v[at], q=s.q[at], sig=s.sig[at], eps=s.eps[at],
                   site_mask=s.site_mask[at], mass=s.mass[at], group=np.stack([i, i + 1], 1),
                   excl=np.zeros((0, 2), np.int32))
    one = Engine(few, p)
    one.set_positions(few.r)
    one.compute()
    ref = one.forces()
    assert (np.abs(ref).max(1) > 0.01).all()
    assert np.abs(f[at] - ref).max() <= 1e-5 * np.abs(ref).max()
    f[at] = 0
    assert not f.any()
