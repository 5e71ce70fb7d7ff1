"""Charge spreading at the edges of its two forms: every assignment order,
column blocks from one column to eight, blocks whose columns wrap round the
mesh, and charges on both sides of the bound up to which contributions take
the short fixed-point conversion (2^18 internal charge units).

Both forms accumulate exact integers of the same FP32 products, so every
shape gives the same mesh, and the field read back from it is compared bit
for bit; one shape is compared with the FP64 oracle at the repository's bar
for the mesh (1e-5 relative)."""
import numpy as np
import pytest

import oracle_lib as O
from molmodel_amd import waterbox as W
from molmodel_amd.engine import Engine

pytestmark = pytest.mark.gpu


def rel(a, b):
    return float(np.linalg.norm(np.asarray(a) - np.asarray(b)) / np.linalg.norm(b))


@pytest.mark.parametrize("order", [2, 3, 4, 5, 6, 7])
@pytest.mark.parametrize("big", [1.0, 2.6e5, 2.7e5])
def test_all_shapes_give_one_mesh(gpu_lib, order, big):
    s = W.subset(W.water_box(6, 18.64, 3), np.arange(0, 216, 3))
    s.q = s.q / np.abs(s.q).max()
    s.q[::7] *= big                       # 2^18 = 262144 lies between the two
    p = dict(rc=9.0, smoothing_width=1.0, eta=0.35, kmode=1, mesh=(8, 16, 20), order=order, ik=0,
             skin=W.default_skin(9.0, 18.64), nalias=2, include_lj_correction=1)
    print(f"[spread] order {order} largest charge {np.abs(s.q).max():.4g}", flush=True)
    first = None
    for halo in (0, 1):
        for block in (1, 2, 4, 8):
            e = Engine(s, p, shape=dict(spread_halo=halo, spread_block=block))
            e.set_positions(s.r)
            phi, ev = e.kspace_field()
            if first is None:
                first = phi, ev
                ophi, oev, _, _ = O.p3m_parts(s, p)
                assert rel(phi, ophi) <= 1e-5 and rel(ev, oev) <= 1e-5
            assert np.array_equal(phi, first[0]) and np.array_equal(ev, first[1]), (halo, block)
