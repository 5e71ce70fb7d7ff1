"""A pulling block transforms its own z lines where its columns come in pairs
and fit its LDS; elsewhere, and for spreading by owner, a pass of its own does.
On both sides of that rule (an even and an odd number of y columns on the mesh
and in a block, 2048 points a block and more, two systems that differ in it)
the mesh, and with it potential, field and energy, are the same bit for bit."""
import numpy as np
import pytest

from molmodel_amd import waterbox as W
from molmodel_amd.engine import Engine

pytestmark = pytest.mark.gpu


def par(mesh, ik):
    return dict(rc=9.0, smoothing_width=1.0, eta=0.35, kmode=1, mesh=mesh, order=5, ik=ik,
                skin=W.default_skin(9.0, 18.64), nalias=2, include_lj_correction=1)


@pytest.mark.parametrize("ik", [0, 1])
@pytest.mark.parametrize("meshes", [[(16, 16, 32)], [(16, 16, 36)], [(12, 15, 20)], [(9, 16, 128)],
                                    [(16, 16, 32), (16, 15, 35)]])
def test_every_form_gives_one_mesh(gpu_lib, meshes, ik):
    s = W.subset(W.water_box(6, 18.64, 9), np.arange(0, 216, 2))
    print("[spread lines]", meshes, ik, flush=True)
    first = None
    for halo in (1, 0):
        for block in (1, 2, 4, 8):
            e = Engine([s] * len(meshes), [par(m, ik) for m in meshes],
                       shape=dict(spread_halo=halo, spread_block=block))
            e.set_positions(np.concatenate([s.r] * len(meshes)))
            phi, ev = e.kspace_field()
            now = phi, ev, e.energies()[:, :6]
            if first is None:
                first = now
            for a, b in zip(now, first):
                assert np.array_equal(a, b), (halo, block)
