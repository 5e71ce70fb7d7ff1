"""The mesh transforms over the radices, sizes and shapes they take apart:
every radix from 2 to 10 as first and last stage, one to three stages, odd
line counts (the last mesh line has no partner), meshes whose kz planes are
transformed in one block and larger ones that take a pass per axis, and
batches that mix both, with real-space differentiation and with the field on
the mesh.

The field of one system against the FP64 oracle's P3M; the bars are the
repository's for it (phi and field 1e-5 relative, virial 1e-5: FP32 mesh
arithmetic)."""
import numpy as np
import pytest

import oracle_lib as O
from molmodel_amd import waterbox as W
from molmodel_amd.engine import Engine

pytestmark = pytest.mark.gpu


def rel(a, b):
    return float(np.linalg.norm(np.asarray(a) - np.asarray(b)) / np.linalg.norm(b))


def case(mesh, order, ik, seed=5):
    s = W.subset(W.water_box(5, 24.0, seed), np.arange(0, 125, 2))
    p = dict(rc=9.0, smoothing_width=1.0, eta=0.3, kmode=1, mesh=mesh, order=order, ik=ik,
             skin=W.default_skin(9.0, 24.0), nalias=2, include_lj_correction=1)
    return s, p


MESHES = [(8, 9, 10), (10, 8, 9), (12, 14, 15), (16, 18, 20), (21, 24, 25), (27, 28, 30),
          (32, 35, 36), (40, 42, 45), (49, 50, 54), (56, 63, 48), (64, 64, 64), (72, 75, 16),
          (81, 60, 20), (90, 80, 12), (100, 98, 16), (16, 125, 126), (128, 40, 105), (8, 112, 128)]


@pytest.mark.parametrize("mesh", MESHES, ids=lambda m: "x".join(map(str, m)))
@pytest.mark.parametrize("ik", [0, 1])
def test_field_matches_oracle(gpu_lib, mesh, ik):
    s, p = case(mesh, 3 + sum(mesh) % 4, ik)
    print(f"[meshes] {mesh} order {p['order']} ik {ik}", flush=True)
    e = Engine(s, p)
    e.set_positions(s.r)
    phi, ev = e.kspace_field()
    ophi, oev, _, _ = O.p3m_parts(s, p)
    assert rel(phi, ophi) <= 1e-5 and rel(ev, oev) <= 1e-5


@pytest.mark.parametrize("mesh,ik", [((45, 42, 49), 0), ((45, 42, 49), 1), ((80, 96, 24), 0),
                                     ((80, 96, 24), 1)])
def test_virial_and_forces_only_steps(gpu_lib, mesh, ik):
    s, p = case(mesh, 5, ik)
    print(f"[meshes] virial {mesh} ik {ik}", flush=True)
    e = Engine(s, p)
    e.set_positions(s.r)
    e.compute(virial=True)
    f, en, w = e.forces(), e.energies()[0], e.virial()[0]
    of, oen, ow = O.evaluate(s, p, virial=True)
    assert rel(f, of) <= 1e-5
    assert abs(en[0] - oen[0]) <= 1e-5 * abs(oen[3])
    assert rel(w, ow.reshape(3, 3)) <= 1e-5


def test_batch_of_one_block_planes_and_passes(gpu_lib):
    """Systems of both kinds in one engine give what engines of their own
    give, bit for bit."""
    mem = [case((80, 96, 24), 5, 0), case((45, 42, 49), 4, 1, 6), case((30, 30, 30), 6, 0, 7)]
    e = Engine([m[0] for m in mem], [m[1] for m in mem])
    e.set_positions(np.concatenate([m[0].r for m in mem]))
    e.compute()
    f = e.forces()
    for k, (s, p) in enumerate(mem):
        one = Engine(s, p)
        one.set_positions(s.r)
        one.compute()
        assert np.array_equal(f[e.offsets[k]:e.offsets[k + 1]], one.forces()), k
