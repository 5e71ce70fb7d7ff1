"""Transfers through the engine's pinned buffer at the sizes where its parts
begin and end: one site, parts of 16384 sites and one more, more sites than
the buffer holds (2^18), and energies of more systems than the buffer holds
for so few sites.  What goes in comes out bit for bit, and the device's planes
hold each site's own values: a rigid shift of one coordinate shows in that
coordinate alone, and energies of every system are those of the system alone."""
import numpy as np
import pytest

from molmodel_amd import waterbox as W
from molmodel_amd.engine import Engine

pytestmark = pytest.mark.gpu


def points(n):
    """n neutral points, one a group, in a large box: no pair within reach."""
    side = int(np.ceil(n ** (1 / 3)))
    L = 4.0 * max(side, 8)
    k = np.arange(n)
    r = 4.0 * np.stack([k % side, k // side % side, k // side ** 2], 1) + 1.0
    z, i = np.zeros(n), np.arange(n, dtype=np.int32)
    s = W.System(boxl=L, r=r, v=np.zeros((n, 3)), q=z, sig=z, eps=z,
                 site_mask=np.zeros(n, np.int32), mass=np.ones(n),
                 group=np.stack([i, i + 1], 1), excl=np.zeros((0, 2), np.int32))
    return s, dict(rc=3.0, smoothing_width=0.2, eta=1.0, kmode=2, mesh=(0, 0, 0), order=0, ik=0,
                   skin=0.2, nalias=0, include_lj_correction=0)


@pytest.mark.parametrize("n", [1, 16384, 16385, 262144, 262145])
def test_round_trip(gpu_lib, n):
    s, p = points(n)
    print("[stage] sites", n, flush=True)
    e = Engine(s, p)
    rng = np.random.default_rng(n)
    r = s.r + rng.uniform(-0.3, 0.3, (n, 3))
    v = rng.normal(size=(n, 3))
    e.set_positions(r)
    e.set_velocities(v)
    assert np.array_equal(e.positions(), r) and np.array_equal(e.velocities(), v)
    e.compute()
    assert not e.forces().any() and not e.potential().any()
    assert np.array_equal(e.positions(), r) and np.array_equal(e.velocities(), v)


def test_energies_of_many_small_systems(gpu_lib):
    s = W.subset(W.water_box(6, 18.64, 5), [0, 1, 40])
    p = dict(rc=9.0, smoothing_width=1.0, eta=0.35, kmode=2, mesh=(0, 0, 0), order=0, ik=0,
             skin=W.default_skin(9.0, 18.64), nalias=0, include_lj_correction=1)
    n = 150
    e, one = Engine([s] * n, [p] * n), Engine(s, p)
    r = [s.r + [0.001 * k, 0, 0] * (np.arange(s.nsite) < 3)[:, None] for k in range(n)]
    e.set_positions(np.concatenate(r))
    e.compute(virial=True)
    en, w = e.energies(), e.virial()
    for k in (0, 1, 74, 149):
        one.set_positions(r[k])
        one.compute(virial=True)
        assert np.array_equal(en[k][:4], one.energies()[0][:4])
        assert np.array_equal(w[k], one.virial()[0])
