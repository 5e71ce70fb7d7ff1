"""Small plain-Ewald engines build their neighbour list in the launches of the
reciprocal sum; with a P3M system beside them the two go separately.  Both ways
give a system the same list, forces, energies and virial bit for bit: through
rebuilds and steps without one, from one group to several blocks of the pair
search, with and without the sine table, for one system and several, and after
a position that is not finite."""
import numpy as np
import pytest

from molmodel_amd import waterbox as W
from molmodel_amd.engine import Engine

pytestmark = pytest.mark.gpu


def ewald(groups, kc, seed):
    s = W.water_box(6, 18.64, seed)
    p = dict(rc=8.0, smoothing_width=0.7, eta=0.35, kmode=0, kc=kc, mesh=(0, 0, 0), order=0, ik=0,
             skin=0.8, nalias=0, include_lj_correction=1)
    return W.subset(s, np.arange(groups)), p


def p3m():
    s = W.water_box(5, 18.64, 77)
    return s, dict(rc=8.0, smoothing_width=0.7, eta=0.35, kmode=1, mesh=(12, 12, 12), order=4, ik=0,
                   skin=0.8, nalias=2, include_lj_correction=1)


def same(a, b, n, nsys):
    for virial in (False, True):
        a.compute(virial=virial)
        b.compute(virial=virial)
        assert np.array_equal(a.forces(), b.forces()[:n])
        assert np.array_equal(a.energies()[:, :6], b.energies()[:nsys, :6])
        if virial:
            assert np.array_equal(a.virial(), b.virial()[:nsys])
    for k in range(nsys):
        assert np.array_equal(a.nl_pairs(k), b.nl_pairs(k))


@pytest.mark.parametrize("kc", [5.0, 33.0])
@pytest.mark.parametrize("groups", [(1,), (16,), (17,), (216,), (33, 1, 216)])
def test_with_and_without(gpu_lib, groups, kc):
    if kc > 31 and max(groups) > 17:
        pytest.skip("33^3 wave vectors only for the small ones")
    mem = [ewald(g, kc, 50 + k) for k, g in enumerate(groups)]
    print("[ewald list]", groups, kc, flush=True)
    ps, pp = p3m()
    a = Engine([m[0] for m in mem], [m[1] for m in mem])
    b = Engine([m[0] for m in mem] + [ps], [m[1] for m in mem] + [pp])
    r = np.concatenate([m[0].r for m in mem])
    n, rng = len(r), np.random.default_rng(4)
    first = np.zeros(n, int)
    at = 0
    for m in mem:                        # groups move as wholes
        for lo, hi in m[0].group:
            first[at + lo:at + hi] = at + lo
        at += m[0].nsite
    for shift in (0.0, 0.01, 1.5, 0.01, 3.0):
        r = r + shift * rng.uniform(-1, 1, r.shape)[first]
        a.set_positions(r)
        b.set_positions(np.concatenate([r, ps.r]))
        if shift < 1:
            same(a, b, n, len(mem))
        else:   # overlapping waters: the lists alone, past the force evaluation
            for k in range(len(mem)):
                assert np.array_equal(a.nl_pairs(k), b.nl_pairs(k))
    bad = r.copy()
    bad[0, 0] = np.nan
    a.set_positions(bad)
    with pytest.raises(Exception):
        a.compute()
    a.set_positions(np.concatenate([m[0].r for m in mem]))
    b.set_positions(np.concatenate([m[0].r for m in mem] + [ps.r]))
    same(a, b, n, len(mem))


def test_steps(gpu_lib):
    s, p = ewald(216, 6.0, 60)
    ps, pp = p3m()
    p = dict(p, skin=0.15)               # a rebuild every few steps
    pp = dict(pp, skin=0.15)
    a, c, b = Engine(s, p), Engine(ps, pp), Engine([s, ps], [p, pp])
    for e, q, v in ((a, s.r, s.v), (c, ps.r, ps.v), (b, np.concatenate([s.r, ps.r]), np.concatenate([s.v, ps.v]))):
        e.set_positions(q)
        e.set_velocities(v)
        e.md_setup(dt=0.001)
        for n in (1, 2, 25, 12):
            e.md_run(n)
    n = s.nsite
    print("[ewald list] builds", a.nl_builds(), c.nl_builds(), b.nl_builds(), flush=True)
    assert a.nl_builds() >= 3 and a.nl_builds() + c.nl_builds() == b.nl_builds()   # of all systems
    assert np.array_equal(a.positions(), b.positions()[:n])
    assert np.array_equal(a.velocities(), b.velocities()[:n])
    assert np.array_equal(a.energies()[0], b.energies()[0])
