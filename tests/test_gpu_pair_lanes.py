"""The pair kernel gives a group a whole wavefront in engines of up to 2048
groups and 16 lanes in larger ones.  Both add a group's pairs in one order,
so a system alone equals, bit for bit, the same system in an engine beyond
the line, in every variant of the kernel: forces with and without energies,
virial, field; waters, ions and groups of two sites; rows shorter than a
batch and rows of several."""
from dataclasses import replace

import numpy as np
import pytest

from molmodel_amd import waterbox as W
from molmodel_amd.engine import Engine

pytestmark = pytest.mark.gpu


def par(rc, boxl):
    return dict(rc=rc, smoothing_width=0.8, eta=0.33, kmode=1, mesh=(16, 16, 16), order=4, ik=0,
                skin=W.default_skin(rc, boxl), nalias=2, include_lj_correction=1)


def member(kind):
    s = W.water_box(6, 18.64, 41)
    if kind == "waters":
        return s, par(9.0, 18.64)
    if kind == "sparse":        # a few waters, rows of fewer than 16 neighbours
        return W.subset(s, np.arange(0, 216, 11)), par(9.0, 18.64)
    # ions, and every third water without its last site
    s = W.water_box(6, 18.64, 41, ions=(5, 5))
    keep = np.ones(s.nsite, bool)
    keep[s.group[0:216:3, 1] - 1] = False
    new = np.cumsum(keep) - 1
    first = new[s.group[:, 0]]
    group = np.stack([first, np.append(first[1:], keep.sum())], 1).astype(np.int32)
    ex = s.excl[keep[s.excl].all(1)]
    return replace(s, r=s.r[keep], v=s.v[keep], q=s.q[keep], sig=s.sig[keep], eps=s.eps[keep],
                   site_mask=s.site_mask[keep], mass=s.mass[keep], group=group,
                   excl=new[ex].astype(np.int32)), par(9.0, 18.64)


@pytest.mark.parametrize("kind", ["waters", "sparse", "mixed"])
def test_one_wavefront_equals_sixteen_lanes(gpu_lib, kind):
    s, p = member(kind)
    fs, fp = W.water_box(13, 40.39, 42), par(9.0, 40.39)     # 2197 groups: beyond the line
    print("[pair lanes]", kind, "sites", s.nsite, flush=True)
    one, two = Engine(s, p), Engine([s, fs], [p, fp])
    n = s.nsite
    one.set_positions(s.r)
    two.set_positions(np.concatenate([s.r, fs.r]))
    for virial in (False, True):
        one.compute(virial=virial)
        two.compute(virial=virial)
        assert np.array_equal(one.forces(), two.forces()[:n])
        assert np.array_equal(one.energies()[0][:4], two.energies()[0][:4])
        if virial:
            assert np.array_equal(one.virial()[0], two.virial()[0])
    for a, b in zip(one.rspace_field()[:3], two.rspace_field()[:3]):
        assert np.array_equal(a, b[:n])
    if kind != "mixed":                  # forces without energies: inside steps of dynamics
        for e, r, v in ((one, s.r, s.v), (two, np.concatenate([s.r, fs.r]), np.concatenate([s.v, fs.v]))):
            e.set_positions(r)
            e.set_velocities(v)
            e.md_setup(dt=0.001)
            e.md_run(3)
        assert np.array_equal(one.positions(), two.positions()[:n])
