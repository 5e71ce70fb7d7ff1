"""The adjoint's pair pass at the edges of its shape: neighbour rows shorter
than one 64-lane batch, exactly on and just past its multiples, one LJ type
and the most a system may hold, groups of one and three sites.

The gradients are checked against the basis of forward evaluations
(mm_param_gradients_basis), with the bars test_gpu_adjoint.py derives for
that comparison: 1e-5 of the largest energy gradient of its kind and 2e-4 of
the largest loss gradient."""
import numpy as np
import pytest

from molmodel_amd import waterbox as W
from molmodel_amd.engine import Engine

pytestmark = pytest.mark.gpu


def case(n, ngroup, ntype):
    s, p = W.config(f"water{n}_small")
    if ngroup < s.ngroup:
        s = W.subset(s, np.arange(ngroup))
    for t in range(1, ntype):   # every ntype-th molecule a type of its own
        s.sig[3 * t::3 * ntype] *= 1 + 0.01 * t
        s.eps[3 * t::3 * ntype] *= 1 + 0.03 * t
        s.q[3 * t::3 * ntype] *= 1 + 0.005 * t
    return s, p


@pytest.mark.parametrize("n,ngroup,ntype", [(27, 27, 1), (64, 64, 1), (125, 65, 2), (125, 66, 1),
                                            (216, 129, 3), (216, 130, 8), (512, 512, 8)])
def test_gradients_match_basis(gpu_lib, n, ngroup, ntype):
    s, p = case(n, ngroup, ntype)
    f_ref = np.random.default_rng(n + ngroup).normal(0.0, 10.0, s.r.shape)
    e = Engine(s, p)
    e.set_positions(s.r)
    print(f"[adjoint rows] {n} {ngroup} {ntype}", flush=True)
    g = e.param_gradients(0, f_ref=f_ref, maxtypes=24)
    b = e.param_gradients(0, f_ref=f_ref, maxtypes=24, basis=True)
    assert g["ntype"] == b["ntype"]
    for name, tol in (("dE", 1e-5), ("dL", 2e-4)):
        for c in range(3):
            scale = np.abs(b[name][:, c]).max()
            assert np.abs(g[name][:, c] - b[name][:, c]).max() <= tol * scale, (name, c)
