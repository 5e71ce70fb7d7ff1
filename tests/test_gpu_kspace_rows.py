"""The plain Ewald sum at the edges of its kernels' shape: site counts around
the field kernel's 16-site blocks, cutoffs around the structure factors'
eight |nz| per block, fractional cutoffs, more rows than one pass of teams,
wave vectors beyond the field kernel's factor table, and a triclinic cell.

kspace_field (the reference-named drop-in) against the sums written out in
numpy FP64; the kernels are FP64 throughout, so the bar is the repository's
for this path, 1e-11 of the norm (a sum over up to 2e4 wave vectors of terms
good to a few units in the last place of arguments below 1e3)."""
import ctypes as C

import numpy as np
import pytest

from molmodel_amd import engine as E

pytestmark = pytest.mark.gpu
P, D, I = C.c_void_p, C.c_double, C.c_int


def vectors(kc):
    nm = int(np.floor(kc))
    a = np.arange(-nm, nm + 1)
    n = np.stack(np.meshgrid(a, a, a, indexing="ij"), -1).reshape(-1, 3)
    half = (n[:, 0] > 0) | ((n[:, 0] == 0) & ((n[:, 1] > 0) | ((n[:, 1] == 0) & (n[:, 2] > 0))))
    return n[half & ((n * n).sum(1) <= kc * kc + 1e-8)].astype(float)


def direct(r, q, b, V, eta, kc):
    k = vectors(kc) @ b                     # rows of b: reciprocal vectors
    k2 = (k * k).sum(1)
    a = 4 * np.pi / V * np.exp(-k2 / (4 * eta * eta)) / k2
    s, c = np.sin(r @ k.T), np.cos(r @ k.T)
    S, Cc = q @ s, q @ c
    return s @ (2 * a * S) + c @ (2 * a * Cc), (2 * a * (s * Cc - c * S)) @ k


@pytest.mark.parametrize("nsite,kc,tri", [(1, 1.0, 0), (15, 6.0, 1), (16, 7.0, 0), (17, 7.5, 1),
                                          (300, 8.0, 0), (257, 12.0, 1), (5, 17.3, 0),
                                          (3, 21.0, 1), (2, 32.5, 0)])
def test_kspace_field_matches_the_sums(gpu_lib, nsite, kc, tri):
    L = E.lib()
    L.kspace_new.restype = P
    L.kspace_new.argtypes = [D, I]
    L.kspace_field.restype = None
    L.kspace_field.argtypes = [P, P, P, P, D, D, P, P]
    L.kspace_delete.argtypes = [P]
    rng = np.random.default_rng(nsite)
    A = np.diag([18.0, 18.0, 18.0])         # rows: lattice vectors
    if tri:
        A = np.array([[18.0, 0.5, 0.0], [2.0, 17.0, 1.0], [-1.0, 3.0, 19.0]])
    b = 2 * np.pi * np.linalg.inv(A).T
    V = abs(np.linalg.det(A))
    r = rng.uniform(-20, 40, (nsite, 3))
    q = rng.normal(0, 5, nsite)
    eta = 0.35
    phi, ev = np.zeros(nsite), np.zeros((nsite, 3))
    p = lambda a: a.ctypes.data_as(P)
    latv = np.ascontiguousarray(b).reshape(-1)      # tensor_t: column vectors in turn
    print(f"[kspace rows] {nsite} {kc} {tri}", flush=True)
    k = L.kspace_new(kc, nsite)
    L.kspace_field(k, p(r), p(q), p(latv), V, eta, p(phi), p(ev))
    L.kspace_delete(k)
    rphi, rev = direct(r, q, b, V, eta, kc)
    assert np.linalg.norm(phi - rphi) <= 1e-11 * np.linalg.norm(rphi)
    # one site alone feels no field: compare against the size of its terms
    scale = max(np.linalg.norm(rev), np.abs(q).max() / 18.0 ** 2)
    assert np.linalg.norm(ev - rev) <= 1e-11 * scale
