"""The neighbour-list build on both sides of its rule: systems built by one
block (up to 8 192 groups) and larger ones built from cell lists, group counts
around the block's thread count, cells above and below the size that is sorted
in registers, and boxes whose groups lie in a few cells.

The pair set and each pair's PairBinary row against the oracle's build, which
reproduces the reference's; a second update with the same positions must keep
the list, and a third with moved ones must rebuild it."""
import ctypes as C

import numpy as np
import pytest

import oracle_lib as O
from test_gpu_nlist import P, lib, new_list

pytestmark = pytest.mark.gpu


def pairs_of(L, h, n):
    m = L.mm_nlist_rows(h, None, None, 0)
    assert m >= 0, L.mm_last_error()
    start, cols = np.zeros(n + 1, dtype=np.int32), np.zeros(max(m, 1), dtype=np.int32)
    L.mm_nlist_rows(h, start.ctypes.data_as(P), cols.ctypes.data_as(P), m)
    rows = np.repeat(np.arange(n, dtype=np.int64), np.diff(start))
    return np.sort(rows * (1 << 32) + cols[:m])


def oracle_pairs(x, boxl, rc, skin):
    p = np.asarray(O.nl_pairs(x, boxl, rc, skin), dtype=np.int64).reshape(-1, 2)
    return np.sort(p[:, 0] * (1 << 32) + p[:, 1])


@pytest.mark.parametrize("n,clumps", [(2, 0), (63, 0), (1023, 0), (1024, 0), (1025, 3), (4097, 40),
                                      (8192, 0), (8193, 0), (9001, 60), (35200, 0)])
def test_pair_set(gpu_lib, n, clumps):
    L = lib()
    rng = np.random.default_rng(n)
    boxl = 5.0 * max(n, 30) ** (1 / 3)
    rc, skin = min(5.5, 0.4 * boxl), min(1.0, 0.05 * boxl)
    x = rng.uniform(-0.3 * boxl, 1.3 * boxl, (n, 3))
    if clumps:   # cells of about 15 groups
        c = rng.uniform(0, boxl, (clumps, 3))
        x[:15 * clumps] = np.repeat(c, 15, axis=0) + rng.normal(0, 0.12, (15 * clumps, 3))
    x = np.ascontiguousarray(x)
    print(f"[nlist sizes] n {n} clumps {clumps}", flush=True)
    h = new_list(L, n, rc, skin, boxl)
    assert L.mm_nlist_update(h, x.ctypes.data_as(P)) == 1
    assert np.array_equal(pairs_of(L, h, n), oracle_pairs(x, boxl, rc, skin))
    assert L.mm_nlist_update(h, x.ctypes.data_as(P)) == 0
    y = np.ascontiguousarray(x + rng.uniform(-skin, skin, (n, 3)))
    assert L.mm_nlist_update(h, y.ctypes.data_as(P)) == 1
    assert np.array_equal(pairs_of(L, h, n), oracle_pairs(y, boxl, rc, skin))
    L.mm_nlist_destroy(h)
