"""A standalone neighbour list after positions that its build reports, on both
sides of the rule that chooses the build (one block up to 8 192 points, the
cells' lists beyond): a collapse onto one point and a non-finite coordinate.

The same positions are reported again, not taken for a list that is still
good; no rows come out meanwhile; and when only the points at fault come back,
the update rebuilds and the pair set is the oracle's."""
import numpy as np
import pytest

from test_gpu_nlist import P, lib, new_list
from test_gpu_nlist_sizes import oracle_pairs, pairs_of

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kind", ["collapse", "nan"])
@pytest.mark.parametrize("n", [3000, 10000])
@pytest.mark.parametrize("first,calls", [(True, 1), (False, 1), (False, 2)])
def test_reported_then_rebuilt(gpu_lib, n, kind, first, calls):
    L = lib()
    rng = np.random.default_rng(n)
    boxl, rc, skin = 5.0 * n ** (1 / 3), 5.5, 1.0
    good = rng.uniform(0, boxl, (n, 3))
    bad = good.copy()
    if kind == "collapse":
        bad[n - 1000:] = 0.0
    else:
        bad[n - 1, 2] = np.nan
    print(f"[nlist errors] {n} {kind} first {first}", flush=True)
    h = new_list(L, n, rc, skin, boxl)
    ptr = lambda x: x.ctypes.data_as(P)
    if not first:
        assert L.mm_nlist_update(h, ptr(good)) == 1
    for _ in range(calls):
        assert L.mm_nlist_update(h, ptr(bad)) < 0
        assert L.mm_nlist_rows(h, None, None, 0) <= 0
    assert L.mm_nlist_update(h, ptr(good)) == 1
    assert np.array_equal(pairs_of(L, h, n), oracle_pairs(good, boxl, rc, skin))
    assert L.mm_nlist_update(h, ptr(good)) == 0
    L.mm_nlist_destroy(h)
