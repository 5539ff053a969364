"""Edges of the filters' list search on the GPU, against the oracle (exact:
ids and work counts)."""
import numpy as np
import pytest

import oracle
from tests.conftest import VB
from wukonggpu_amd import Device, GStore, Triples

pytestmark = pytest.mark.gpu

LENGTHS = [1, 2, 3, 4, 5, 6, 7, 8, 9, 12, 13, 15, 16, 17, 20, 21, 63, 64, 65, 255, 256, 257, 1000, 4099]


@pytest.fixture(scope="module")
def lists():
    """Subject VB + i has LENGTHS[i] even objects, spread unevenly."""
    rng = np.random.default_rng(3)
    s, o = [], []
    for i, n in enumerate(LENGTHS):
        objs = VB + 2 * np.sort(rng.choice(20000, size=n, replace=False))
        s += [VB + i] * n
        o += objs.tolist()
    p = [2] * len(s)
    gs = GStore.build(Triples.from_arrays(s, p, o))
    return gs, np.array(s), np.array(o)


@pytest.mark.parametrize("sorted_lists", [True, False])
def test_every_entry_and_every_gap(lists, sorted_lists):
    """Each list's entries, their neighbours, both ends' outsides and negative
    cells as the end cell; and one constant against every list."""
    gs, s, o = lists
    dev = Device(0)
    dev.load(gs, sorted_lists=sorted_lists)
    ends = np.concatenate([o, o - 1, o + 1, np.full(len(s), VB - 2), np.full(len(s), VB + 50000),
                           np.full(len(s), -3)])
    tab = np.stack([np.tile(s, 6), ends], axis=1).astype(np.int32)
    tab = tab[np.random.default_rng(4).permutation(len(tab))]
    t, ex = dev.k2k(dev.table(tab), 0, 2, 1, 1)
    want, wex = oracle.run_step(gs, [VB, 2, 1, -1, -1, 2, 1, -2], 1, tab)
    assert ex == wex and np.array_equal(t.to_host(), want)
    for const in (int(o[0]), int(o[-1]), int(o[len(o) // 2]), VB + 1):
        t, ex = dev.k2c(dev.table(tab), 0, 2, 1, const)
        want, wex = oracle.run_step(gs, [VB, 2, 1, -1, -1, 2, 1, const], 1, tab)
        assert ex == wex and np.array_equal(t.to_host(), want)
    dev.close()
