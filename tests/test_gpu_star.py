"""A star arm over few rows that fans out far, then a filter on its new column:
decided once per group of the arm's parents whatever the arm's input size;
against the oracle (exact)."""
import numpy as np
import pytest

import oracle
from tests.conftest import VB
from wukonggpu_amd import Device, GStore, Triples

pytestmark = pytest.mark.gpu

SUBJECTS, FAN = 60, 200  # subjects VB + i: FAN objects by predicate 2, 15 by 3, 100 by 4


@pytest.fixture(scope="module")
def graph():
    rng = np.random.default_rng(4)
    s = VB + np.arange(SUBJECTS)
    tri = []
    for p, d in ((2, FAN), (3, 15), (4, 100)):
        o = np.concatenate([rng.choice(5000, size=d, replace=False) for _ in s])
        tri.append((np.repeat(s, d), np.full(SUBJECTS * d, p), VB + 1000 + o))
    es = np.repeat(VB + 1000 + np.arange(5000), 2)
    tri.append((es, np.full(len(es), 5), VB + 10000 + rng.integers(0, 3000, len(es))))
    gs = GStore.build(Triples.from_arrays(*(np.concatenate(x) for x in zip(*tri))))
    dev = Device(0)
    dev.load(gs)
    yield gs, dev
    dev.close()


# rows before the first arm (FAN times as many after it), second arm's predicate, whether its output
# (15 or 100 times as many again) has the 2^22 rows from which filters go by groups
@pytest.mark.parametrize("rows,pid,groups", [(300, 4, True), (300, 3, False), (700, 4, True), (700, 3, False)])
def test_filter_after_star_arm(graph, rows, pid, groups):
    gs, dev = graph
    rng = np.random.default_rng(rows + pid)
    tab = np.stack([VB + rng.integers(0, SUBJECTS, rows), VB + 10000 + rng.integers(0, 3000, rows)], axis=1)
    tab = tab.astype(np.int32)
    t0 = dev.table(tab)
    t1, _ = dev.k2u(t0, 0, 2, 1)
    assert t1.shape[0] == rows * FAN
    pre = [VB, 2, 1, -1]
    mid, _ = oracle.run_step(gs, pre + [-1, 2, 1, -3], 1, tab, threads=8)
    wide, wex = oracle.run_step(gs, pre + [-1, pid, 1, -4], 1, mid, threads=8)
    assert (wide.shape[0] >= 1 << 22) == groups
    t2, ex = dev.k2u(t1, 0, pid, 1)
    assert ex == wex and np.array_equal(t2.to_host(), wide)
    dev.profile(True)
    try:
        f, ex = dev.k2k(t2, 3, 5, 1, 1)
        want, wex = oracle.run_step(gs, pre + [-4, 5, 1, -2], 1, wide, threads=8)
        assert ex == wex and np.array_equal(f.to_host(), want)
        f, ex = dev.k2c(t2, 3, 5, 1, VB + 10007)
        want, wex = oracle.run_step(gs, pre + [-4, 5, 1, VB + 10007], 1, wide, threads=8)
        assert ex == wex and np.array_equal(f.to_host(), want)
        assert dev.profile_read("lineage_filters")[2] == (2 if groups else 0)
    finally:
        dev.profile(False)
