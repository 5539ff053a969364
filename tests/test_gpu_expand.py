"""Expand and compaction from the probe's lists: block and tile edges, sparse
hits, guessed tables that do not fit, lineage; against the oracle (exact)."""
import numpy as np
import pytest

import oracle
from tests.conftest import VB
from wukonggpu_amd import Device, GStore, Triples

pytestmark = pytest.mark.gpu

SINGLE, DOZEN, HUB = VB, VB + 40000, VB + 90000  # subjects with 1 object, with 12, the one with 5000


@pytest.fixture(scope="module")
def graph():
    s = np.concatenate([SINGLE + np.arange(30000), np.repeat(DOZEN + np.arange(4000), 12), np.full(5000, HUB)])
    rng = np.random.default_rng(2)
    o = VB + rng.integers(0, 60000, len(s))
    o[-5000:] = VB + np.arange(5000)
    p = np.full(len(s), 2)
    gs = GStore.build(Triples.from_arrays(np.concatenate([s, s[:40000]]), np.concatenate([p, p[:40000] + 1]),
                                          np.concatenate([o, o[:40000] + 1])))
    dev = Device(0)
    dev.load(gs)
    yield gs, dev
    dev.close()


def _table(rng, rows, cols, hits, first, n):
    t = rng.integers(VB, VB + 60000, (rows, cols)).astype(np.int32)
    t[:, 0] = VB + 200000  # no edges
    at = np.sort(rng.choice(rows, size=hits, replace=False))
    t[at, 0] = first + rng.integers(0, n, hits)
    return t


CASES = [
    # rows, columns, rows with edges, their kind: (first, how many)
    (1, 1, 1, (HUB, 1)),
    (1024, 1, 1024, (SINGLE, 30000)),      # one block of output rows exactly
    (1025, 2, 1025, (SINGLE, 30000)),      # and one more
    (2500, 3, 2049, (SINGLE, 30000)),
    (600, 4, 600, (HUB, 1)),               # 3M rows: more than the guessed table
    (50000, 5, 40, (HUB, 1)),              # blocks inside one hit
    (524288, 1, 700, (SINGLE, 30000)),     # 2048 tiles, most of them empty: the largest of two launches
    (524289, 2, 524289, (DOZEN, 4000)),    # more than the guessed table, from every row
    (1048577, 1, 900, (SINGLE, 30000)),    # one tile too many, a block over hundreds of tiles
    (1200000, 2, 1200, (SINGLE, 30000)),   # a block over more tiles than it stages
    (1100000, 1, 1000000, (SINGLE, 30000)),
    (1100003, 3, 300000, (DOZEN, 4000)),   # fans out: from the lists, with lineage
    (1100003, 2, 150, (HUB, 1)),           # fans out more: by merge path
    (1100000, 2, 0, (SINGLE, 30000)),
    (1100000, 46, 330000, (DOZEN, 4000)),  # an input past the memory-side cache that fans out: by merge path
]


@pytest.mark.parametrize("rows,cols,hits,kind", CASES)
def test_steps(graph, rows, cols, hits, kind):
    gs, dev = graph
    rng = np.random.default_rng(rows + hits)
    tab = _table(rng, rows, cols, hits, *kind)
    dt = dev.table(tab)
    pre = [VB, 2, 1, -1]
    want, wex = oracle.run_step(gs, pre + [-1, 2, 1, -(cols + 1)], 1, tab, threads=8)
    t, ex = dev.k2u(dt, 0, 2, 1)
    assert ex == wex and np.array_equal(t.to_host(), want)
    # the next arm of a star from the same column (once per parent row where the table fans out and is
    # large), and a filter
    if len(want) < 8_000_000 and want.size:
        want2, wex2 = oracle.run_step(gs, pre + [-1, 3, 1, -(cols + 2)], 1, want, threads=8)
        dev.profile(True)
        got, ex2 = dev.k2u(t, 0, 3, 1)
        by_parents = dev.profile_read("lineage_steps")[2]
        dev.profile(False)
        assert ex2 == wex2 and np.array_equal(got.to_host().reshape(want2.shape), want2)
        assert by_parents == (len(want) >= 4 * hits and len(want) >= 1 << 19)
    want, wex = oracle.run_step(gs, pre + [-1, 2, 1, VB + 7], 1, tab, threads=8)
    f, ex = dev.k2c(dt, 0, 2, 1, VB + 7)
    assert ex == wex and np.array_equal(f.to_host(), want)
    if cols > 1:
        tab[: rows // 2, 1] = VB + 11
        dt = dev.table(tab)
        want, wex = oracle.run_step(gs, pre + [-1, 2, 1, -2], 1, tab, threads=8)
        f, ex = dev.k2k(dt, 0, 2, 1, 1)
        assert ex == wex and np.array_equal(f.to_host(), want)


@pytest.mark.parametrize("rows,hits", [(300, 1), (60000, 10), (60000, 0)])
def test_held_results_cost_their_size(graph, rows, hits):
    """A few hundred small results held at once take their own size of the
    table budget, whatever room their steps began with."""
    gs, _ = graph
    budget = 64 << 20
    dev = Device(0, table_budget_bytes=budget)
    try:
        dev.load(gs)
        tab = _table(np.random.default_rng(rows), rows, 2, hits, SINGLE, 30000)
        want, _ = oracle.run_step(gs, [VB, 2, 1, -1, -1, 2, 1, -3], 1, tab)
        dt = dev.table(tab)
        base = dev.pool_stats()["live_bytes"]
        held = [dev.k2u(dt, 0, 2, 1)[0] for _ in range(400)]
        assert dev.pool_stats()["live_bytes"] - base <= 400 * 4096 + budget // 256
        rest = (budget - base - 400 * 4096) // (2 << 20) * (2 << 20)  # large blocks are multiples of 2 MiB
        big = dev.table(np.zeros((rest // 4, 1), dtype=np.int32))  # the rest of the budget is there to use
        for t in held:
            assert np.array_equal(t.to_host().reshape(want.shape), want)
            t.free()
        big.free()
        t, _ = dev.k2u(dt, 0, 2, 1)
        assert np.array_equal(t.to_host().reshape(want.shape), want)
    finally:
        dev.close()
