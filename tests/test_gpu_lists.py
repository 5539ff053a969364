"""The fan-out filter through its lists: shared lists, repeated targets,
filter lists at the edges of the inline, long and chunked forms, many kept
rows; against the oracle's two steps (exact)."""
import numpy as np
import pytest

import oracle
from tests.conftest import VB
from wukonggpu_amd import STEP_K2C, STEP_K2K, Device, GStore, Triples

pytestmark = pytest.mark.gpu

ENTRIES = 3000  # of the longest list; entry i is vertex VB + 1000 + i
DEGREES = [0, 1, 1, 2, 3, 4, 5, 15, 16, 17, 18, 63, 0, 1, 0, 1, 2, 1, 1, 0]


@pytest.fixture(scope="module", params=[True, False], ids=["tags", "no tags"])
def graph(request):
    rng = np.random.default_rng(6)
    tri = []
    for h, n in enumerate((ENTRIES, 1500, 700, 300, 0, 40)):  # subject VB + h: a list of n entries
        e = VB + 1000 + np.sort(rng.choice(ENTRIES, size=n, replace=False))
        tri += [(VB + h, 2, x) for x in e]
    for i in range(ENTRIES):  # entry i's filter list
        d = DEGREES[i % len(DEGREES)]
        d = {40: 1023, 80: 1024, 120: 1025, 160: 2500}.get(i, d)
        tri += [(VB + 1000 + i, 3, VB + 10000 + x) for x in rng.choice(6000, size=d, replace=False)]
        if i % 2 == 0:
            tri.append((VB + 1000 + i, 4, VB + 10000))  # predicate 4: half of all entries, one object
    gs = GStore.build(Triples.from_arrays(*(np.array(x) for x in zip(*tri))))
    dev = Device(0)
    dev.load(gs, graph_budget_bytes=0 if request.param else gs.image_nbytes())  # (which leaves no room for tag words)
    dev.set_group_filter_rows(0)
    yield gs, dev
    dev.close()


# parents, distinct targets among them, filter predicate
@pytest.mark.parametrize("parents,targets,pid", [(513, 6000, 3), (2000, 300, 3), (5000, 1, 3), (3000, 50000, 3),
                                                 (700, 1, 4), (513, 1, 4), (100000, 6000, 3),
                                                 (2048, 1, 3), (2049, 2, 3), (4096, 5, 3)])
def test_fused_filter(graph, parents, targets, pid):
    gs, dev = graph
    rng = np.random.default_rng(parents + targets)
    tab = np.empty((parents, 3), dtype=np.int32)
    tab[:, 0] = VB + rng.choice(5, size=parents, p=[0.6, 0.2, 0.1, 0.05, 0.05])  # (VB + 4 has no list)
    tab[:, 1] = VB + 10000 + rng.integers(0, targets, parents)
    tab[rng.random(parents) < 0.01, 1] = -7
    tab[:, 2] = np.arange(parents)
    if parents == 100000:  # few rows keep anything
        tab[500:, 1] = VB + 20000
    pre, fan = [VB, 2, 1, -1], [-1, 2, 1, -4]
    mid, ex1 = oracle.run_step(gs, pre + fan, 1, tab, threads=8)
    dt = dev.table(tab)
    for kind, end, const in ((STEP_K2K, 1, -1), (STEP_K2C, -1, int(VB + 10000 + targets // 2)), (STEP_K2C, -1, 1 << 40)):
        tail = [-4, pid, 1, -2] if kind == STEP_K2K else [-4, pid, 1, const]
        if mid.shape[0] > 60_000_000 and kind == STEP_K2C:
            continue  # (the oracle's time)
        want, ex2 = oracle.run_step(gs, pre + tail, 1, mid, threads=8)
        out, fused, e1, e2 = dev.k2u_filter(dt, 0, 2, 1, kind, pid, 1, end, const)
        assert fused and (e1, e2) == (ex1, ex2)
        assert np.array_equal(out.to_host().reshape(want.shape), want)


@pytest.mark.parametrize("parents,subject", [(2000, VB + 5), (7000, VB + 1), (20000, VB + 2)])
def test_declined_before_any_launch(graph, parents, subject):
    """Short lists, and more parents than one workgroup should hash, go to the
    other forms without a launch of the list form."""
    gs, dev = graph
    tab = np.full((parents, 2), subject, dtype=np.int32)
    tab[:, 1] = VB + 10000 + np.arange(parents) % 6000
    mid, _ = oracle.run_step(gs, [VB, 2, 1, -1, -1, 2, 1, -3], 1, tab, threads=8)
    want, wex = oracle.run_step(gs, [VB, 2, 1, -1, -3, 3, 1, -2], 1, mid, threads=8)
    dt = dev.table(tab)
    launches = []
    try:
        for on in (True, False):
            dev.set_fanout_blocks(on)
            dev.profile(True)
            out, fused, _, ex = dev.k2u_filter(dt, 0, 2, 1, STEP_K2K, 3, 1, 1, -1)
            assert fused and ex == wex and np.array_equal(out.to_host().reshape(want.shape), want)
            launches.append(dev.profile_read("lineage")[0])
            dev.profile(False)
    finally:
        dev.set_fanout_blocks(True)
    assert launches[0] == launches[1]


@pytest.mark.parametrize("pid,parents,targets", [(3, 900, 400), (4, 700, 1)])
def test_kept_list_overflow(graph, pid, parents, targets):
    """Kept rows at the size of their list and one more: then they go through
    bits, from a written fan-out and from one that never was."""
    gs, dev = graph
    rng = np.random.default_rng(pid)
    tab = np.stack([VB + rng.integers(0, 4, parents), VB + 10000 + rng.integers(0, targets, parents)], axis=1)
    tab = tab.astype(np.int32)
    mid, _ = oracle.run_step(gs, [VB, 2, 1, -1, -1, 2, 1, -3], 1, tab, threads=8)
    want, wex = oracle.run_step(gs, [VB, 2, 1, -1, -3, pid, 1, -2], 1, mid, threads=8)
    kept = want.shape[0]
    dt = dev.table(tab)
    wide, _ = dev.k2u(dt, 0, 2, 1)
    try:
        for cap, over in ((kept, kept > 32768), (kept - 1, True), (1, True)):
            dev.set_fanout_blocks(True, cap)
            dev.profile(True)
            out, fused, _, ex = dev.k2u_filter(dt, 0, 2, 1, STEP_K2K, pid, 1, 1, -1)
            assert fused and ex == wex and np.array_equal(out.to_host().reshape(want.shape), want)
            out, ex = dev.k2k(wide, 2, pid, 1, 1)
            assert ex == wex and np.array_equal(out.to_host().reshape(want.shape), want)
            out, ex = dev.k2c(wide, 2, pid, 1, VB + 10000)
            c, cex = oracle.run_step(gs, [VB, 2, 1, -1, -3, pid, 1, VB + 10000], 1, mid, threads=8)
            assert ex == cex and np.array_equal(out.to_host().reshape(c.shape), c)
            assert dev.profile_read("fanout_filters")[2] == 3  # each by one form alone
            assert dev.profile_read("fanout_kept_overflow")[2] == 2 * over + (c.shape[0] > min(cap, 32768))
            dev.profile(False)
    finally:
        dev.set_fanout_blocks(True)
