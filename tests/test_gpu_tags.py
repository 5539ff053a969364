"""The probe's tag words on the GPU: chains, tag collisions, absent keys and
runs of equal keys, against the oracle (exact)."""
import numpy as np
import pytest

import oracle
from tests.conftest import VB
from wukonggpu_amd import Device, GPUEngine, GStore, Triples

pytestmark = pytest.mark.gpu

SUBJECTS = 90000  # about 12k buckets a direction: hundreds hold two keys of one tag


@pytest.fixture(scope="module")
def triples():
    rng = np.random.default_rng(8)
    n = 120000
    s = VB + 2 * rng.integers(0, SUBJECTS, n)  # odd ids never have edges
    return Triples.from_arrays(s, np.full(n, 2), VB + 2 * rng.integers(0, SUBJECTS, n))


@pytest.mark.parametrize("load,rows,run", [(0.2, 700, 1), (0.75, 65537, 1), (0.75, 70000, 4), (1.0, 180000, 1),
                                           (1.0, 40001, 3)])
def test_probe_through_tags(triples, load, rows, run):
    gs = GStore.build(triples, main_load=load)
    rng = np.random.default_rng(rows)
    keys = VB + rng.permutation(2 * SUBJECTS)[:(rows + run - 1) // run]
    tab = np.stack([np.repeat(keys, run)[:rows], np.arange(rows)], axis=1).astype(np.int32)
    tab[rng.random(rows) < 0.01, 0] = -2
    devs = [Device(0), Device(0), Device(0)]
    devs[0].load(gs)
    devs[1].build(triples, main_load=load)
    devs[2].load(gs, graph_budget_bytes=gs.image_nbytes())  # no room for tag words: whole buckets
    for dev in devs:
        dt = dev.table(tab)
        for d in (0, 1):
            want, wex = oracle.run_step(gs, [VB, 2, 1, -1, -1, 2, d, -3], 1, tab)
            for tile in (0, 256, 2048):
                dev.set_probe_tile_rows(tile)
                t, ex = dev.k2u(dt, 0, 2, d)
                assert ex == wex and np.array_equal(t.to_host(), want), (d, tile)
            (out,), _ = dev.step_batch([dict(kind=2, pid=2, dir=d, start_col=0, input=dt)])
            assert np.array_equal(out.to_host(), want), d
            dev.set_probe_tile_rows(0)
            const = VB + 2 * (rows % SUBJECTS)
            want, wex = oracle.run_step(gs, [VB, 2, 1, -1, -1, 2, d, const], 1, tab)
            f, ex = dev.k2c(dt, 0, 2, d, const)
            assert ex == wex and np.array_equal(f.to_host().reshape(want.shape), want), d
        dev.close()


def test_budget_without_room_for_tags(triples):
    """A graph budget that holds the image but not the tag words (8 B per main
    bucket): resident all the same, and the statistics tell the two apart;
    whole queries, the executor and step rounds answer as with them."""
    gs = GStore.build(triples)
    rng = np.random.default_rng(3)
    qs = [[2, 0, d, -1, -1, 2, 1 - d, -2, -2, 2, d, -3] for d in (0, 1)]
    qs += [[int(v), 2, d, -1, -1, 2, 1 - d, -2] for v in rng.integers(VB, VB + 2 * SUBJECTS, 40) for d in (0, 1)]
    want = [oracle.run_query(gs, q)[:2] for q in qs]
    sizes = []
    for budget in (0, gs.image_nbytes(), gs.image_nbytes() + (1 << 30)):
        dev = Device(0)
        dev.load(gs, graph_budget_bytes=budget)
        sizes.append(dev.stats()["resident_bytes"])
        eng = GPUEngine(dev)
        for rs in ([eng.run_query(q) for q in qs], eng.run_batched(qs), eng.run_rounds(qs)):
            for r, (t, ex) in zip(rs, want):
                assert r.expanded == ex and np.array_equal(r.table.reshape(t.shape), t)
        eng.close()
        dev.close()
    assert sizes[1] == gs.image_nbytes() < sizes[0] == sizes[2]
    assert (sizes[0] - sizes[1]) % 8 == 0
