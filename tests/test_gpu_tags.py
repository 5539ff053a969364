"""The probe's tag words on the GPU: chains, tag collisions, absent keys and
runs of equal keys, against the oracle (exact)."""
import numpy as np
import pytest

import oracle
from tests.conftest import VB
from wukonggpu_amd import Device, GStore, Triples

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
    devs = [Device(0), Device(0)]
    devs[0].load(gs)
    devs[1].build(triples, main_load=load)
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
        dev.close()
