"""Performance cases of the graph-exploration engine.

Every case runs on one loaded dataset, as a user's program does: a 100M-triple
graph (10M entities, 64 predicates, Zipf-1.0 subject degrees, type indexes
from 1 to 500k members, linked predicate pairs, one million-edge hub and
planted triangles -- the shapes of `wukonggpu_amd.workloads`), built on the
device once per process. A case fixes which vertices, queries and end cells
its inputs hold (so every seed's answer has the same number of rows); the
seed decides the order in which they come and the other columns' bindings.

Kinds
  point   one 2-hop query from a constant (the latency of the smallest query)
  plain   selective 3-4 pattern queries, one after another on the plain path
  mix     the same kind of queries as one batch on the device-resident executor
  heavy   the star query's steps from a table of start vertices: two hops, a hub
          fan-out, a second arm and a closing edge (10^7..10^8-row tables)
  cycle   the 6-pattern cycle's steps from a table of start vertices, the hub
          fan-out fused with its filter
  k2u     one known_to_unknown step over a table
  k2k     one known_to_known step (is the row's end cell a neighbour?)
  k2c     one known_to_const step (is the constant a neighbour?)
  split   fork-join exchange of one table: split by owner, replies merged
"""
import ctypes
import math

import numpy as np
import torch

from wukonggpu_amd import Device, GPUEngine, Triples, workloads
from wukonggpu_amd.engine import Batch, plan_of
from wukonggpu_amd import _native as native
from wukonggpu_amd.gstore import VID_BASE

IN, OUT = 0, 1
ENTITIES, PREDS, TRIPLES = 10_000_000, 64, 100_000_000
HUB_PRED, HUB_DEGREE, PLANTED_PRED = 2, 1_000_000, 50
T0 = 2 + PREDS  # the 500k-member type; T0 + 1 .. T0 + 511 are the others
TYPE_SIZES = [500_000] + [int(x) for x in np.exp(np.random.default_rng(2).uniform(0.0, math.log(1e5), 511))]
# per predicate: subjects, objects, edges (about; every predicate follows one rule)
SUBJECTS, OBJECTS, EDGES = 130_900, 1_448_000, 1_562_500


class Dataset:
    """The loaded graph, its engine, and the index lists that inputs are drawn from."""

    def __init__(self):
        triples = Triples.generate(seed=2, num_entities=ENTITIES, num_preds=PREDS, num_triples=TRIPLES, zipf_s=1.0,
                                   type_sizes=TYPE_SIZES, num_linked=PREDS // 2, link_frac=0.25, num_hubs=1,
                                   hub_degree=HUB_DEGREE, siblings=[(HUB_PRED, PLANTED_PRED)])
        self.dev = Device(0)
        self.dev.build(triples)
        triples.close()
        self.engine = GPUEngine(self.dev)
        # the executor as a tuned program keeps it: up to 1024 queries, tiles dealt statically
        self.batch = Batch(self.dev, 1024, 8, 16 << 30)
        self.batch.set_tuning(probe_wg_per_cu=4, expand_wg_per_cu=8, aux_wg_per_cu=2, probe_tile_rows=1024,
                              expand_tile_items=1024, schedule=1)
        self._lists, self._degrees, self._edges, self._points = {}, {}, {}, {}

    def index(self, pid, d):
        """Vertices with a (pid, d) list: the predicate's subjects (OUT) or objects (IN), ascending."""
        if (pid, d) not in self._lists:
            t, _ = self.dev.i2u(pid, IN if d == OUT else OUT)
            self._lists[pid, d] = t.to_host()[:, 0]
        return self._lists[pid, d]

    def edges(self, pid):
        """(subject, object) of every edge of pid, by subject."""
        if pid not in self._edges:
            start = self.dev.table(self.index(pid, OUT)[:, None])
            t, _ = self.dev.k2u(start, 0, pid, OUT)
            self._edges[pid] = t.to_host()
        return self._edges[pid]

    def degrees(self, pid):
        """Out-degree of every subject of pid, in index order."""
        if pid not in self._degrees:
            self._degrees[pid] = np.unique(self.edges(pid)[:, 0], return_counts=True)[1]
        return self._degrees[pid]

    def points(self, degree):
        """2-hop queries from constants of about this degree whose answers have one row count."""
        if degree not in self._points:
            rng = np.random.default_rng([degree, 3])
            qs = []
            for p1 in rng.choice(np.arange(3, 50), size=12, replace=False):
                near = np.argsort(np.abs(self.degrees(int(p1)) - degree), kind="stable")[:8]
                for c in self.index(int(p1), OUT)[near]:
                    for p2 in rng.choice(np.setdiff1d(np.arange(3, 50), [p1]), size=6, replace=False):
                        qs.append([int(c), int(p1), OUT, -1, -1, int(p2), IN, -2])
            rows = np.array([r.rows for r in self.engine.run_plain(qs)])
            sizes, counts = np.unique(rows[rows > 0], return_counts=True)
            usual = sizes[np.argmax(counts)]
            self._points[degree] = [q for q, r in zip(qs, rows) if r == usual]
        return self._points[degree]

    def hub(self, pid):
        return int(self.index(pid, OUT)[np.argmax(self.degrees(pid))])


_dataset = None


def dataset():
    global _dataset
    if _dataset is None:
        _dataset = Dataset()
    return _dataset


class _Cells:
    """A device table's cells for torch.as_tensor (no copy; keeps the table)."""

    def __init__(self, table):
        self.table = table
        ptr = ctypes.cast(native.hip_lib().wkg_table_device_ptr(table._h), ctypes.c_void_p).value
        self.__cuda_array_interface__ = {"shape": table.shape, "typestr": "<i4", "data": (ptr, False), "version": 2}


def _tensor(table):
    if not table.shape[0]:
        return torch.empty(table.shape, dtype=torch.int32, device="cuda")
    return torch.as_tensor(_Cells(table), device="cuda")


# ---- cases --------------------------------------------------------------------

def listed():
    return [
        # a lookup behind a web request: ~1000 neighbours, then one hop from each
        {"name": "point_1000", "kind": "point", "degree": 1000},
        # interactive queries, one at a time
        {"name": "plain_16", "kind": "plain", "queries": 16},
        # a proxy's batch of gathered queries
        {"name": "mix_512", "kind": "mix", "queries": 512},
        # analytical queries: a star over hubs, and a cycle through the largest hub
        {"name": "heavy_star", "kind": "heavy", "rows": 500_000, "pa": 2 + 46, "pb": 4},
        {"name": "hub_cycle", "kind": "cycle", "rows": 100_000, "pa": 40},
        # a step of an interactive query, its table from another server or the host
        {"name": "k2u_300", "kind": "k2u", "rows": 300, "cols": 2, "pid": 4, "dir": OUT, "hit": 0.8, "run": 1},
        # a middling ragged step, repeated start cells as after an earlier fan-out
        {"name": "k2u_ragged", "kind": "k2u", "rows": 100_003, "cols": 5, "pid": 7, "dir": IN, "hit": 0.6, "run": 3},
        # a wide table fanned out over skewed lists
        {"name": "k2u_fanout", "kind": "k2u", "rows": 2_000_003, "cols": 3, "pid": 20, "dir": OUT, "hit": 0.8,
         "run": 1},
        # a large one-column table of ids, most of them without the predicate: lookups of random keys
        {"name": "k2u_keys", "kind": "k2u", "rows": 24_000_001, "cols": 1, "pid": 33, "dir": IN, "hit": 0.25,
         "run": 1},
        # filters: a closing edge, and a type-like check against a popular constant
        {"name": "k2k_3m", "kind": "k2k", "rows": 3_000_017, "cols": 3, "pid": 12, "dir": OUT, "hit": 0.5, "run": 1},
        {"name": "k2c_12m", "kind": "k2c", "rows": 12_000_000, "cols": 2, "pid": 9, "dir": IN, "hit": 0.7, "run": 1},
        # the exchange step of a sharded deployment on one server's table
        {"name": "split_8", "kind": "split", "rows": 8_000_009, "cols": 4, "parts": 8},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(("point", "plain", "mix", "heavy", "cycle", "k2u", "k2u", "k2u", "k2k", "k2c", "split"))
    if kind == "point":
        return {"kind": kind, "degree": _log_int(rng, 40, 2000)}
    if kind == "plain":
        return {"kind": kind, "queries": _log_int(rng, 1, 16)}
    if kind == "mix":
        return {"kind": kind, "queries": _log_int(rng, 16, 512)}
    if kind == "heavy":
        return {"kind": kind, "rows": _log_int(rng, 50_000, 500_000), "pa": rng.randint(24, 49),
                "pb": 2 * rng.randint(2, 11)}
    if kind == "cycle":
        return {"kind": kind, "rows": _log_int(rng, 2_000, 100_000), "pa": rng.randint(3, 49)}
    if kind == "split":
        cols = rng.randint(1, 8)
        return {"kind": kind, "rows": _log_int(rng, 1_000, 32_000_000 // cols), "cols": cols,
                "parts": _log_int(rng, 2, 256)}
    d = rng.randint(IN, OUT)
    cols = rng.randint(1 if kind == "k2u" else 2, 6)
    most = 24_000_000 if kind != "k2u" or d == IN else 2_500_000  # an OUT hop's output is ten times its input
    return {"kind": kind, "rows": _log_int(rng, 100, most // cols), "cols": cols, "pid": rng.randint(3, 49), "dir": d,
            "hit": round(rng.uniform(0.1, 1.0), 2), "run": rng.choice((1, 1, 2, 5))}


# ---- inputs -------------------------------------------------------------------

def _fixed(case, salt):
    """The generator of what a case holds whatever the seed."""
    return np.random.default_rng([salt, *(int(1000 * v) for v in case.values() if not isinstance(v, str))])


def _order(n, seed):
    return torch.randperm(n, generator=torch.Generator("cuda").manual_seed(int(seed)), device="cuda",
                          dtype=torch.int32 if n < 1 << 31 else torch.int64).cpu().numpy()


def _ids(rng, n):
    return rng.integers(VID_BASE, VID_BASE + ENTITIES, n, dtype=np.int32)


def _members(g, case, seed):
    """Start vertices of a query's first hop, without the few that have more than 2000 pa edges."""
    ids = _ids(_fixed(case, 11), case["rows"])
    big = g.index(case["pa"], OUT)[g.degrees(case["pa"]) > 2000]
    ids[np.isin(ids, big)] = VID_BASE
    return ids[_order(len(ids), seed)]


def _step_table(g, case, seed):
    """(host table, start column, end column) of a single step: start cells
    are ids with the case's list (share `hit`) among uniform ones, in runs of
    `run` rows on average; the start column is the newest binding. For
    known_to_known, half of the (start, end) pairs are edges."""
    n, cols, pid, d = case["rows"], case["cols"], case["pid"], case["dir"]
    fixed, rng = _fixed(case, 13), np.random.default_rng([seed, 17])
    keys = max(1, n // case["run"])
    known = g.index(pid, d)
    start = _ids(fixed, keys)
    hit = fixed.random(keys, dtype=np.float32) < case["hit"]
    start[hit] = known[fixed.integers(0, len(known), int(hit.sum()), dtype=np.int32)]
    end = None
    if case["kind"] == "k2k":
        end = _ids(fixed, keys)
        walked = np.nonzero(fixed.random(keys, dtype=np.float32) < 0.5)[0]
        e = g.edges(pid)[fixed.integers(0, len(g.edges(pid)), len(walked), dtype=np.int32)]
        s, o = (0, 1) if d == OUT else (1, 0)
        start[walked], end[walked] = e[:, s], e[:, o]
    at = _order(keys, seed)
    if case["run"] > 1:
        times = np.bincount(fixed.integers(0, keys, n, dtype=np.int32), minlength=keys)
        at = np.repeat(at, times[at])
    t = np.empty((n, cols), dtype=np.int32)
    for c in range(cols - 1):
        t[:, c] = _ids(rng, n)
    t[:, cols - 1] = start[at]
    if end is not None:
        t[:, cols - 2] = end[at]
    return t, cols - 1, cols - 2


def prepare(case, seed):
    g, kind = dataset(), case["kind"]
    st = {"g": g, "kind": kind}
    if kind == "point":
        pool = g.points(case["degree"])
        st["query"] = pool[seed % len(pool)]
    elif kind in ("plain", "mix"):
        queries = workloads.batched_queries(PREDS, list(range(T0 + 1, T0 + len(TYPE_SIZES))), case["queries"], 7)
        queries = [queries[i] for i in _order(len(queries), seed)]
        if kind == "plain":
            st["queries"] = queries
        else:
            st["n"] = len(queries)
            st["plans"], st["offsets"] = Batch._plans([plan_of(q) for q in queries])
            st["results"] = (native.BatchResult * len(queries))()
    elif kind == "heavy":
        st.update(table=g.dev.table(_members(g, case, seed)[:, None]), pa=case["pa"], pb=case["pb"])
    elif kind == "cycle":
        hub, e = g.hub(HUB_PRED), g.edges(HUB_PRED)
        st.update(table=g.dev.table(_members(g, case, seed)[:, None]), pa=case["pa"],
                  const=int(e[np.searchsorted(e[:, 0], hub), 1]))
    elif kind == "split":
        rng = np.random.default_rng([seed, 19])
        t = rng.integers(VID_BASE, VID_BASE + ENTITIES, (case["rows"], case["cols"]), dtype=np.int32)
        st.update(table=g.dev.table(t), col=case["rows"] % case["cols"], parts=case["parts"])
    else:
        t, start, end = _step_table(g, case, seed)
        st.update(table=g.dev.table(t), start=start, end=end, pid=case["pid"], dir=case["dir"])
        if kind == "k2c":
            # a popular constant: the predicate's hub (IN), or a neighbour of one of the start cells (OUT)
            st["const"] = g.hub(case["pid"])
            if case["dir"] == OUT:
                e = g.edges(case["pid"])
                first = np.intersect1d(t[:, start], g.index(case["pid"], OUT))[0]
                st["const"] = int(e[np.searchsorted(e[:, 0], first), 1])
    return st


# ---- one pass -----------------------------------------------------------------

def _then_filter(dev, t, start, pid, d, filter_pid, filter_dir, end):
    """A hop and a closing edge on its new column, as the engine makes them."""
    new = t.shape[1]
    out, fused, hop, closed = dev.k2u_filter(t, start, pid, d, native.STEP_K2K, filter_pid, filter_dir, end)
    if not fused:
        out, closed = dev.k2k(out, new, filter_pid, filter_dir, end)
    return out, hop + closed


def run(st):
    g, kind = st["g"], st["kind"]
    dev = g.dev
    if kind == "point":
        r = g.engine.run_query(st["query"])
        return {"table": r.table, "expanded": r.expanded}
    if kind == "plain":
        rs = g.engine.run_plain(st["queries"])
        return {"rows": np.array([r.rows for r in rs]), "expanded": np.array([r.expanded for r in rs]),
                "cells": np.concatenate([r.table.reshape(-1) for r in rs])}
    if kind == "mix":
        cells, ncells = ctypes.POINTER(ctypes.c_int32)(), ctypes.c_uint64()
        dev._check(native.hip_lib().wkg_batch_run(g.batch._h, st["n"], st["plans"], st["offsets"], st["results"],
                                                  ctypes.byref(cells), ctypes.byref(ncells)))
        # a record is offset, rows, (cols, status), expanded; the tables lie in the batch's pinned result buffer
        rec = np.frombuffer(st["results"], dtype=np.int64).reshape(-1, 4)
        flat = np.ctypeslib.as_array(cells, shape=(ncells.value,))
        ends = rec[:, 0] + rec[:, 1] * (rec[:, 2] & 0xffffffff)
        return {"rows": rec[:, 1], "expanded": rec[:, 3],
                "cells": np.concatenate([flat[a:b] for a, b in zip(rec[:, 0].tolist(), ends.tolist())])}
    if kind == "split":
        t, rows, head = dev.table_split(st["table"], st["col"], st["parts"])
        # the replies come back in another order than they went out
        parts = [dev.table_slice(t, head[p], rows[p]) for p in reversed(range(st["parts"]))]
        merged = dev.table_concat(parts)
        return {"split": _tensor(t), "rows": rows, "merged": _tensor(merged)}
    if kind == "heavy":  # ?x pa ?y . ?z pb ?y . ?z pb ?u . ?z pc ?w . ?z pb ?w
        pb = st["pb"]
        t, e1 = dev.k2u(st["table"], 0, st["pa"], OUT)
        t, e2 = dev.k2u(t, 1, pb, IN)
        t, e3 = dev.k2u(t, 2, pb, OUT)
        t, e4 = _then_filter(dev, t, 2, pb + 1, OUT, pb, IN, 2)
        return {"table": t.to_host(), "expanded": np.array([e1, e2, e3, e4])}
    if kind == "cycle":  # ?a pa ?b . ?c ph ?b . ?c ph ?d . ?d pc ?b . ?c ph const
        t, e1 = dev.k2u(st["table"], 0, st["pa"], OUT)
        t, e2 = dev.k2u(t, 1, HUB_PRED, IN)
        t, e3 = _then_filter(dev, t, 2, HUB_PRED, OUT, PLANTED_PRED, OUT, 1)
        t, e4 = dev.k2c(t, 2, HUB_PRED, OUT, st["const"])
        return {"table": t.to_host(), "expanded": np.array([e1, e2, e3, e4])}
    if kind == "k2u":
        t, expanded = dev.k2u(st["table"], st["start"], st["pid"], st["dir"])
    elif kind == "k2k":
        t, expanded = dev.k2k(st["table"], st["start"], st["pid"], st["dir"], st["end"])
    else:
        t, expanded = dev.k2c(st["table"], st["start"], st["pid"], st["dir"], st["const"])
    return {"table": _tensor(t), "expanded": expanded}


# ---- what a pass cannot do without ----------------------------------------------

def work(case):
    """Bytes: the input cells read once, each distinct key's bucket (128 B)
    and each distinct list entry (4 B) read once, the output cells written
    once. Expected values of the generator's rules; the query kinds use the
    averages of their drawn queries."""
    kind = case["kind"]
    if kind == "point":
        n = case["degree"]
        return {"bytes": 128.0 + 4 * n + 128 * n + 0.15 * n * (4 + 8), "flops": 0}
    if kind in ("plain", "mix"):
        # a query: ~8.5k start members, a hop (a bucket each), a second with ~5k keys, ~20k result cells
        return {"bytes": case["queries"] * (4.0 * 8500 + 128 * (8500 + 5000) + 4 * 20000), "flops": 0}
    if kind == "heavy":
        # the start keys' buckets, the hub fan-out's rows (4 columns) written
        m = case["rows"] / 500_000
        return {"bytes": m * (132.0 * 500_000 + 130e6 * 16), "flops": 0}
    if kind == "cycle":
        # the start and second-hop keys, the hub's list and its entries' buckets
        return {"bytes": 132.0 * 1.3 * case["rows"] + 132.0 * HUB_DEGREE, "flops": 0}
    n, c = case["rows"], case["cols"]
    if kind == "split":
        return {"bytes": 16.0 * n * c, "flops": 0}  # read and written by the split, and again by the merge
    lists = SUBJECTS if case["dir"] == OUT else OBJECTS
    keys = n / case["run"]
    hits = keys * case["hit"]
    distinct = lists * (1 - math.exp(-hits / lists)) + ENTITIES * (1 - math.exp(-(keys - hits) / ENTITIES))
    share = (case["hit"] + (1 - case["hit"]) * lists / ENTITIES)  # of rows with a list
    read = 4.0 * n * c + 128 * distinct
    if kind == "k2u":
        out = n * share * EDGES / lists
        return {"bytes": read + 4 * min(out, EDGES) + 4 * out * (c + 1), "flops": 0}
    return {"bytes": read + 4 * min(n * share, EDGES) + 4 * c * n * share * (0.45 if kind == "k2k" else 0.08),
            "flops": 0}
