"""Which engine mines a database, and what it gives there: the packed form's
branches for operations with many references, single-vertex plans, graph ids
far apart; the slot engine and the serving loop over it on a database that is
not packed (an edge between two of its graphs).  Against the oracle, all whole
numbers."""
import numpy as np
import pytest

import geneva_amd as G
from geneva_amd import configs

pytestmark = pytest.mark.gpu


def _query(labels, edges):
    return "".join(f"v {i} {l}\n" for i, l in enumerate(labels)) + "".join(f"e {a} {b} 1\n" for a, b in edges)


def _path(labels):
    return _query(labels, [(i, i + 1) for i in range(len(labels) - 1)])


def _clique(n):
    return _query([1] * n, [(i, j) for i in range(n) for j in range(i)])


def _launches(eng, call):
    """call()'s result and the k_resident launches it made."""
    eng.profile(True, count_bytes=False)
    r = call()
    n = eng.profile_read()["k_resident"][0]
    eng.profile(False)
    return r, n


def _check(ds, qs, single_v=False):
    import oracle as O
    og, eng = O.OracleGraph.of(ds), G.Engine(ds)
    want = [og.mine(q, threads=8) for q in qs]
    (batch, _), n = _launches(eng, lambda: eng.mine_batch(qs, single_v=single_v))
    assert n >= 1
    for i, (q, w) in enumerate(zip(qs, want)):
        r, n = _launches(eng, lambda q=q: eng.mine(q, single_v=single_v))
        assert n >= 1 or w.count == 0, (i, q)
        for x in (r, batch[i]):
            assert x.count == w.count, (i, q)
            assert x.graph_ids == w.graph_ids, (i, q)
            if not single_v:   # the oracle's plan, and so its bytes
                assert x.alg_bytes == w.alg_bytes, (i, q)
    eng.close()


# one label on dense and on sparse graphs: cliques (up to 6 back columns),
# paths (up to 13 same-label columns and copies, levels of 16 columns), rings
MANY = [
    (25, 12, 16, 8.0, [_clique(4), _clique(5), _clique(6), _path([1] * 6)]),
    (60, 10, 24, 2.0, [_path([1] * 9), _path([1] * 12), _path([1] * 14),
                       _query([1] * 6, [(i, (i + 1) % 6) for i in range(6)])]),
]


@pytest.mark.parametrize("single_v", [False, True])
@pytest.mark.parametrize("many", MANY, ids=["dense", "sparse"])
def test_operations_with_many_references(require_gpu, many, single_v):
    n, nmin, nmax, deg, qs = many
    _check(G.Dataset.database(n, nmin, nmax, deg, 0.0, 1, 0.0, 31), qs, single_v)


def test_leaf_groups_below_many_core_columns(require_gpu):
    """A leaf group whose label four and five core columns hold."""
    ds = G.Dataset.database(120, 20, 40, 3.0, 0.4, 2, 0.0, 32)
    qs = [_query([2, 1, 1, 1, 1, 2, 1, 1], [(0, 1), (1, 2), (2, 3), (3, 4), (4, 5), (3, 6), (3, 7)]),
          _query([2, 1, 1, 1, 1, 1, 2, 1, 1], [(0, 1), (1, 2), (2, 3), (3, 4), (4, 5), (5, 6), (3, 7), (3, 8)])]
    for single_v in (False, True):
        _check(ds, qs, single_v)


@pytest.mark.parametrize("single_v", [False, True])
@pytest.mark.parametrize("step", [1, 97])
def test_walk_queries_and_graph_ids_far_apart(require_gpu, step, single_v):
    """Graph ids 97 apart end a block by the ids it may span, not by its size."""
    ds = G.Dataset.database(300, 5, 40, 3.0, 0.3, 5, 0.0, 33)
    ds = G.Dataset.from_arrays(ds.vlabel, ds.edges, ds.graph_of * step, ds.ngraphs * step)
    ds.add_walk_queries(12, 2, 7, seed=3)
    _check(ds, ds.queries, single_v)


def test_more_operations_than_one_launch_takes(require_gpu):
    """More than 256 counted operations: a second launch."""
    ds = G.Dataset.database(120, 20, 60, 4.0, 0.5, 24, 0.3, 9)
    ds.add_walk_queries(330, 5, 8, seed=11)
    eng = G.Engine(ds)
    _, n = _launches(eng, lambda: eng.mine_batch(ds.queries))
    assert n >= 2
    eng.close()


@pytest.fixture(scope="module")
def joined(require_gpu):
    """The scaled database of workload 3 with an edge between its first two
    graphs, 40 walk queries and what the oracle says."""
    import oracle as O
    ds = configs.workload3(scale=0.005, nqueries=0)
    go, e = ds.graph_of, ds.edges
    first = [int(np.nonzero(go[1:] == g)[0][0]) + 1 for g in (0, 1)]
    ds = G.Dataset.from_arrays(ds.vlabel, np.concatenate([e, np.array([first + [1]], dtype=np.uint32)]), go, ds.ngraphs)
    ds.add_walk_queries(40, 3, 8, seed=6)
    og = O.OracleGraph.of(ds)
    qs = ds.queries + ds.queries[:12]   # some twice: the same steps
    return ds, qs, [og.mine(q, threads=8) for q in qs]


def _equal(res, want):
    for i, (r, w) in enumerate(zip(res, want)):
        assert r.count == w.count and r.alg_bytes == w.alg_bytes and r.graph_ids == w.graph_ids, i


@pytest.mark.parametrize("row_cap", [1 << 22, 1 << 13])
def test_slot_engine_shares_and_defers(joined, row_cap):
    """Shared tables, followers that restart under a small row cap, sizing
    groups and each switch off: the same results, from the slot engine."""
    ds, qs, want = joined
    eng = G.Engine(ds)
    eng.batch_config(slots=64, slot_bytes=8 << 20, row_cap=row_cap)
    (res, st), n = _launches(eng, lambda: eng.mine_batch(qs))
    assert n == 0 and st["graph_launches"] > 1
    _equal(res, want)
    shared, restarted = eng.batch_share_stats()
    assert shared > 0
    print("row_cap", row_cap, "shared", shared, "restarted", restarted, flush=True)
    assert restarted > 0 or row_cap > 1 << 13
    rows = eng.batch_fused_rows()
    assert rows > 0
    for off in (eng.batch_share, eng.batch_fuse_sizing, eng.batch_pair_start):
        off(False)
        before = eng.batch_share_stats(), eng.batch_fused_rows()
        _equal(eng.mine_batch(qs)[0], want)
        if off is eng.batch_share:
            assert eng.batch_share_stats() == before[0]
        if off is eng.batch_fuse_sizing:
            assert eng.batch_fused_rows() == before[1]
        off(True)
    eng.close()


@pytest.mark.parametrize("ipt,bpc", [(1, 4), (2, 32), (8, 4)])
def test_slot_engine_tunings(joined, ipt, bpc):
    ds, qs, want = joined
    eng = G.Engine(ds)
    eng.batch_config(slots=64, slot_bytes=8 << 20, row_cap=1 << 22, ipt=ipt, blocks_per_cu=bpc)
    _equal(eng.mine_batch(qs)[0], want)
    eng.close()


# (row cap, slot bytes, requests a second, memory bound)
@pytest.mark.parametrize("row_cap,slot_bytes,rate,budget", [
    (1 << 22, 8 << 20, 3000.0, 16 << 30), (1 << 13, 8 << 20, 20000.0, 16 << 30),
    (1 << 22, 1 << 18, 20000.0, 16 << 30), (1 << 22, 8 << 20, 20000.0, 1)])
def test_serving_on_the_slot_engine(joined, row_cap, slot_bytes, rate, budget):
    """Admission, deferral, overflow to the side worker and a tight memory
    bound: every request its own count and graph ids."""
    ds, qs, want = joined
    eng = G.Engine(ds)
    eng.batch_config(slots=16, slot_bytes=slot_bytes, row_cap=row_cap)
    arr = np.cumsum(np.random.default_rng(9).exponential(1 / rate, size=len(qs))).tolist()
    lat, cnt, st, ids = eng.serve(qs, arr, mem_budget=budget, with_graphs=True)
    print("stats", st, flush=True)
    assert cnt == [w.count for w in want]
    assert [frozenset(i) for i in ids] == [w.graph_ids for w in want]
    assert all(l > 0 for l in lat)
    if rate > 10000:
        assert st["iterations"] > 0
    eng.close()
