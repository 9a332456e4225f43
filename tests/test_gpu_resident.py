"""Databases of small graphs mined out of LDS (gv_resident_mine): counts,
algorithmic bytes and matched graph ids against the oracle where the packed
form, its blocks and its levels have their edges.  All whole numbers."""
import ctypes as C

import numpy as np
import pytest

import geneva_amd as G

pytestmark = pytest.mark.gpu


def _blocks(eng):
    """Blocks of the packed form (0: mined by the table engines)."""
    L = G.lib()
    L.gh_engine_resident_blocks.restype = C.c_uint32
    L.gh_engine_resident_blocks.argtypes = [C.c_void_p]
    return L.gh_engine_resident_blocks(eng._h)


def _edge_labelled(ds, n, seed):
    e = ds.edges
    e[:, 2] = np.random.default_rng(seed).integers(1, n + 1, size=len(e))
    ds = G.Dataset.from_arrays(ds.vlabel, e, ds.graph_of, ds.ngraphs)
    ds.reorder_intervals()
    return ds


def _check(ds, qs, single_v=False, packed=True):
    import oracle as O
    og = O.OracleGraph.of(ds)
    eng = G.Engine(ds)
    assert (_blocks(eng) > 0) == packed
    want = [og.mine(q, threads=8) for q in qs]
    batch, st = eng.mine_batch(qs)
    for i, (q, w) in enumerate(zip(qs, want)):
        for r in (eng.mine(q), batch[i]):
            assert r.count == w.count, (i, q)
            assert r.alg_bytes == w.alg_bytes, (i, q)
            assert r.graph_ids == w.graph_ids, (i, q)
    eng.close()


# (graphs, nmin, nmax, degree, share of hub graphs, labels, zipf, edge labels,
# kmin, kmax): pairs and triangles only, one label, more label segments than
# one and two mask words hold, graphs of several hundred vertices (blocks of
# one graph), more rows at a level than it holds, deep queries
SHAPES = [
    (40, 2, 3, 1.0, 0.0, 2, 0.0, 1, 2, 3),
    (2, 30, 30, 4.0, 0.5, 1, 0.0, 1, 3, 4),
    (500, 5, 40, 3.0, 0.3, 5, 0.0, 1, 2, 6),
    (97, 20, 90, 4.0, 0.5, 33, 1.0, 1, 3, 7),
    (150, 10, 60, 4.0, 0.5, 70, 0.5, 1, 3, 7),
    (60, 30, 80, 4.0, 0.5, 22, 1.0, 4, 3, 6),
    (7, 400, 700, 4.0, 0.5, 12, 1.0, 1, 3, 5),
    (30, 60, 120, 6.0, 1.0, 3, 0.0, 1, 3, 5),
    (200, 15, 40, 3.5, 0.2, 16, 0.5, 2, 9, 12),
]


@pytest.mark.parametrize("shape", SHAPES)
def test_packed_database_equals_oracle(require_gpu, shape):
    n, nmin, nmax, deg, ba, labels, zipf, el, kmin, kmax = shape
    ds = G.Dataset.database(n, nmin, nmax, deg, ba, labels, zipf, 77 + n)
    if el > 1:
        ds = _edge_labelled(ds, el, 5)
    ds.add_walk_queries(10, kmin, kmax, seed=3)
    ds.add_walk_queries(5, min(max(kmin, 3), 6), min(kmax, 6), induced=True, seed=4)
    print(shape, flush=True)
    _check(ds, ds.queries)


def test_more_operations_than_one_launch(require_gpu):
    """A batch whose queries have more steps than one launch holds."""
    ds = G.Dataset.database(120, 20, 60, 4.0, 0.5, 24, 0.3, 9)
    ds.add_walk_queries(330, 5, 8, seed=11)
    _check(ds, ds.queries)


def test_databases_that_are_not_packed(require_gpu):
    """An edge between two graphs, a graph beyond a block, too many labels:
    the table engines mine these, with the same results."""
    ds = G.Dataset.database(50, 10, 30, 3.0, 0.0, 4, 0.0, 21)
    go = ds.graph_of
    e = ds.edges
    other = int(np.nonzero(go[1:] == go[e[0, 0]] + 1)[0][0]) + 1
    joined = np.concatenate([e, np.array([[e[0, 0], other, 1]], dtype=np.uint32)])
    j = G.Dataset.from_arrays(ds.vlabel, joined, go, ds.ngraphs)
    j.add_walk_queries(6, 3, 5, seed=1)
    _check(j, j.queries, packed=False)
    big = G.Dataset.database(3, 4000, 4200, 4.0, 0.0, 20, 0.0, 22)
    big.add_walk_queries(5, 3, 5, seed=2)
    _check(big, big.queries, packed=False)
    many = G.Dataset.database(80, 20, 60, 4.0, 0.0, 300, 0.0, 23)
    many.add_walk_queries(5, 3, 5, seed=2)
    _check(many, many.queries, packed=False)
