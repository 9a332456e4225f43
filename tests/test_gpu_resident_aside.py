"""Databases whose work sits in few blocks: a wave of k_resident that has done
much in one block leaves the next tables to another launch.  Counts,
algorithmic bytes and matched graph ids against the oracle, and more than one
launch, one query at a time and in one call.  All whole numbers."""
import pytest

import geneva_amd as G

pytestmark = pytest.mark.gpu


def _launches(eng, call):
    """call()'s result and the k_resident launches it made."""
    eng.profile(True, count_bytes=False)
    r = call()
    n = eng.profile_read()["k_resident"][0]
    eng.profile(False)
    return r, n


# (graphs, nmin, nmax, labels, zipf, degree share of hub graphs, queries, kmin,
# kmax): one block in hundreds holds a star's centre; 16 blocks of hub graphs
# and several launches; more tables set aside than a launch may (the rest is
# mined where it is)
SHAPES = [
    (800, 20, 400, 12, 0.7, 0.5, 200, 5, 8),
    (16, 280, 300, 3, 0.0, 1.0, 14, 4, 8),
    (64, 180, 200, 1, 0.0, 1.0, 3, 6, 6),
]


@pytest.mark.parametrize("shape", SHAPES)
def test_tables_set_aside_equal_oracle(require_gpu, shape):
    import oracle as O
    n, nmin, nmax, labels, zipf, ba, nq, kmin, kmax = shape
    ds = G.Dataset.database(n, nmin, nmax, 4.0, ba, labels, zipf, 5 if n < 100 else 9)
    ds.add_walk_queries(nq, kmin, kmax, seed=3)
    ds.add_walk_queries(3, 5, 6, induced=True, min_extra=1, seed=4)
    og, eng = O.OracleGraph.of(ds), G.Engine(ds)
    qs = ds.queries
    want = [og.mine(q, threads=8) for q in qs]
    (batch, _), nbatch = _launches(eng, lambda: eng.mine_batch(qs))
    single = [_launches(eng, lambda q=q: eng.mine(q)) for q in qs]
    print(shape, "launches of the batch", nbatch, "of single queries", sorted({s[1] for s in single}), flush=True)
    assert nbatch > 1 and max(s[1] for s in single) > 1
    assert min(s[1] for s in single) >= 1
    for i, w in enumerate(want):
        for r in (single[i][0], batch[i]):
            assert r.count == w.count, (i, qs[i])
            assert r.alg_bytes == w.alg_bytes, (i, qs[i])
            assert r.graph_ids == w.graph_ids, (i, qs[i])
    eng.close()
