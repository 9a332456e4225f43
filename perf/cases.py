"""The work that a user of this framework has it do, as cases to be timed.

A case is a dict of plain values; listed() names the usual ones, draw(rng)
gives more of the same ranges, prepare(case, seed) makes what a program holds
before the call (data set, engine, queries), run(state) makes one pass through
the package's public entry points and work(case) says what the pass cannot do
without.  Three kinds of input:

  db      a database of many small labelled graphs (half Erdos-Renyi, half
          Barabasi-Albert or as ba_fraction says) with random-walk queries;
  graph   one large Chung-Lu graph with hubs, with the five 5-vertex shapes
          or induced cyclic walk queries;
  files   the same database as .mygraph / .metadata files, for the driver
          that has the reference's shape.

All results are whole numbers (embedding counts, algorithmic bytes, matched
graphs), so there is nothing to compare with floating point.
"""
import os
import shutil
import tempfile
import weakref

import numpy as np

import geneva_amd as G


def _db(name, how, graphs, nmin, nmax, labels, zipf, queries, kmin, kmax, deg=4.0, ba=0.5, **more):
    c = {"kind": "db", "how": how, "graphs": graphs, "nmin": nmin, "nmax": nmax, "deg": deg, "ba": ba,
         "labels": labels, "zipf": zipf, "queries": queries, "kmin": kmin, "kmax": kmax, **more}
    return {"name": name, **c} if name else c


def _graph(name, how, vertices, gamma, deg, wmax, labels, zipf, **more):
    c = {"kind": "graph", "how": how, "vertices": vertices, "gamma": gamma, "deg": deg, "wmax": wmax,
         "labels": labels, "zipf": zipf, **more}
    return {"name": name, **c} if name else c


def _files(name, graphs, nmin, nmax, labels, queries, k, plan):
    c = {"kind": "files", "graphs": graphs, "nmin": nmin, "nmax": nmax, "labels": labels,
         "queries": queries, "k": k, "plan": plan}
    return {"name": name, **c} if name else c


def listed():
    return [
        # a small collection of small molecules-like graphs, asked one query at
        # a time: launches and host work per call are what the user waits for
        _db("mine_small_db", "mine", 1000, 10, 30, 8, 0.0, 10, 4, 4, deg=3.0, ba=0.0),
        # an ordinary database, one query per call, as an interactive user asks
        _db("mine_db", "mine", 20000, 20, 200, 32, 1.1, 24, 4, 8),
        # larger graphs with three edge labels (vertices renumbered for the
        # stored format), an odd number of them, single-vertex plans
        _db("mine_db_edge_labels", "mine", 3001, 60, 500, 20, 1.0, 13, 3, 7, edge_labels=3, single_v=True),
        # a handful of queries on the small collection in one call
        _db("batch_small_db", "batch", 1000, 10, 30, 8, 0.0, 10, 4, 4, deg=3.0, ba=0.0),
        # an ordinary batch: ragged numbers of graphs and queries
        _db("batch_db", "batch", 17321, 20, 200, 32, 1.1, 131, 3, 9),
        # the largest: 100,000 graphs, 256 queries of 4-8 vertices
        _db("batch_large_db", "batch", 100000, 20, 200, 32, 1.1, 256, 4, 8),
        # a burst of requests at a server that holds an ordinary database
        _db("serve_burst", "serve", 20000, 20, 200, 32, 1.1, 600, 3, 10),
        # the five 5-vertex shapes on a social-network-like graph, mid-sized
        # (other labels in every set of inputs) and large (the same labels)
        _graph("shapes_100k", "shapes", 100000, 2.1, 20.0, 600.0, 16, 1.2),
        _graph("shapes_1m", "shapes", 1000000, 2.1, 20.0, 1200.0, 16, 1.2, shape_seed=0x47454E02 + 100),
        # induced cyclic queries of 6-8 vertices on a graph with heavy hubs
        _graph("cyclic_hub_graph", "cyclic", 40000, 1.9, 30.0, 1000.0, 64, 1.0, queries=12, kmin=6, kmax=8),
        # walk queries on one large graph, all in one call
        _graph("batch_hub_graph", "batch", 50000, 2.1, 8.0, 200.0, 32, 1.0, queries=24, kmin=3, kmax=5),
        # the driver with the reference's phases and launchers, from files to
        # counts, one query file after the other
        _files("phase_driver", 5000, 10, 30, 8, 4, 4, "auto"),
    ]


def _spread(rng, lo, hi):
    """A whole number spread over the logarithm of [lo, hi]."""
    return int(round(lo * (hi / lo) ** rng.random()))


def draw(rng):
    family = rng.choice(("mine", "batch", "serve", "mine", "batch", "shapes", "cyclic", "batch_graph", "files"))
    if family in ("mine", "batch", "serve"):
        labels = rng.choice((12, 20, 32, 48, 64))
        kmax = rng.randint(4, 6 if labels < 20 else 8)
        kmin = rng.randint(3, kmax)
        nmin = rng.choice((10, 20, 40))
        nmax = rng.choice((31, 64, 130, 200, 400)) + rng.randint(0, 60)
        graphs = _spread(rng, 150, 2_500_000 // nmax)
        n = {"mine": rng.randint(3, 24), "batch": _spread(rng, 3, 200), "serve": _spread(rng, 30, 500)}[family]
        more = {"single_v": True} if family != "serve" and rng.random() < 0.25 else {}
        if rng.random() < 0.3:
            more["edge_labels"] = rng.randint(2, 4)
        return _db(None, family, graphs, nmin, max(nmax, nmin + 5), labels, rng.choice((0.0, 0.7, 1.1)), n, kmin,
                   kmax, deg=rng.choice((3.0, 4.0)), ba=rng.choice((0.0, 0.3, 0.5)), **more)
    if family == "shapes":
        return _graph(None, "shapes", _spread(rng, 20_000, 400_000), rng.choice((2.1, 2.3)),
                      rng.choice((10.0, 15.0, 20.0)), float(rng.randint(200, 600)), rng.choice((16, 24)), 1.2)
    if family == "cyclic":
        nv = _spread(rng, 12_000, 40_000)
        return _graph(None, "cyclic", nv, rng.choice((1.9, 2.1)), rng.choice((20.0, 30.0)), float(nv // 40), 64, 1.0,
                      queries=rng.randint(4, 12), kmin=5, kmax=7)
    if family == "batch_graph":
        return _graph(None, "batch", _spread(rng, 5_000, 50_000), 2.1, rng.choice((6.0, 8.0)), 200.0, 32, 1.0,
                      queries=rng.randint(5, 24), kmin=3, kmax=5)
    return _files(None, _spread(rng, 300, 8000), 10, rng.randint(20, 40), rng.choice((8, 12)), rng.randint(1, 4),
                  rng.randint(3, 5), rng.choice(("auto", "dv", "sv")))


def _database(case, seed):
    ds = G.Dataset.database(case["graphs"], case["nmin"], case["nmax"], case.get("deg", 3.0), case.get("ba", 0.0),
                            case["labels"], case.get("zipf", 0.0), 0x51000000 + seed)
    if case.get("edge_labels", 1) > 1:
        edges = ds.edges
        edges[:, 2] = np.random.default_rng(seed).integers(1, case["edge_labels"] + 1, size=len(edges))
        ds = G.Dataset.from_arrays(ds.vlabel, edges, ds.graph_of, ds.ngraphs)
        ds.reorder_intervals()   # the stored format holds at most 256 source intervals a label
    return ds


def prepare(case, seed):
    s = {"case": dict(case)}
    if case["kind"] == "db":
        ds = _database(case, seed)
        ds.add_walk_queries(case["queries"], case["kmin"], case["kmax"], seed=seed + 7)
        s["engine"] = G.Engine(ds)
        if case["how"] == "batch":
            s["engine"].batch_config(slots=264, slot_bytes=96 << 20, row_cap=1 << 28, ipt=8)
        elif case["how"] == "serve":
            s["engine"].batch_config(slots=128, slot_bytes=64 << 20, row_cap=1 << 27, ipt=8)
        s["queries"] = ds.queries
    elif case["kind"] == "graph":
        ds = G.Dataset.chung_lu(case["vertices"], case["gamma"], case["deg"], case["wmax"], case["labels"],
                                case["zipf"], 0x52000000 + seed)
        if case["how"] == "shapes":
            ds.add_shape_queries(case.get("shape_seed", seed + 7))
        elif case["how"] == "cyclic":
            ds.add_walk_queries(case["queries"], case["kmin"], case["kmax"], induced=True, min_extra=2,
                                seed=seed + 7, min_deg=2)
        else:
            ds.add_walk_queries(case["queries"], case["kmin"], case["kmax"], seed=seed + 7)
        # tables of a large graph get more room than the default
        s["engine"] = G.Engine(ds, level_bytes=2 << 30)
        if case["how"] == "batch":
            s["engine"].batch_config(slots=32, slot_bytes=256 << 20, row_cap=1 << 28, ipt=8)
        s["queries"] = ds.queries
    else:
        ds = _database(case, seed)
        ds.add_walk_queries(case["queries"], case["k"], case["k"], seed=seed + 7)
        d = tempfile.mkdtemp(prefix="geneva_cases_")
        holder = _Folder(d)
        ds.write(os.path.join(d, "db"))
        files = []
        for i, q in enumerate(ds.queries):
            files.append(os.path.join(d, f"q{i}.query"))
            with open(files[-1], "w") as f:
                f.write(q)
        s.update(folder=holder, mygraph=os.path.join(d, "db.mygraph"), metadata=os.path.join(d, "db.metadata"),
                 files=files, single_v={"auto": None, "dv": False, "sv": True}[case["plan"]])
    return s


class _Folder:
    """A temporary folder that goes with its state."""

    def __init__(self, path):
        self.path = path
        self._end = weakref.finalize(self, shutil.rmtree, path, True)


def _results(res):
    """Counts, algorithmic bytes and the matched-graph bitsets as they came
    back (MineResult.graph_ids decodes them when asked)."""
    out = {"count": np.array([r.count for r in res], dtype=np.uint64).view(np.int64),
           "alg_bytes": np.array([r.alg_bytes for r in res], dtype=np.uint64).view(np.int64)}
    if res[0]._words is not None:
        out["graphs"] = np.stack([r._words for r in res]).view(np.int32)
    return out


def run(s):
    case = s["case"]
    single_v = bool(case.get("single_v", False))
    if case["kind"] == "files":
        # the count, as the reference's own driver prints it
        got = [G.phase_mine(s["mygraph"], s["metadata"], f, single_v=s["single_v"], arena_bytes=64 << 20,
                            keep_rows=False) for f in s["files"]]
        return {"count": np.array([r.count for r in got], dtype=np.int64)}
    if case["how"] == "serve":
        # every request is there at once: the server works off a full queue
        _, counts, _ = s["engine"].serve(s["queries"], [0.0] * len(s["queries"]))
        return {"count": np.array(counts, dtype=np.uint64).view(np.int64)}
    if case["how"] == "batch":
        res, _ = s["engine"].mine_batch(s["queries"], single_v=single_v)
        return _results(res)
    return _results([s["engine"].mine(q, single_v=single_v) for q in s["queries"]])


def work(case):
    """Bytes: the graph read once (4 B a vertex for its label, 4 B per
    directed edge) by every call, and each query's results written once.
    The path has no floating point work."""
    if case["kind"] == "graph":
        vertices, degree, graphs = case["vertices"], case["deg"], 1
    else:
        graphs = case["graphs"]
        vertices = graphs * (case["nmin"] + case["nmax"]) / 2
        degree = case.get("deg", 3.0) * (1 - case.get("ba", 0.0)) + 4.0 * case.get("ba", 0.0)
    read = 4.0 * vertices * (1 + degree)
    queries = case.get("queries", 5)
    calls = 1 if case.get("how") in ("batch", "serve") else queries
    bits = graphs / 8 if graphs > 1 and case.get("how") in ("batch", "mine") else 0
    return {"bytes": calls * read + queries * (16.0 + bits), "flops": 0.0}


def exact(case, seed):
    """No floating point results: counts, bytes and ids are equal or wrong."""
    return None
