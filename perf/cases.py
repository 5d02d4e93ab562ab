"""Measured cases: what users of this library have it compute, through its
Python entry points (x-ted_amd/xted.py), from one pair of 100-node trees to
4096 pairs at once and one pair of 20,000 nodes.

Four kinds of call:

  pair    Context.ted on two host trees: upload, preprocessing, plan, forest
          DP and, with "table", the full n_x x n_y tree-distance table back
          on the host (the drop-in path).
  batch   Context.batch over pairs of a pool that is resident on the device:
          the distances of all pairs (and, with "table", their tables).
  matrix  Context.all_pairs: the distance matrix of a set of host trees.
  serve   the continuous-batching server: queries over a resident pool
          submitted at once, polled until every one is answered.

Trees come from the library's seeded generators: "rrt" (random recursive),
"deep" (narrow, fan-out 0..3), "wide" (shallow, about 40 children of the
root) or "mixed" (deep or wide, half and half). Node counts of a set are
uniform in [lo, hi], or log-uniform for the server's pool. "costs" runs
under a per-label cost model (deletions and insertions in 1..8, renames in
0..16), otherwise costs are one. "stored" applies the tuned granularity rule
that the package ships (x-ted_amd/tuning.json), as bench.py does; the rest
run with a new context's defaults.
"""
import math
import os
import sys

import numpy as np

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))),
                                "x-ted_amd"))

import autotune  # noqa: E402
import xted  # noqa: E402

_KIND = {"rrt": xted.GEN_RRT, "deep": xted.GEN_DEEP, "wide": xted.GEN_SHALLOW}
# Integer operations one interior forest cell takes: two adds, a compare or
# second add, two minima.
_OPS_PER_CELL = 5


def _pair(name, shape, nx, ny, alphabet, table, costs=False):
    return {"name": name, "kind": "pair", "shape": shape, "nx": nx, "ny": ny,
            "alphabet": alphabet, "table": table, "costs": costs}


def _batch(name, pairs, lo, hi, alphabet=200, shape="mixed", table=False, costs=False,
           stored=False):
    return {"name": name, "kind": "batch", "shape": shape, "pairs": pairs, "lo": lo, "hi": hi,
            "alphabet": alphabet, "table": table, "costs": costs, "stored": stored}


def listed():
    return [
        # The smallest call: one pair, distance and table; latency and
        # launches are all of it.
        _pair("pair_rrt_100", "rrt", 100, 100, 50, True),
        # The drop-in's ordinary use: 1000-node pairs of either shape, with
        # the table copied out (4 MB).
        _pair("pair_deep_1000", "deep", 1000, 1000, 200, True),
        _pair("pair_wide_1000", "wide", 1000, 1000, 1000, True),
        # A large tree against a small odd-sized one.
        _pair("pair_uneven_4999x237", "deep", 4999, 237, 200, True),
        # The largest single pair, distance only (its table stays on the device).
        _pair("pair_rrt_20000", "rrt", 20000, 20000, 500, False),
        # A handful of small resident pairs: a request of an interactive tool.
        _batch("batch_33_small", 33, 20, 150, alphabet=50, shape="rrt"),
        # Pairs whose tables are wanted too (for mappings, subtree joins).
        _batch("batch_128_tables", 128, 100, 600, table=True),
        # The throughput workload: thousands of uneven pairs, tuned rule.
        _batch("batch_4096", 4096, 100, 1000, stored=True),
        # Weighted edits (per-label costs), default rule.
        _batch("batch_1024_costs", 1024, 100, 1000, costs=True),
        # Similarity join of a data set, uploaded and joined in one call.
        {"name": "matrix_96", "kind": "matrix", "shape": "mixed", "trees": 96, "lo": 50,
         "hi": 1000, "alphabet": 200},
        # Serving: a burst of queries of very different sizes.
        {"name": "serve_64", "kind": "serve", "shape": "mixed", "queries": 64, "pool": 512,
         "lo": 50, "hi": 5000, "alphabet": 200},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["pair", "pair", "batch", "batch", "batch", "matrix", "serve"])
    if kind == "pair":
        # Sizes over 100..20,000; the largest pairs distance only, as in use.
        nx, ny = _log_int(rng, 100, 20000), _log_int(rng, 100, 20000)
        table = nx * ny <= 1 << 24
        # Deep and wide trees above 5000 nodes are not in use here.
        shape = rng.choice(["rrt", "deep", "wide"]) if max(nx, ny) <= 5000 else "rrt"
        c = _pair("", shape, nx, ny, rng.choice([50, 200, 500, 1000]), table)
    elif kind == "batch":
        pairs = _log_int(rng, 33, 2048)
        hi = _log_int(rng, 150, 1000)
        lo = max(20, hi // rng.randint(2, 10))
        costs = rng.random() < 0.3
        table = pairs <= 160 and rng.random() < 0.5
        c = _batch("", pairs, lo, hi, alphabet=rng.choice([50, 200]),
                   shape=rng.choice(["rrt", "mixed", "mixed"]), table=table, costs=costs,
                   stored=rng.random() < 0.5)
    elif kind == "matrix":
        c = {"kind": "matrix", "shape": "mixed", "trees": rng.randint(24, 96), "lo": 50,
             "hi": _log_int(rng, 200, 1000), "alphabet": 200}
    else:
        c = {"kind": "serve", "shape": "mixed", "queries": _log_int(rng, 8, 64),
             "pool": rng.randint(64, 512), "lo": 50, "hi": _log_int(rng, 500, 5000),
             "alphabet": 200}
    c.pop("name", None)
    return c


# ---- inputs ------------------------------------------------------------------

def _tree(case, n, seed, index):
    s = xted.derive_seed(seed, index)
    shape = case["shape"]
    if shape == "mixed":
        shape = "deep" if (s >> 40) & 1 else "wide"
    return xted.generate(_KIND[shape], n, case["alphabet"], s)


def _sizes(case, count):
    # One list of node counts a case: seeds change the trees, not how large
    # the k-th of them is (so that the tables have the same shapes).
    rng = np.random.default_rng([count, case["lo"], case["hi"]])
    if case["kind"] == "serve":
        return np.exp(rng.uniform(math.log(case["lo"]), math.log(case["hi"]), count)).round()
    return rng.integers(case["lo"], case["hi"] + 1, count)


def _trees(case, seed):
    if case["kind"] == "pair":
        sizes = [case["nx"], case["ny"]]
    else:
        count = {"batch": 2 * case.get("pairs", 0), "matrix": case.get("trees", 0),
                 "serve": case.get("pool", 0)}[case["kind"]]
        sizes = _sizes(case, count)
    return [_tree(case, int(n), seed, i) for i, n in enumerate(sizes)]


def _costs(case, seed):
    a = case["alphabet"]
    rng = np.random.default_rng([seed, 2])
    dele = rng.integers(1, 9, a).astype(np.int32)
    ins = rng.integers(1, 9, a).astype(np.int32)
    ren = rng.integers(0, 17, (a, a)).astype(np.int32)
    np.fill_diagonal(ren, 0)
    return dele, ins, ren


def _queries(case, seed):
    rng = np.random.default_rng([seed, 3])
    return (rng.integers(0, case["pool"], case["queries"]),
            rng.integers(0, case["pool"], case["queries"]))


def prepare(case, seed):
    trees = _trees(case, seed)
    ctx = xted.Context(0)
    if case.get("stored"):
        autotune.apply(ctx, autotune.load())
    if case.get("costs"):
        ctx.set_costs(_costs(case, seed))
    state = {"case": case, "ctx": ctx, "trees": trees}
    if case["kind"] in ("batch", "serve"):
        ids = ctx.pool_add(trees)
        if case["kind"] == "batch":
            state["xs"], state["ys"] = ids[0::2].copy(), ids[1::2].copy()
            if case["table"]:
                state["shapes"] = [(len(trees[2 * i][0]), len(trees[2 * i + 1][0]))
                                   for i in range(case["pairs"])]
        else:
            qx, qy = _queries(case, seed)
            state["queries"] = [(int(ids[x]), int(ids[y])) for x, y in zip(qx, qy)]
            state["server"] = xted.Server(ctx, hbm_budget=32 << 30)
    return state


def run(state):
    case, ctx = state["case"], state["ctx"]
    if case["kind"] == "pair":
        dist, td, _ = ctx.ted(state["trees"][0], state["trees"][1], want_td=case["table"])
        return [dist, td] if case["table"] else [dist]
    if case["kind"] == "batch":
        dist, tds, _ = ctx.batch(state["xs"], state["ys"], state.get("shapes"))
        # The tables one after another, as a caller that stores them has them.
        return [dist, np.concatenate([t.ravel() for t in tds])] if tds else [dist]
    if case["kind"] == "matrix":
        return [ctx.all_pairs(state["trees"])[0]]
    server, queries = state["server"], state["queries"]
    for tag, (x, y) in enumerate(queries):
        server.submit(x, y, tag)
    dist = np.full(len(queries), -1, np.int64)
    left = len(queries)
    while left:
        for tag, status, d, _, _ in server.poll(cap=len(queries), timeout_ms=20):
            if status != xted.OK:
                raise RuntimeError(f"query {tag}: status {status}")
            dist[tag] = d
            left -= 1
    return [dist]


def _index_pairs(case, seed):
    """Index pairs (into _trees) whose distances one pass computes."""
    if case["kind"] == "pair":
        return [(0, 1)]
    if case["kind"] == "batch":
        return [(2 * i, 2 * i + 1) for i in range(case["pairs"])]
    if case["kind"] == "matrix":
        n = case["trees"]
        return [(i, j) for i in range(n) for j in range(i + 1, n)]
    qx, qy = _queries(case, seed)
    return list(zip(qx.tolist(), qy.tolist()))


def work(case):
    """Bytes: every input tree (parent and label) once, every distance and
    every returned table once. Operations: the interior forest cells of all
    keyroot-pair tables (S_x * S_y a pair, S the summed keyroot subtree
    sizes) of one seed's trees."""
    trees = _trees(case, 1)
    s = [xted.tree_stats(t[0])[0] for t in trees]
    n = [len(t[0]) for t in trees]
    pairs = _index_pairs(case, 1)
    cells = sum(s[i] * s[j] for i, j in pairs)
    out = 4 * sum(n[i] * n[j] for i, j in pairs) if case.get("table") else 0
    used = sorted({i for p in pairs for i in p})
    return {"bytes": 8 * sum(n[i] for i in used) + 4 * len(pairs) + out,
            "flops": _OPS_PER_CELL * cells}


# ---- exact values --------------------------------------------------------------

def _structure(parent):
    """orl (last node of each subtree) and the keyroots (the root and every
    node that is not a last child), ascending."""
    n = len(parent)
    orl = np.arange(n)
    for i in range(n - 1, 0, -1):
        orl[parent[i]] = max(orl[parent[i]], orl[i])
    return orl, [i for i in range(n) if i == 0 or orl[i] != orl[parent[i]]]


def _table(x, y, costs):
    """The tree-distance table of x and y in 64-bit numbers: the textbook
    recurrence, keyroot pairs from the last to the first, a row at a time."""
    (px, lx), (py, ly) = x, y
    if costs is None:
        dele, ins = np.ones(len(px), np.int64), np.ones(len(py), np.int64)
        ren = (lx[:, None] != ly[None, :]).astype(np.int64)
    else:
        dele, ins = costs[0].astype(np.int64)[lx], costs[1].astype(np.int64)[ly]
        ren = costs[2].astype(np.int64)[np.ix_(lx, ly)]
    ox, kx = _structure(px)
    oy, ky = _structure(py)
    td = np.zeros((len(px), len(py)), np.int64)
    pins = np.concatenate([[0], np.cumsum(ins)])
    for j0 in reversed(ky):
        j1 = int(oy[j0]) + 1
        w = j1 - j0
        q = pins[j1] - pins[j0:j1 + 1]  # inserting the nodes from each column on
        far_col = oy[j0:j1] + 1 - j0
        tree_col = oy[j0:j1] == j1 - 1
        for i0 in reversed(kx):
            i1 = int(ox[i0]) + 1
            f = np.zeros((i1 - i0 + 1, w + 1), np.int64)
            f[-1] = q
            for i in range(i1 - 1, i0 - 1, -1):
                r = i - i0
                far = f[int(ox[i]) + 1 - i0][far_col] + td[i, j0:j1]
                if ox[i] == i1 - 1:
                    far = np.where(tree_col, f[r + 1, 1:] + ren[i, j0:j1], far)
                a = np.empty(w + 1, np.int64)
                a[:-1] = np.minimum(far, f[r + 1, :-1] + dele[i])
                a[-1] = f[r + 1, -1] + dele[i]
                f[r] = np.minimum.accumulate((a - q)[::-1])[::-1] + q
                if ox[i] == i1 - 1:
                    td[i, j0:j1] = np.where(tree_col, f[r, :-1], td[i, j0:j1])
    return td


def exact(case, seed):
    trees = _trees(case, seed)
    stats = [xted.tree_stats(t[0]) for t in trees]
    pairs = _index_pairs(case, seed)
    rows = sum(stats[i][0] * stats[j][2] for i, j in pairs)
    cells = sum(stats[i][0] * stats[j][0] for i, j in pairs)
    if rows > 400_000 or cells > 100_000_000:
        return None
    costs = _costs(case, seed) if case.get("costs") else None
    tds = [_table(trees[i], trees[j], costs) for i, j in pairs]
    dist = np.array([t[0, 0] for t in tds])
    if case["kind"] == "pair":
        return [int(dist[0]), tds[0]] if case["table"] else [int(dist[0])]
    if case["kind"] == "batch":
        return [dist, np.concatenate([t.ravel() for t in tds])] if case["table"] else [dist]
    if case["kind"] == "matrix":
        m = np.zeros((case["trees"],) * 2, np.int64)
        for (i, j), d in zip(pairs, dist):
            m[i, j] = m[j, i] = d
        return [m]
    return [dist]
