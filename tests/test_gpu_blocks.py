"""Column-blocked and swept tables at the edges of their blocks, lines and row
groups, against the oracle: column counts around whole blocks, row counts
around the 16-row lines and 64-row metadata chunks the edge waves work in,
right paths nested deeper than one lane per depth across a block edge, blocks
inside a captured graph that is replayed, and tables one wave sweeps 512
columns at a time."""
import numpy as np
import pytest

import oracle
import xted

pytestmark = pytest.mark.gpu


def tree(kind, n, index):
    return xted.generate(kind, n, 6, xted.derive_seed(9202, index))


def comb(n, alphabet=4):
    """Right paths nested n / 2 deep: every node of the spine has the rest of
    the spine as its first child and a leaf as its last."""
    parent = np.full(n, -1, np.int32)
    spine = n - n // 2
    parent[1:spine] = np.arange(spine - 1)
    for k in range(n // 2):
        parent[spine + k] = max(spine - 2 - k, 0)
    return parent, (np.arange(n) * 7 % alphabet).astype(np.int32)


def cost_model(seed, alphabet=6):
    rng = np.random.default_rng(seed)
    ren = rng.integers(0, 17, (alphabet, alphabet)).astype(np.int32)
    np.fill_diagonal(ren, 0)
    return (rng.integers(1, 9, alphabet).astype(np.int32),
            rng.integers(1, 9, alphabet).astype(np.int32), ren)


def expected(x, y, model):
    if model is None:
        return oracle.ted(x, y, threads=8)[:2]
    return oracle.ted_costs(x, y, model)


@pytest.mark.parametrize("form", range(6))
@pytest.mark.parametrize("seq_rows", [0, 1 << 20])
@pytest.mark.parametrize("costs", [False, True])
def test_block_and_line_edges(form, seq_rows, costs):
    width = xted.XL_BW[form]
    model = cost_model(41) if costs else None
    kinds = (xted.GEN_RRT, xted.GEN_DEEP, xted.GEN_SHALLOW)
    with xted.Context(0) as ctx:
        ctx.set_costs(model)
        ctx.force_class(27 + form, lane_enable=False)
        ctx.set_xl_rule(seq_rows)
        k = 0
        cols = [width - 1, width, width + 1]
        if width <= 512:
            cols += [2 * width, 3 * width + 1]
        for c in cols:
            for r in (2, 15, 17, 64, 66) if width <= 1024 else (17, 66):
                x, y = tree(kinds[k % 3], r, 2 * k), tree(kinds[(k // 3) % 3], c, 2 * k + 1)
                d, td, _ = ctx.ted(x, y)
                od, otd = expected(x, y, model)
                assert d == od and np.array_equal(td, otd), (r, c)
                k += 1


@pytest.mark.parametrize("form", [2, 3, 4, 5])
@pytest.mark.parametrize("costs", [False, True])
def test_nested_columns_across_blocks(form, costs):
    model = cost_model(42) if costs else None
    with xted.Context(0) as ctx:
        ctx.set_costs(model)
        ctx.force_class(27 + form, lane_enable=False)
        for depth in (62, 63, 64, 130, 255):
            y = comb(2 * depth + 1)
            for seq_rows in (0, 1 << 20):
                ctx.set_xl_rule(seq_rows)
                x = tree(xted.GEN_RRT, 40, depth)
                d, td, _ = ctx.ted(x, y)
                od, otd = expected(x, y, model)
                assert d == od and np.array_equal(td, otd), (depth, seq_rows)


def test_blocks_in_a_replayed_graph():
    """Every replay of captured launches tags its words anew."""
    with xted.Context(0) as ctx:
        ctx.force_class(27 + 5, lane_enable=False)
        ctx.set_xl_rule(0)
        trees = [tree(xted.GEN_DEEP, 300, 500 + i) for i in range(4)]
        ids = ctx.pool_add(trees)
        want = [oracle.ted(trees[0], trees[1], threads=8)[0],
                oracle.ted(trees[2], trees[3], threads=8)[0]]
        xs, ys = ids[[0, 2]].copy(), ids[[1, 3]].copy()
        for k in range(6):
            assert list(ctx.batch(xs, ys)[0]) == want
            if k == 2:
                assert list(ctx.batch(xs[1:], ys[1:])[0]) == want[1:]


@pytest.mark.parametrize("costs", [False, True])
def test_swept_tables(costs):
    """Many pairs of a short and a wide tree: the wide tables are a small part
    of their level, so one wave sweeps each."""
    model = cost_model(43) if costs else None
    with xted.Context(0) as ctx:
        ctx.set_costs(model)
        shapes = ((2, 1025, xted.GEN_RRT), (4, 1535, xted.GEN_SHALLOW), (5, 1536, xted.GEN_RRT),
                  (63, 1537, xted.GEN_SHALLOW), (17, 9000, xted.GEN_RRT), (40, 1600, xted.GEN_DEEP))
        for i, (r, c, kind) in enumerate(shapes):
            x, y = tree(xted.GEN_SHALLOW, r, 700 + i), tree(kind, c, 800 + i)
            od, otd = expected(x, y, model)
            ids = ctx.pool_add([x, y])
            xs, ys = np.full(2400, ids[0], np.int32), np.full(2400, ids[1], np.int32)
            ctx.set_profile(True)
            d, _, _ = ctx.batch(xs, ys)
            swept = ctx.class_profile().get(xted.CLASS_SWEEP)
            ctx.set_profile(False)
            assert swept is not None, (r, c)
            assert (d == od).all(), (r, c)
            shape = (len(x[0]), len(y[0]))
            d, tds, _ = ctx.batch(xs, ys, [shape if k % 1199 == 0 else None for k in range(2400)])
            assert (d == od).all()
            assert all(np.array_equal(t, otd) for t in tds if t is not None)
            ctx.pool_clear()
