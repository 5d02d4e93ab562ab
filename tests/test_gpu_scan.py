"""On-chip row scans at the edges of their blocks, rings and row groups, full
tables against the oracle: column counts around whole blocks of 64 columns
per lane and wave, row counts around the prefetch ring, the row groups the
waves agree on and the 64-row metadata chunks, right paths nested deeper than
one lane per depth (more than 62 imports across a block edge), and the form
with shared slot rows that takes tables whose imports do not fit LDS."""
import numpy as np
import pytest

import oracle
import xted

pytestmark = pytest.mark.gpu


def row_class(waves, cpl):
    return 1 + 5 * (waves.bit_length() - 1) + (cpl.bit_length() - 1)


def tree(kind, n, index):
    return xted.generate(kind, n, 6, xted.derive_seed(9101, index))


def comb(n, alphabet=4):
    """Every second node's first child holds the rest of the tree and its last
    child is a leaf: right paths nested n / 2 deep."""
    parent = np.full(n, -1, np.int32)
    m = n // 2  # spine nodes 0 .. n-m-1 in preorder, then their leaves inside out
    spine = n - m
    for i in range(1, spine):
        parent[i] = i - 1
    for k in range(m):
        parent[spine + k] = spine - 2 - k if spine - 2 - k >= 0 else 0
    label = (np.arange(n) * 7 % alphabet).astype(np.int32)
    return parent, label


def check(ctx, x, y, costs=None):
    d, td, _ = ctx.ted(x, y)
    if costs is None:
        od, otd, _ = oracle.ted(x, y, threads=8)
    else:
        od, otd = oracle.ted_costs(x, y, costs)
    assert d == od
    assert np.array_equal(td, otd)


def cost_model(alphabet, seed):
    rng = np.random.default_rng(seed)
    ren = rng.integers(0, 17, (alphabet, alphabet)).astype(np.int32)
    np.fill_diagonal(ren, 0)
    return (rng.integers(1, 9, alphabet).astype(np.int32),
            rng.integers(1, 9, alphabet).astype(np.int32), ren)


@pytest.mark.parametrize("waves,cpl", [(1, 1), (1, 16), (2, 1), (2, 4), (4, 1), (4, 2), (8, 1)])
@pytest.mark.parametrize("costs", [False, True])
def test_block_and_row_group_edges(waves, cpl, costs):
    block = 64 * cpl
    full = block * waves
    model = cost_model(6, 31) if costs else None
    with xted.Context(0) as ctx:
        ctx.set_costs(model)
        ctx.force_class(row_class(waves, cpl), lane_enable=False)
        kinds = (xted.GEN_RRT, xted.GEN_DEEP, xted.GEN_SHALLOW)
        cols = sorted({min(full, max(2, c)) for c in (block - 1, block, block + 1, full - 1, full)})
        rows = (2, 4, 5, 8, 9, 63, 64, 65)
        k = 0
        for c in cols:
            for r in rows:
                if r > c:
                    continue
                x, y = tree(kinds[k % 3], r, 2 * k), tree(kinds[(k // 3) % 3], c, 2 * k + 1)
                check(ctx, x, y, model)
                if k % 4 == 0:
                    check(ctx, y, x, model)
                k += 1


@pytest.mark.parametrize("waves,cpl", [(2, 2), (4, 1), (2, 4)])
@pytest.mark.parametrize("costs", [False, True])
def test_deeply_nested_columns(waves, cpl, costs):
    """Column keyroots nested 31, 63, 64, 65 and 120 deep: the imports of a
    saved row fit one lane each up to 62."""
    model = cost_model(6, 32) if costs else None
    with xted.Context(0) as ctx:
        ctx.set_costs(model)
        ctx.force_class(row_class(waves, cpl), lane_enable=False)
        for depth in (31, 62, 63, 64, 65, 120):
            if 2 * depth + 1 > 64 * waves * cpl:
                continue
            y = comb(2 * depth + 1)
            for i, kind in enumerate((xted.GEN_RRT, xted.GEN_DEEP, xted.GEN_SHALLOW)):
                check(ctx, tree(kind, 25, 300 + i), y, model)
            check(ctx, comb(20), y, model)


def test_shared_slot_rows():
    """A deep column keyroot whose imports do not fit beside the slot rows."""
    x, y = comb(120), comb(1100)
    with xted.Context(0) as ctx:
        ctx.set_profile(True)
        check(ctx, x, y)
        classes = ctx.class_profile()
        assert any(xted.class_name(c).startswith("shared") for c in classes), classes
        with pytest.raises(xted.XtedError):
            ctx.force_class(xted.CLASS_SHARED)


@pytest.mark.parametrize("waves,cpl", [(4, 8), (8, 4), (16, 2)])
def test_forced_class_on_tall_tables(waves, cpl):
    """The rule splits the largest tables of this pair over workgroups; a
    forced row-scan class takes them all the same."""
    x, y = tree(xted.GEN_RRT, 400, 900), tree(xted.GEN_RRT, 1300, 901)
    split = range(27, 33)
    with xted.Context(0) as ctx:
        ctx.set_profile(True)
        check(ctx, x, y)
        assert any(c in split for c in ctx.class_profile())
        cls = row_class(waves, cpl)
        ctx.force_class(cls, lane_enable=True)
        check(ctx, x, y)
        assert set(ctx.class_profile()) == {xted.CLASS_LANE, cls}


def comb_and_star(comb_nodes, leaves):
    """A root over a comb and that many leaves: nested as deep as the comb."""
    parent, _ = comb(comb_nodes)
    n = 1 + comb_nodes + leaves
    out = np.zeros(n, np.int32)
    out[0] = -1
    out[1:1 + comb_nodes] = parent + 1
    return out, (np.arange(n) * 5 % 4).astype(np.int32)


@pytest.mark.parametrize("waves,rows,leaves", [(4, 100, 900), (8, 60, 2000), (16, 30, 4500)])
@pytest.mark.parametrize("costs", [False, True])
def test_every_shared_slot_form(waves, rows, leaves, costs):
    """Columns nested 299 deep, above what column blocks hold, in trees of
    1501, 2601 and 5101 nodes whose waves' imports do not fit LDS."""
    model = cost_model(4, 33) if costs else None
    x, y = comb(rows), comb_and_star(600, leaves)
    with xted.Context(0) as ctx:
        ctx.set_costs(model)
        ctx.set_profile(True)
        check(ctx, x, y, model)
        assert f"shared_w{waves}_c8" in {xted.class_name(c) for c in ctx.class_profile()}
        check(ctx, y, x, model)


@pytest.mark.parametrize("waves,cpl", [(2, 8), (2, 16), (8, 2), (8, 8), (16, 8)])
@pytest.mark.parametrize("costs", [False, True])
def test_edges_of_wide_forms(waves, cpl, costs):
    """Several active waves of 8 and 16 columns per lane, and 16 of them."""
    block = 64 * cpl
    full = block * waves
    model = cost_model(6, 34) if costs else None
    with xted.Context(0) as ctx:
        ctx.set_costs(model)
        ctx.force_class(row_class(waves, cpl), lane_enable=False)
        ctx.set_profile(True)
        kinds = (xted.GEN_RRT, xted.GEN_SHALLOW)
        k = 0
        for c in (block + 1, full - block, full - 1, full):
            for r in (2, 9, 65):
                x, y = tree(kinds[k % 2], r, 600 + 2 * k), tree(kinds[(k + 1) % 2], c, 601 + 2 * k)
                check(ctx, x, y, model)
                assert set(ctx.class_profile()) == {row_class(waves, cpl)}
                k += 1
