"""Tables on their way out (Context::copy_tables): batches whose tables fill
the pinned buffer several times over, tables left out, and a caller's tables
that overlap, which are written one after another."""
import ctypes

import numpy as np
import pytest

import oracle
import xted

pytestmark = pytest.mark.gpu


def tree(n, index):
    return xted.generate(xted.GEN_RRT, n, 9, xted.derive_seed(9505, index))


def batch_into(ctx, xs, ys, outs):
    """xted_batch with the int32 tables' addresses given (0: not wanted)."""
    dist = np.empty(len(xs), np.int32)
    arr = (ctypes.c_void_p * len(xs))(*[o or None for o in outs])
    ints = ctypes.POINTER(ctypes.c_int32)
    st = xted.lib().xted_batch(ctx._h, len(xs), xs.ctypes.data_as(ints), ys.ctypes.data_as(ints),
                               dist.ctypes.data_as(ints), ctypes.cast(arr, ctypes.c_void_p), None)
    assert st == xted.OK
    return dist


@pytest.mark.parametrize("groups", [1, 2])
def test_tables_that_fill_the_buffer_again_and_again(groups):
    """12 million entries, 2 million to a half of the buffer; every third
    table is not wanted."""
    sizes = [(1700, 1600), (1, 1), (300, 7), (1500, 1900), (256, 256), (1601, 1999), (65, 3)]
    trees = [(tree(m, 2 * i), tree(n, 2 * i + 1)) for i, (m, n) in enumerate(sizes)] * 2
    want = {i: oracle.ted(*p, threads=8) for i, p in enumerate(trees[:len(sizes)])}
    with xted.Context(0) as ctx:
        ctx.set_batch_groups(groups, split_min=2)
        ids = ctx.pool_add([t for p in trees for t in p])
        shapes = [(len(x[0]), len(y[0])) if i % 3 else None for i, (x, y) in enumerate(trees)]
        for _ in range(2):
            dist, tds, _ = ctx.batch(ids[0::2].copy(), ids[1::2].copy(), shapes)
            for i, td in enumerate(tds):
                assert dist[i] == want[i % len(sizes)][0]
                assert td is None if i % 3 == 0 else np.array_equal(td, want[i % len(sizes)][1]), i


def test_tables_that_overlap():
    """Two tables in one place, the second's end in the first's, and one of
    them alone: the memory holds what writing them in order leaves."""
    pairs = [(tree(400, 50), tree(500, 51)), (tree(300, 52), tree(420, 53)),
             (tree(500, 54), tree(400, 55))]
    want = [oracle.ted(*p, threads=8)[1].ravel() for p in pairs]
    with xted.Context(0) as ctx:
        ids = ctx.pool_add([t for p in pairs for t in p])
        xs, ys = ids[0::2].copy(), ids[1::2].copy()
        for at in ((0, 0, 0), (0, 100_000, 150_001), (150_000, 60_000, 0), (0, 200_000, 326_000)):
            buf = np.full(800_000, -7, np.int32)
            ref = buf.copy()
            for o, w in zip(at, want):
                ref[o:o + len(w)] = w
            batch_into(ctx, xs, ys, [buf.ctypes.data + 4 * o for o in at])
            assert np.array_equal(buf, ref), at
