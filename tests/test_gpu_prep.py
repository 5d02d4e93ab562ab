"""Tree preparation at the sizes where it changes form: the smallest trees,
the step from 4 to 16 waves (256 nodes), the largest trees whose working
arrays fit LDS (5485 nodes) and the first that do not; trees of every shape
(paths, stars, combs nested half their nodes deep, random ones), full tables
against the oracle."""
import numpy as np
import pytest

import oracle
import xted

pytestmark = pytest.mark.gpu


def shaped(shape, n):
    parent = np.full(n, -1, np.int32)
    if shape == "path":
        parent[1:] = np.arange(n - 1)
    elif shape == "star":
        parent[1:] = 0
    elif shape == "comb":
        spine = n - n // 2
        parent[1:spine] = np.arange(spine - 1)
        for k in range(n // 2):
            parent[spine + k] = max(spine - 2 - k, 0)
    else:
        kind = {"rrt": xted.GEN_RRT, "deep": xted.GEN_DEEP, "wide": xted.GEN_SHALLOW}[shape]
        return xted.generate(kind, n, 5, xted.derive_seed(9303, n))
    return parent, (np.arange(n) * 11 % 5).astype(np.int32)


SHAPES = ("path", "star", "comb", "rrt", "deep", "wide")


@pytest.mark.parametrize("shape", SHAPES)
@pytest.mark.parametrize("n", [1, 2, 3, 4, 5, 7, 17, 64, 65, 255, 256, 257, 1025])
def test_small_trees(gpu_ctx, shape, n):
    y = shaped(shape, n)
    for x in (shaped("rrt", 23), y if n <= 300 else shaped(shape, 60)):
        d, td, _ = gpu_ctx.ted(x, y)
        od, otd, _ = oracle.ted(x, y, threads=8)
        assert d == od and np.array_equal(td, otd)


@pytest.mark.parametrize("shape", ["path", "star", "rrt", "deep", "wide"])
@pytest.mark.parametrize("n", [5485, 5486])
def test_trees_at_the_lds_limit(gpu_ctx, shape, n):
    x, y = shaped("rrt", 12), shaped(shape, n)
    d, td, _ = gpu_ctx.ted(x, y)
    od, otd, _ = oracle.ted(x, y, threads=8)
    assert d == od and np.array_equal(td, otd)


@pytest.mark.parametrize("shape", SHAPES)
@pytest.mark.parametrize("n", [5484, 5485])
def test_largest_tree_in_lds_and_the_next(gpu_ctx, shape, n):
    """5484 nodes fill the 150 KiB of LDS that preparation may take."""
    x, y = shaped("rrt", 12), shaped(shape, n)
    d, td, _ = gpu_ctx.ted(x, y)
    od, otd, _ = oracle.ted(x, y, threads=8)
    assert d == od and np.array_equal(td, otd)
