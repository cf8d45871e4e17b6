"""The FP64 matrix-core kernel (PLAIN64, BATCHED64, the recompute) where its
tiling can go wrong: vectors and family counts at the edges of 16-row tiles
and 16-family blocks, root ranges on either side of the vectors' length, all
launch shapes, more leaves than it stages in LDS, and polytomies.

Values are held to 1e-9 relative of the oracle (the path's bar); every launch
shape and both paths sum in the same order, so they agree bit for bit."""
import numpy as np
import pytest

from cafe5_amd import native, workloads as wl
from cafe5_amd.model import BaseModel
from oracle_lib import Oracle

pytestmark = pytest.mark.gpu
LAM = 0.004


@pytest.fixture(scope="module")
def eng():
    e = native.Engine(0)
    yield e
    e.close()


def _counts(tree, F, B, seed):
    rng = np.random.default_rng(seed)
    return wl.simulate_families(tree, 1 + rng.integers(0, max(1, B // 2), F), np.full(tree.n_nodes, LAM), seed,
                                cap=B)


def _lnl(eng, tree, counts, B, R, path):
    m = BaseModel(eng, tree, counts, B, R, path=path)
    m.infer_family_likelihoods(lambda r: Oracle.prior_uniform(r, r), LAM)
    return m.results.copy()


@pytest.mark.parametrize("B,R,F", [(1, 1, 1), (14, 15, 15), (15, 14, 16), (16, 16, 17), (31, 40, 33), (47, 20, 31),
                                   (63, 64, 65), (80, 33, 100), (130, 130, 48)])
def test_tile_edges(eng, B, R, F):
    tree = wl.yule_tree(9, 3)
    counts = _counts(tree, F, B, 100 + B)
    want = Oracle.evaluate(tree, np.full(tree.n_nodes, LAM), counts, B, R, Oracle.prior_uniform(R, R), threads=4)["lnl"]
    plain = _lnl(eng, tree, counts, B, R, native.PATH_PLAIN64)
    assert np.all(np.abs(plain - want) <= 1e-9 * np.abs(want))
    assert np.array_equal(plain, _lnl(eng, tree, counts, B, R, native.PATH_BATCHED64))


@pytest.mark.parametrize("shape", [(0, 1, True), (0, 1, False), (0, 2, False), (2, 1, True), (2, 2, False)])
@pytest.mark.parametrize("B", [30, 75, 120])
def test_shapes_agree(eng, shape, B):
    kernel, ntw, lds = shape
    tree = wl.yule_tree(12, 5)
    counts = _counts(tree, 75, B, 7)
    nt = (B + 1 + 15) // 16
    base = _lnl(eng, tree, counts, B, B, native.PATH_PLAIN64)
    w = (nt + ntw - 1) // ntw
    eng.tuning_set(native.PATH_BATCHED64, nt, tree.n_leaves, kernel, ntw, w, lds, 1)
    try:
        assert np.array_equal(base, _lnl(eng, tree, counts, B, B, native.PATH_BATCHED64))
    finally:
        eng.tuning_clear()


def _caterpillar(levels, size):
    """A chain of nodes, each over the node below it and `size` leaves."""
    n = levels * size + levels
    parent = np.full(n, -1, dtype=np.int32)
    col = np.full(n, -1, dtype=np.int32)
    for i in range(levels * size):
        parent[i], col[i] = levels * size + i // size, i
    parent[levels * size:n - 1] = np.arange(levels * size + 1, n)
    return wl.Tree(parent, col, np.where(parent < 0, 0.0, 2.0), [f"n{i}" for i in range(n)])


@pytest.mark.parametrize("levels,size", [(4, 3), (130, 4)])   # 12 leaves; 520, past the 512 staged ones
def test_polytomies_and_many_leaves(eng, levels, size):
    tree = _caterpillar(levels, size)
    B = 20
    counts = np.minimum(1 + np.random.default_rng(levels).integers(0, 3, (19, tree.n_leaves)), B).astype(np.int32)
    want = Oracle.evaluate(tree, np.full(tree.n_nodes, LAM), counts, B, B, Oracle.prior_uniform(B, B), threads=4)["lnl"]
    got = _lnl(eng, tree, counts, B, B, native.PATH_PLAIN64)
    ok = np.isfinite(want)
    assert np.array_equal(np.isfinite(got), ok)
    assert np.all(np.abs(got[ok] - want[ok]) <= 1e-9 * np.abs(want[ok]))
