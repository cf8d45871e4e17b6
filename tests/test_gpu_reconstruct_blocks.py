"""Block edges of the reconstruction kernel: vectors that end inside, at and
just past a block of child sizes and a pass of rows, family counts around a
wave's four and around the one-per-wave rule, nodes with one and three
children, families close to the bound (no block can be skipped), and the
fixed scratch with and without room for the table of block maxima.  States are
integers: equal to the oracle's."""
import numpy as np
import pytest

from cafe5_amd import native, priors, workloads as wl
from oracle_lib import Oracle

pytestmark = pytest.mark.gpu

# ((0,1,2)6,((3,4)7)8,5)9: three children, one child, a leaf below the root
PARENT = np.array([6, 6, 6, 7, 7, 9, 9, 8, 9, -1], dtype=np.int32)
LEAF = np.array([0, 1, 2, 3, 4, 5, -1, -1, -1, -1], dtype=np.int32)


@pytest.fixture(scope="module")
def eng():
    e = native.Engine(0)
    yield e
    e.close()


@pytest.mark.parametrize("B,R,F", [(1, 1, 3), (15, 15, 9), (16, 9, 5), (127, 127, 511), (128, 90, 513), (129, 160, 514),
                                   (255, 255, 515), (512, 512, 514)])
def test_edges(eng, B, R, F):
    tree = wl.Tree(PARENT, LEAF, np.full(10, 7.0), [f"n{i}" for i in range(10)])
    lam = 0.01
    rng = np.random.default_rng(B)
    counts = np.minimum(rng.poisson(3.0, (F, 6)), B).astype(np.int32)
    counts[-1] = rng.integers(max(0, B - 3), B + 1, 6)
    counts[F // 2] = rng.integers(0, B + 1, 6)
    eng.set_tree(tree)
    eng.set_families(counts, B, R)
    keys = native.KeyTable()
    slots = keys.node_slots(tree, np.full((1, 10), lam))
    lq, tq = keys.arrays()
    N = max(B, R) + 4
    eng.matrix_reset(N, len(lq))
    eng.matrix_build(lq, tq, 0, native.BUILD_RECURRENCE)
    prior = priors.uniform(R, min(B, R) + 1)
    mats = (np.stack([eng.matrix_get(k) for k in range(len(lq))]), slots[0])   # the engine's own matrices
    got = eng.reconstruct(slots, prior, B, R)
    assert np.array_equal(eng.reconstruct(slots, prior, B, R, noalloc=True), got)
    for f in sorted({0, 1, F // 2, F - 2, F - 1}):
        want = Oracle.reconstruct(tree, counts[f], lam, B, R, prior, N=N, matrices=mats)
        assert np.array_equal(got[f], want), (f, counts[f], got[f], want)


def test_fixed_scratch_without_the_table(eng):
    # 127 interior branches at B = 900: the table (57 x 456 doubles each) would
    # leave the families less than half of the 32 MiB
    n_leaves = 129
    parent = np.full(2 * n_leaves - 1, -1, dtype=np.int32)
    leaf = np.full(2 * n_leaves - 1, -1, dtype=np.int32)
    leaf[:n_leaves] = np.arange(n_leaves)
    level, nxt = list(range(n_leaves)), n_leaves
    while len(level) > 1:
        up = []
        for a, b in zip(level[::2], level[1::2]):
            parent[a] = parent[b] = nxt
            up.append(nxt)
            nxt += 1
        level = up + level[len(level) // 2 * 2:]
    tree = wl.Tree(parent, leaf, np.full(len(parent), 5.0), [f"n{i}" for i in range(len(parent))])
    B = R = 900
    counts = np.random.default_rng(1).integers(0, 40, (5, n_leaves)).astype(np.int32)
    eng.set_tree(tree)
    eng.set_families(counts, B, R)
    keys = native.KeyTable()
    slots = keys.node_slots(tree, np.full((1, tree.n_nodes), 0.002))
    lq, tq = keys.arrays()
    eng.matrix_reset(B + 1, len(lq))
    eng.matrix_build(lq, tq, 0, native.BUILD_RECURRENCE)
    prior = priors.uniform(R, R + 1)
    got = eng.reconstruct(slots, prior, B, R)
    assert np.array_equal(eng.reconstruct(slots, prior, B, R, noalloc=True), got)
    mats = (np.stack([eng.matrix_get(k) for k in range(len(lq))]), slots[0])
    want = Oracle.reconstruct(tree, counts[2], 0.002, B, R, prior, N=B + 1, matrices=mats)
    assert np.array_equal(got[2], want)
