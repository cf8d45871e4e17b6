"""Subtree patterns where one size class holds buckets of several bounds: the
per-lane kernel's instance is the class's, so a bucket whose own vectors would
take the 21-row instance writes and reads columns of 33 rows beside a larger
one.  Likelihoods against the FP64 path, and against the same families in pieces
too small to share, within the bars of the reduced paths."""
import numpy as np
import pytest

from bars import reduced_ok
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


def _prior(r):
    return Oracle.prior_uniform(r, r)


def _lnl(eng, tree, counts, B, path):
    m = BaseModel(eng, tree, counts, B, B, path=path)
    m.infer_family_likelihoods(_prior, LAM)
    return m.results.copy()


@pytest.mark.parametrize("path", native.REDUCED_PATHS)
@pytest.mark.parametrize("small,large", [(20, 28), (17, 32), (20, 22), (16, 31)])
def test_two_bounds_of_one_class(eng, path, small, large):
    # many families without a gene in some clade: the size-0 entry of their
    # columns is the one that a longer neighbour would overwrite
    tree = wl.yule_tree(20, 6)
    F = 2400
    rng = np.random.default_rng(small * large)
    counts = wl.simulate_families(tree, 1 + rng.integers(0, 6, F), np.full(tree.n_nodes, LAM), 9, cap=small)
    for a in range(0, tree.n_leaves, 4):
        counts[rng.random(F) < 0.4, a:a + 4] = 0
    counts[:, 0] = np.maximum(counts[:, 0], 1)
    B = np.where(np.arange(F) % 2, small, large).astype(np.int32)   # two buckets of 1,200
    got = _lnl(eng, tree, counts, B, path)
    want = _lnl(eng, tree, counts, B, native.PATH_PLAIN64)
    assert np.isfinite(want).all()
    assert np.all(reduced_ok(got, want)), np.argwhere(~reduced_ok(got, want))[:5]
    for i in range(0, F, 600):   # 300 families a bucket
        part = _lnl(eng, tree, counts[i:i + 600], B[i:i + 600], path)
        assert np.all(reduced_ok(got[i:i + 600], part)), i


def _comb(n):
    """A spine of n / 2 two-leaf clades (n leaves)."""
    h = n // 2
    parent = np.empty(n + h + h - 1, dtype=np.int32)
    leaf = np.full(len(parent), -1, dtype=np.int32)
    leaf[:n] = np.arange(n)
    parent[:n] = n + np.arange(n) // 2
    spine = n + h + np.arange(h - 1)   # spine[i] joins clade i + 1 and what is before it
    parent[n] = spine[0]
    parent[n + 1:n + h] = spine
    parent[spine[:-1]] = spine[1:]
    parent[spine[-1]] = -1
    length = np.where(leaf >= 0, 6.0, 1.0)
    length[spine[-1]] = 0.0
    return wl.Tree(parent, leaf, length, [f"n{i}" for i in range(len(parent))])


def wide_table(F, n):
    """Families whose two-leaf clades have few patterns and larger clades many."""
    rng = np.random.default_rng(n)
    base = 1 + rng.integers(0, 12, F)
    return (base[:, None] + np.where(rng.random((F, n)) < 0.08, rng.choice([-1, 1], (F, n)), 0)).astype(np.int32)


@pytest.mark.parametrize("n", [640, 700])
def test_wide_trees(eng, n):
    # with 32-family tiles the two-leaf clades' columns would take 160 KB of
    # LDS and more, the leaves half of it; 512 and more leaves share nothing
    # on the FP64 path
    tree = _comb(n)
    counts = wide_table(8300, n)
    B = np.full(len(counts), 40, dtype=np.int32)
    got = _lnl(eng, tree, counts, B, native.PATH_BATCHED32)
    want = _lnl(eng, tree, counts, B, native.PATH_PLAIN64)
    assert np.isfinite(want).all()
    assert np.all(reduced_ok(got, want)), np.argwhere(~reduced_ok(got, want))[:5]
