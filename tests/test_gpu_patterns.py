"""Subtree patterns: tables of 512 families and more share the work of equal
subtrees, smaller ones do not.  A table evaluated whole and in pieces of 300 has
to give the same values: the FP64 paths bit for bit (a shared column holds the
same sums), the reduced paths within their bars.  Trees with nodes of one and
three children and units under the root; counts at the bound; several sizes,
points and categories; error models."""
import numpy as np
import pytest

from bars import reduced_ok
from cafe5_amd import native, workloads as wl
from cafe5_amd.model import BaseModel, GammaModel
from oracle_lib import Oracle

pytestmark = pytest.mark.gpu
LAM = 0.004

# (((0,1,2)11,(3,4)12)14,((5)13,6)15,7)17-(8,9)16 under the root 18, leaf 10 beside
PARENT = np.array([11, 11, 11, 12, 12, 13, 15, 17, 16, 16, 18, 14, 14, 15, 17, 17, 18, 18, -1], dtype=np.int32)
LEAF = np.array(list(range(11)) + [-1] * 8, dtype=np.int32)


def _odd_tree():
    return wl.Tree(PARENT, LEAF, 4.0 + np.arange(19) % 5, [f"n{i}" for i in range(19)])


@pytest.fixture(scope="module")
def eng():
    e = native.Engine(0)
    yield e
    e.close()


def _counts(tree, F, B, seed):
    rng = np.random.default_rng(seed)
    c = wl.simulate_families(tree, np.where(rng.random(F) < 0.9, 1 + rng.integers(0, 4, F), 1 + rng.integers(0, B, F)),
                             np.full(tree.n_nodes, LAM), seed, cap=B)
    c[0] = B
    c[F - 1] = rng.integers(0, B + 1, tree.n_leaves)
    return c


def _prior(r):
    return Oracle.prior_uniform(r, r)


def _lnl(eng, tree, counts, B, R, path, err=None):
    m = BaseModel(eng, tree, counts, B, R, path=path, error_model=err)
    m.infer_family_likelihoods(_prior, LAM)
    return m.results.copy()


def _pieces(eng, tree, counts, B, R, path, err=None):
    B, R = np.broadcast_to(B, len(counts)), np.broadcast_to(R, len(counts))
    return np.concatenate([_lnl(eng, tree, counts[i:i + 300], B[i:i + 300], R[i:i + 300], path, err)
                           for i in range(0, len(counts), 300)])


def _same(path, got, want):
    if path in native.REDUCED_PATHS:   # (equal infinities are equal)
        assert np.array_equal(np.isfinite(got), np.isfinite(want))
        fin = np.isfinite(want)
        assert np.array_equal(got[~fin], want[~fin])
        assert np.all(reduced_ok(got[fin], want[fin])), np.argwhere(~reduced_ok(got[fin], want[fin]))[:5]
    else:
        assert np.array_equal(got, want), np.argwhere(got != want)[:5]


PATHS = [native.PATH_PLAIN64, native.PATH_BATCHED64, native.PATH_BATCHED32, native.PATH_BATCHED16]


@pytest.mark.parametrize("path", PATHS)
@pytest.mark.parametrize("odd,B,R,F", [(True, 40, 33, 1025), (True, 63, 64, 1100), (False, 100, 100, 1300),
                                       (True, 130, 150, 1031), (False, 260, 200, 1024), (True, 540, 540, 1027)])
def test_whole_against_pieces(eng, path, odd, B, R, F):
    tree = _odd_tree() if odd else wl.yule_tree(14, 3)
    counts = _counts(tree, F, B, B + F)
    got = _lnl(eng, tree, counts, B, R, path)
    _same(path, got, _pieces(eng, tree, counts, B, R, path))
    for f in (0, 1, F // 2, F - 1) if B <= 130 else ():
        want = Oracle.evaluate(tree, np.full(tree.n_nodes, LAM), counts[f:f + 1], B, R, _prior(R), threads=1)["lnl"]
        assert abs(got[f] - want[0]) <= 1e-5 * abs(want[0]), f


@pytest.mark.parametrize("path", PATHS)
def test_two_sizes_and_an_error_model(eng, path):
    tree = _odd_tree()
    counts = _counts(tree, 1700, 44, 5)
    B = np.where(np.arange(1700) % 17 < 10, 50, 120).astype(np.int32)   # one bucket of 1,000, one of 700
    e = 0.05
    err = np.tile([e, 1.0 - 2 * e, e], (121, 1))
    err[0] = (0.0, 1.0 - e, e)
    _same(path, _lnl(eng, tree, counts, B, B, path, err), _pieces(eng, tree, counts, B, B, path, err))


@pytest.mark.parametrize("path", PATHS)
def test_categories_and_points(eng, path):
    tree = wl.yule_tree(16, 9)
    counts = _counts(tree, 900, 60, 11)
    args = (60, 60, np.full(3, 1 / 3), np.array([0.3, 0.9, 1.8]))
    whole = GammaModel(eng, tree, counts, *args, path=path)
    whole.infer_family_likelihoods(_prior, LAM)
    got = whole.results["lnl"].copy()
    parts = []
    for i in range(0, 900, 300):
        m = GammaModel(eng, tree, counts[i:i + 300], *args, path=path)
        m.infer_family_likelihoods(_prior, LAM)
        parts.append(m.results["lnl"].copy())
    _same(path, got, np.concatenate(parts))
    m = BaseModel(eng, tree, counts, 60, 60, path=path)
    m.infer_grid(_prior, [0.002, LAM, 0.006])
    grid = m.grid_lnl[1].copy()
    _same(path, grid, _lnl(eng, tree, counts, 60, 60, path))


def test_patterns_follow_the_table(eng):
    # another table, another tree, the first again: each finds its own patterns
    a, b = wl.yule_tree(14, 3), _odd_tree()
    ca, cb = _counts(a, 1200, 48, 1), _counts(b, 1300, 48, 2)
    first = _lnl(eng, a, ca, 48, 48, native.PATH_BATCHED64)
    other = _lnl(eng, b, cb, 48, 48, native.PATH_BATCHED64)
    assert np.array_equal(first, _lnl(eng, a, ca, 48, 48, native.PATH_BATCHED64))
    assert np.array_equal(other, _pieces(eng, b, cb, 48, 48, native.PATH_BATCHED64))
    keys = native.KeyTable()   # the tree set again after the families
    slots = keys.node_slots(a, np.full((1, a.n_nodes), LAM))
    eng.set_tree(a)
    eng.set_families(ca, bound_B=np.full(1200, 48), bound_R=np.full(1200, 48))
    eng.set_tree(a)
    eng.matrix_reset(49, len(keys.keys))
    eng.matrix_build(*keys.arrays())
    r = eng.evaluate(slots, _prior(48), native.PATH_BATCHED64)
    assert np.array_equal(r["lnl"][0], first)


@pytest.mark.parametrize("path", native.REDUCED_PATHS)
@pytest.mark.parametrize("B,R,F,error", [(20, 20, 1100, False), (9, 14, 600, False), (20, 12, 1025, True),
                                         (32, 32, 1300, False), (24, 30, 777, True)])
def test_one_family_per_lane(eng, path, B, R, F, error):
    # the per-lane kernel's sizes: columns of 21 and 33 rows
    err = None
    if error:
        err = np.tile([0.04, 0.92, 0.04], (B + 1, 1))
        err[0] = (0.0, 0.96, 0.04)
    for tree in (_odd_tree(), wl.yule_tree(30, 4)):
        counts = np.minimum(_counts(tree, F, B, 3 * B + F), B - 1)
        got = _lnl(eng, tree, counts, B, R, path, err)
        _same(path, got, _pieces(eng, tree, counts, B, R, path, err))
        plain = _lnl(eng, tree, counts, B, R, native.PATH_PLAIN64, err)
        _same(path, got, plain)
