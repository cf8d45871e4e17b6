"""When the search for shared subtrees runs: not for setting families, root
vectors or reconstructions, which share nothing, and once for a table that is
set again unchanged (a model that sets tree and families for every score)."""
import time

import numpy as np
import pytest

from cafe5_amd import native, workloads as wl
from device_memory import free_bytes
from oracle_lib import Oracle

pytestmark = pytest.mark.gpu
LAM, F, B, R = 0.004, 200000, 40, 10


def _table():
    tree = wl.yule_tree(34, 3)
    rng = np.random.default_rng(1)
    counts = wl.simulate_families(tree, 1 + rng.integers(0, 6, F), np.full(tree.n_nodes, LAM), 2, cap=B)
    keys = native.KeyTable()
    return tree, counts, keys, keys.node_slots(tree, np.full((1, tree.n_nodes), LAM))


def test_nothing_is_searched_where_nothing_is_shared():
    tree, counts, keys, slots = _table()
    warm = native.Engine(0)   # (kernels loaded)
    warm.set_tree(tree)
    warm.set_families(counts[:100], B, R)
    warm.matrix_reset(B + 1, len(keys.keys))
    warm.matrix_build(*keys.arrays())
    prior = Oracle.prior_uniform(R, R)
    warm.root_vectors(slots, prior, native.PATH_PLAIN64)
    eng = native.Engine(0)
    eng.set_tree(tree)
    eng.matrix_reset(B + 1, len(keys.keys))
    eng.matrix_build(*keys.arrays())
    eng.timings()
    f0 = free_bytes()
    eng.set_families(counts, B, R)
    f1 = free_bytes()
    # the counts and their order; the search's tables hold the counts again
    # and a row per shared node
    assert f0 - f1 < 1.4 * counts.nbytes, f0 - f1
    eng.root_vectors(slots, prior, native.PATH_PLAIN64)
    # vectors, values and lists of every family: 8 R and about 60 bytes
    assert f1 - free_bytes() < F * (8 * R + 60) + counts.nbytes // 2, f1 - free_bytes()
    warm.close()
    eng.close()


def test_the_same_table_is_searched_once():
    tree, counts, keys, slots = _table()
    other = counts.copy()
    other[7, 5] ^= 1
    prior = Oracle.prior_uniform(R, R)
    eng = native.Engine(0)
    eng.matrix_reset(B + 1, len(keys.keys))
    eng.matrix_build(*keys.arrays())

    def score(c):
        t = time.perf_counter()
        eng.set_tree(tree)
        eng.set_families(c, B, R)
        r = eng.evaluate(slots, prior, native.PATH_BATCHED64)["lnl"][0]
        return time.perf_counter() - t, r

    _, a = score(counts)   # (buffers)
    changed = [score(other), score(counts), score(other), score(counts)]
    same = [score(counts), score(counts), score(counts), score(counts)]
    print("changed", [round(1e3 * t, 1) for t, _ in changed], "same", [round(1e3 * t, 1) for t, _ in same])
    assert np.array_equal(changed[0][1], changed[2][1])
    assert np.flatnonzero(changed[0][1] != a).tolist() == [7]
    for _, r in (changed[1], changed[3], *same):
        assert np.array_equal(r, a)
    assert min(t for t, _ in same) < 0.75 * min(t for t, _ in changed)
    eng.close()
