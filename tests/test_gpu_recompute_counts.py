"""How many families the recompute of a reduced path redoes: the plan's own
counter, which leaves out what n_fallback adds to it (families near the
subnormal range, as all of these are).  Lists of up to 16 tiles of 16 families
run level by level where the partial vectors pass LDS -- here a balanced tree of
32 leaves, five partial vectors at least, 2 KB per 16 rows each -- and longer
ones on the matrix cores."""
import numpy as np
import pytest

from cafe5_amd import native, workloads as wl
from oracle_lib import Oracle

pytestmark = pytest.mark.gpu
LAM = 0.0005
LEVEL_TILES = 16


def _balanced(leaves):
    parent, leaf, level, n = [], list(range(leaves)), list(range(leaves)), leaves
    parent = [-1] * (2 * leaves - 1)
    while len(level) > 1:
        nxt = []
        for a, b in zip(level[::2], level[1::2]):
            parent[a] = parent[b] = n
            nxt.append(n)
            n += 1
        level = nxt
    leaf += [-1] * (leaves - 1)
    length = np.full(n, 8.0)
    length[n - 1] = 0.0
    return wl.Tree(np.array(parent, dtype=np.int32), np.array(leaf, dtype=np.int32), length, [f"n{i}" for i in range(n)])


@pytest.mark.parametrize("path", native.REDUCED_PATHS)
@pytest.mark.parametrize("B,F,few", [(256, 1, True), (256, 256, True), (400, 17, True), (256, 257, False),
                                     (300, 400, False)])
def test_every_family_is_redone(path, B, F, few):
    assert ((B + 1 + 15) // 16) * 5 * 2 > 150   # KB of partial vectors: past LDS
    assert ((F + 15) // 16 <= LEVEL_TILES) == few
    tree = _balanced(32)
    counts = np.random.default_rng(B + F).integers(0, B - 4, (F, 32)).astype(np.int32)
    keys = native.KeyTable()
    slots = keys.node_slots(tree, np.full((1, tree.n_nodes), LAM))
    prior = Oracle.prior_uniform(B, B)
    eng = native.Engine(0)
    eng.set_tree(tree)
    eng.set_families(counts, B, B)
    eng.matrix_reset(B + 1, len(keys.keys))
    out = []
    for p in (native.PATH_PLAIN64, path):
        plan = eng.plan(slots, prior, *keys.arrays(), path=p)
        plan.execute()
        out.append(plan.results()["lnl"].copy())
        if p == path:
            assert plan.recompute_counts()[0] == F
        plan.close()
    assert np.array_equal(out[0], out[1])
    eng.close()
