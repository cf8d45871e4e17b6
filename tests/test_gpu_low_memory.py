"""Evaluations on a device with little memory left: the columns of shared
subtrees are what an evaluation can do without, so a table that fits without
them is evaluated, with the same values."""
import numpy as np
import pytest

from bars import reduced_ok
from cafe5_amd import native, workloads as wl
from device_memory import MB, Filled, free_bytes
from oracle_lib import Oracle

pytestmark = pytest.mark.gpu
LEFT = 128 * MB


@pytest.mark.parametrize("path", [native.PATH_PLAIN64, native.PATH_BATCHED32])
def test_no_room_for_columns(path):
    tree = wl.yule_tree(14, 3)
    F, B, P = 6000, 100, 96
    rng = np.random.default_rng(1)
    counts = wl.simulate_families(tree, 1 + rng.integers(0, 20, F), np.full(tree.n_nodes, 0.004), 2, cap=B)
    lams = 0.002 + 0.00005 * np.arange(P)
    keys = native.KeyTable()
    slots = keys.node_slots(tree, np.repeat(lams[:, None], tree.n_nodes, axis=1))
    prior = Oracle.prior_uniform(B, B)

    def ready():
        e = native.Engine(0)
        e.set_tree(tree)
        e.set_families(counts, B, B)
        e.matrix_reset(B + 1, len(keys.keys))
        e.matrix_build(*keys.arrays())
        e.timings()   # (built)
        return e

    eng = ready()
    before = free_bytes()
    want = eng.evaluate(slots, prior, path)["lnl"].copy()
    assert before - free_bytes() > LEFT + 128 * MB   # most of it columns
    eng.close()
    eng = ready()
    rest = Filled(LEFT)
    try:
        got = eng.evaluate(slots, prior, path)["lnl"]
    finally:
        rest.release()
        eng.close()
    if path == native.PATH_PLAIN64:
        assert np.array_equal(got, want)
    else:
        assert np.all(reduced_ok(got, want))
