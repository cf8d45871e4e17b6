"""Evaluations on a device with little memory left: the columns of shared
subtrees are what an evaluation can do without, so a table that fits without
them is evaluated, with the same values."""
import numpy as np
import pytest

from bars import reduced_ok
from cafe5_amd import native, workloads as wl
from oracle_lib import Oracle

pytestmark = pytest.mark.gpu
MB = 1 << 20
LEFT = 128 * MB


@pytest.mark.parametrize("path", [native.PATH_PLAIN64, native.PATH_BATCHED32])
def test_no_room_for_columns(path):
    import torch

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

    def free():
        torch.cuda.empty_cache()
        return torch.cuda.mem_get_info(0)[0]

    eng = ready()
    before = free()
    want = eng.evaluate(slots, prior, path)["lnl"].copy()
    assert before - free() > LEFT + 128 * MB   # most of it columns
    eng.close()
    eng = ready()
    hold = []   # everything but LEFT, in blocks
    for size in (64 << 30, 8 << 30, 1 << 30, 16 * MB):
        try:
            while True:
                hold.append(torch.empty(size, dtype=torch.uint8, device="cuda:0"))
        except torch.cuda.OutOfMemoryError:
            pass
    assert len(hold) > LEFT // (16 * MB)
    del hold[-(LEFT // (16 * MB)):]
    free()
    try:
        got = eng.evaluate(slots, prior, path)["lnl"]
    finally:
        hold.clear()
        free()
        eng.close()
    if path == native.PATH_PLAIN64:
        assert np.array_equal(got, want)
    else:
        assert np.all(reduced_ok(got, want))
