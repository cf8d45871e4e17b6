"""A closed context gives its device memory back, the reconstruction's rows
among it."""
import numpy as np
import pytest

from cafe5_amd import native, workloads as wl
from device_memory import free_bytes
from oracle_lib import Oracle

pytestmark = pytest.mark.gpu


def test_closed_after_a_reconstruction():
    tree = wl.yule_tree(34, 3)
    F, B = 4000, 200
    counts = wl.simulate_families(tree, 1 + np.arange(F) % 9, np.full(tree.n_nodes, 0.003), 2, cap=B)
    keys = native.KeyTable()
    slots = keys.node_slots(tree, np.full((1, tree.n_nodes), 0.003))
    prior = np.append(0.0, Oracle.prior_uniform(B, B))
    free = []
    for _ in range(3):   # (the first one loads the kernels)
        eng = native.Engine(0)
        eng.set_tree(tree)
        eng.set_families(counts, B, B)
        eng.matrix_reset(B + 1, len(keys.keys))
        eng.matrix_build(*keys.arrays())
        eng.reconstruct(slots, prior, B, B)
        eng.close()
        free.append(free_bytes())
    assert free[0] - free[2] < 32 << 20, free   # a context's rows: 200 MB
