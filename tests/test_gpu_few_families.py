"""BATCHED32 of few families runs one row tile per wave: vectors of one tile up
to one past the sixteen waves, tables around a tile of families, against
PLAIN64 within the reduced paths' bars."""
import numpy as np
import pytest

from bars import reduced_ok
from cafe5_amd import native, workloads as wl
from cafe5_amd.model import BaseModel
from oracle_lib import Oracle

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def eng():
    e = native.Engine(0)
    yield e
    e.close()


@pytest.mark.parametrize("F", [1, 16, 45])
@pytest.mark.parametrize("B,R", [(40, 47), (63, 60), (64, 64), (127, 100), (128, 127), (130, 150), (255, 255), (256, 256)])
def test_against_plain(eng, B, R, F):
    tree = wl.yule_tree(40, 2)
    rng = np.random.default_rng(B + F)
    counts = wl.simulate_families(tree, 1 + rng.integers(0, B // 4, F), np.full(tree.n_nodes, 0.003), B, cap=B)
    out = []
    for path in (native.PATH_PLAIN64, native.PATH_BATCHED32):
        m = BaseModel(eng, tree, counts, B, R, path=path)
        m.infer_family_likelihoods(lambda r: Oracle.prior_uniform(r, r), 0.003)
        out.append(m.results.copy())
    assert np.all(reduced_ok(out[1], out[0]))
