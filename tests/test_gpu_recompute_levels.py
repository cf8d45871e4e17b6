"""The recompute of a few families of long vectors, level by level: families
whose likelihoods no reduced path can hold are all redone in FP64, so their
values equal PLAIN64's bit for bit -- few of them (level by level) and more than
that takes (matrix cores), vectors at the edges of its column groups and row
chunks, with an error model and as gamma categories."""
import numpy as np
import pytest

from cafe5_amd import native, workloads as wl
from cafe5_amd.model import BaseModel, GammaModel
from oracle_lib import Oracle

pytestmark = pytest.mark.gpu
LAM = 0.0005


@pytest.fixture(scope="module")
def eng():
    e = native.Engine(0)
    yield e
    e.close()


def _prior(r):
    return Oracle.prior_uniform(r, r)


@pytest.mark.parametrize("path", native.REDUCED_PATHS)
@pytest.mark.parametrize("B,R,F,error", [(256, 250, 1, False), (288, 288, 17, False), (319, 330, 40, True),
                                         (511, 512, 5, False), (512, 500, 3, True), (700, 700, 9, False),
                                         (300, 300, 400, False)])
def test_equal_to_plain(eng, path, B, R, F, error):
    tree = wl.yule_tree(24, 3)
    rng = np.random.default_rng(B + F)
    counts = rng.integers(0, B - 4, (F, tree.n_leaves)).astype(np.int32)
    err = None
    if error:
        err = np.tile([0.05, 0.9, 0.05], (B + 1, 1))
        err[0] = (0.0, 0.95, 0.05)
    plain = BaseModel(eng, tree, counts, B, R, path=native.PATH_PLAIN64, error_model=err)
    plain.infer_family_likelihoods(_prior, LAM)
    want = plain.results.copy()
    m = BaseModel(eng, tree, counts, B, R, path=path, error_model=err)
    m.infer_family_likelihoods(_prior, LAM)
    assert m.last["n_fallback"] >= F   # every family was redone
    assert np.array_equal(m.results, want), (m.results[:3], want[:3])


def test_categories(eng):
    tree = wl.yule_tree(24, 3)
    counts = np.random.default_rng(3).integers(0, 296, (6, tree.n_leaves)).astype(np.int32)
    args = (300, 300, np.full(2, 0.5), np.array([0.5, 1.5]))
    out = []
    for path in (native.PATH_PLAIN64, native.PATH_BATCHED32):
        m = GammaModel(eng, tree, counts, *args, path=path)
        m.infer_family_likelihoods(_prior, LAM)
        out.append(m.results["cat"].copy())
    assert np.array_equal(out[0], out[1], equal_nan=True)
