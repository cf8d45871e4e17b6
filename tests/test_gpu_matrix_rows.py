"""Matrices as the host gets them, turned on the host (small) and on the device, at
sizes around its 32 x 32 tiles and the 256 rows of the closed form's blocks: every entry of both builds
against the oracle's term-by-term matrix (FP64 sums of non-negative terms: both
within 2e-12 of it, relative), the saturated and the zero key included."""
import numpy as np
import pytest

from cafe5_amd import native
from oracle_lib import Oracle

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def eng():
    e = native.Engine(0)
    yield e
    e.close()


@pytest.mark.parametrize("algo", [native.BUILD_CLOSED_FORM, native.BUILD_RECURRENCE])
@pytest.mark.parametrize("N", [2, 33, 64, 200, 256, 257, 288, 289])
def test_entries(eng, algo, N):
    lam, t = [0.002, 0.01, 0.0, 0.5], [30.0, 7.0, 10.0, 9.0]
    eng.matrix_reset(N, 4)
    eng.matrix_build(lam, t, algo=algo)
    for k in range(4):
        want = Oracle.matrix(lam[k], t[k], N)
        got = eng.matrix_get(k)
        assert got.shape == (N, N)
        assert np.all(np.abs(got - want) <= 2e-12 * np.abs(want) + 1e-290), (k, np.abs(got - want).max())
