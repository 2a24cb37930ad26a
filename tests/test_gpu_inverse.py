"""The 64 x 64 block inverse of the band solver where a pivot cannot serve.

Rows k - 1 and k hold [[1, 1], [1, 1]] and are coupled to nothing else: pivot k is
exactly zero, is replaced by 1e-13 of its original diagonal entry, and the solve
goes on.  The pair's inverse has entries of 1e13 / 1, so its product with b has an
error of up to 4 eps 1e13 max|b| and is held to that; every other row is its own
equation, a reciprocal and a product (1e-15 of it)."""
import numpy as np
import pytest

from giraffe_amd import runtime

pytestmark = pytest.mark.gpu


# first and last rows of a 16 x 16 leaf, of a 64 x 64 block, and of a later block
@pytest.mark.parametrize("k", [1, 15, 17, 31, 63, 65, 128])
def test_vanishing_pivot_is_replaced(k):
    n = 130
    rows = np.zeros((n, 3))
    rows[:, 1] = np.linspace(1.0, 3.0, n)
    rows[k - 1] = [0.0, 1.0, 1.0]
    rows[k] = [1.0, 1.0, 0.0]
    b = np.linspace(-1.0, 2.0, n)
    b[k - 1] = b[k] = 1.0
    x, fail = runtime.bandsystem(rows, 1, b)
    assert fail == 0
    pair = np.isin(np.arange(n), (k - 1, k))
    want = b / rows[:, 1]
    assert np.abs(x - want)[~pair].max() <= 2e-15
    assert np.abs(x - np.where(np.arange(n) == k, 0.0, 1.0))[pair].max() <= 4 * 2.3e-16 * 1e13


@pytest.mark.parametrize("k", [0, 16, 100])
def test_pivot_that_is_not_finite_fails(k):
    n = 130
    rows = np.zeros((n, 3))
    rows[:, 1] = 2.0
    rows[k, 1] = np.inf
    _, fail = runtime.bandsystem(rows, 1, np.ones(n))
    assert fail == 1
