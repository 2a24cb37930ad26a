"""Pivots of the chunked FP64 cyclic reduction (gf_btdsystem): blocks whose diagonal
pivots, taken as they come, have multipliers of 3, 8 and 15 at every one of them and
entries that grow by as much; the same with columns scaled over twelve decades; and
random blocks without a dominant diagonal.  One block row (the last block's sweep) and
chunks of them (the eliminated rows' sweeps) with weak couplings.

The bar: elimination with interchanges that keep its entries' growth small has a
backward error of a few m ulp of the block, and each of the log2 n levels adds one
more, so the solution is within 8 m (1 + log2 n) condition numbers' ulp of the exact
one.  The condition is that of the system before its columns are scaled, and the error
is taken in that system's unknowns: a column's scale changes neither multipliers
nor interchanges.  (Grown entries lose (1 + multiplier)^(m - 1) ulp.)"""
import numpy as np
import pytest

from giraffe_amd import runtime

pytestmark = pytest.mark.gpu

EPS = np.finfo(float).eps


def _block(kind, m, mu, rng):
    B = np.eye(m)
    if kind == "triangle":  # -mu below the diagonal, ones in the last column
        B -= mu * np.tril(rng.uniform(0.9, 1.0, (m, m)), -1)
        B[:, -1] = 1.0
    elif kind == "subdiagonal":
        B[np.arange(1, m), np.arange(m - 1)] = mu * rng.choice([-1.0, 1.0], m - 1)
        B[1:, -1] += rng.uniform(0.5, 1.0, m - 1)
    else:  # "random", mu: the diagonal's share
        B = rng.normal(size=(m, m)) + mu * np.sqrt(m) * B
    return B


@pytest.mark.parametrize("scaled", [False, True])
@pytest.mark.parametrize("kind,mu", [("triangle", 3), ("triangle", 8), ("triangle", 15), ("subdiagonal", 3),
                                     ("subdiagonal", 8), ("subdiagonal", 15), ("random", 0.0), ("random", 0.5),
                                     ("random", 1.0)])
@pytest.mark.parametrize("m,n", [(6, 1), (12, 1), (16, 1), (24, 1), (32, 1), (12, 11), (16, 20), (24, 9), (32, 10)])
def test_growth_is_bounded(m, n, kind, mu, scaled):
    rng = np.random.default_rng(1000 * m + 10 * n + int(mu))
    B = np.array([_block(kind, m, mu, rng) for _ in range(n)])
    A, C = (1e-3 / m * rng.uniform(-1, 1, (n, m, m)) for _ in range(2))
    A[0] = C[-1] = 0.0
    K = np.zeros((n * m, n * m))
    for i in range(n):
        K[i * m:(i + 1) * m, i * m:(i + 1) * m] = B[i]
        if i:
            K[i * m:(i + 1) * m, (i - 1) * m:i * m] = A[i]
            K[(i - 1) * m:i * m, i * m:(i + 1) * m] = C[i - 1]
    y = rng.uniform(0.5, 1.0, n * m) * rng.choice([-1.0, 1.0], n * m)
    b = (K.astype(np.longdouble) @ y.astype(np.longdouble)).astype(float)
    s = 2.0 ** rng.integers(-20, 21, (n, m)) if scaled else np.ones((n, m))  # (exact)
    x, fail = runtime.btdsystem(A * np.roll(s, 1, 0)[:, None, :], B * s[:, None, :], C * np.roll(s, -1, 0)[:, None, :], b)
    assert fail == 0
    bar = 8 * m * (1 + np.log2(n)) * np.linalg.cond(K) * EPS
    assert np.linalg.norm(x * s.ravel() - y) <= bar * np.linalg.norm(y)
