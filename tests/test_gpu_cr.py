"""The chunked FP64 cyclic reduction (gf_btdsystem) at the sizes where its chunks,
levels and launches change, against numpy block elimination from the first row
to the last.

Diagonal blocks are 4 m I plus entries in [-1, 1] (condition below 3, rows
permuted in the second half of the cases so that the sweeps take interchanges),
so the error is rounding alone: at most 32 rows a block, 13 levels, a few ulp a
step and a growth of 2 at each interchange stay below 1e-12."""
import numpy as np
import pytest

from giraffe_amd import runtime

pytestmark = pytest.mark.gpu


def _reference(A, B, C, b):
    n, m = B.shape[:2]
    b = b.reshape(n, m)
    Y, z = np.zeros((n, m, m)), np.zeros((n, m))
    for i in range(n):
        D = B[i] - A[i] @ Y[i - 1] if i else B[i]
        f = b[i] - A[i] @ z[i - 1] if i else b[i]
        s = np.linalg.solve(D, np.concatenate([C[i], f[:, None]], 1))
        Y[i], z[i] = s[:, :m], s[:, m]
    x = z.copy()
    for i in range(n - 2, -1, -1):
        x[i] -= Y[i] @ x[i + 1]
    return x.reshape(-1)


# one workgroup (1 .. 16 rows, or 8 of more than 16), chunks of 8, chunks of 32
# from 4,096 rows on; remainders of one row and of a chunk less one
@pytest.mark.parametrize("m,n", [(1, 1), (16, 1), (16, 2), (15, 3), (16, 8), (12, 9), (16, 16), (16, 17), (5, 33),
                                 (16, 64), (16, 65), (3, 1025), (12, 4095), (12, 4096), (6, 4097), (17, 1), (17, 8),
                                 (32, 9), (31, 16), (24, 65), (32, 513)])
@pytest.mark.parametrize("permuted", [False, True])
def test_chunk_edges(m, n, permuted):
    rng = np.random.default_rng(100 * m + n)
    A, C = rng.uniform(-1, 1, (n, m, m)), rng.uniform(-1, 1, (n, m, m))
    B = rng.uniform(-1, 1, (n, m, m)) + 4.0 * m * np.eye(m)
    if permuted:
        for i in range(0, n, 2):
            B[i] = B[i][rng.permutation(m)]
    b = rng.uniform(-1, 1, n * m)
    x, fail = runtime.btdsystem(A, B, C, b)
    ref = _reference(A, B, C, b)
    assert fail == 0
    assert np.abs(x - ref).max() <= 1e-12 * np.abs(ref).max()


@pytest.mark.parametrize("m,n,row", [(16, 40, 0), (16, 40, 39), (12, 1, 0), (20, 30, 17)])
def test_bad_pivot_is_reported(m, n, row):
    """A decoupled diagonal block that is zero, or holds a NaN, in each kind of row."""
    rng = np.random.default_rng(m + n + row)
    Z = np.zeros((n, m, m))
    for value in (0.0, np.nan):
        B = rng.uniform(-1, 1, (n, m, m)) + 4.0 * m * np.eye(m)
        B[row] = value
        _, fail = runtime.btdsystem(Z, B, Z, rng.uniform(-1, 1, n * m))
        assert fail == 1
