"""The solve sweeps at the edges of their groups and tiles.

A column's result does not depend on the columns beside it, bitwise, and it solves the system to
the rounding of the sweeps' sums.
"""
import numpy as np
import pytest

import gen
import rivrs_sparse as rs
import workloads

pytestmark = pytest.mark.gpu

SYSTEMS = {
    # fronts of up to 576 columns, rows not a multiple of 128, and many fused small fronts
    "helmholtz24": lambda: workloads.helmholtz(24, seed=5)[0],
    "helmholtz9": lambda: workloads.helmholtz(9, seed=6)[0],
    # 2x2 pivots and delayed columns
    "kkt20": lambda: workloads.kkt(20, seed=7)[0],
}


@pytest.mark.parametrize("name", sorted(SYSTEMS))
def test_columns_are_independent_of_their_group(name):
    A = SYSTEMS[name]()
    s = rs.SparseLDLT.analyze_with_matrix(A, rs.AnalyzeOptions(rs.OrderingStrategy.MatchOrderMetis))
    s.factor(A)
    B = np.asfortranarray(np.random.default_rng(11).standard_normal((A.n, 65)))
    X = s.solve(B)
    # groups of 4 (1 .. 32 columns, remainders) and of 8 (33 .. 65)
    for k in (1, 2, 3, 4, 5, 7, 8, 9, 16, 31, 32, 33, 40, 41, 64):
        print("%s columns %d" % (name, k), flush=True)
        assert np.array_equal(s.solve(np.asfortranarray(B[:, :k])), X[:, :k])
    one = np.stack([s.solve(np.ascontiguousarray(B[:, j])) for j in (0, 40, 64)], axis=1)
    assert np.array_equal(one, X[:, [0, 40, 64]])


# One dense front of m columns: blocks of 128 and their halves of 64, their 16-row tiles, and odd
# remainders.  The two sweeps are sums of at most m products, each rounded once per term, on
# factors whose product may exceed the matrix by a small growth: 8 m eps of ||A|| ||x|| + ||b||.
@pytest.mark.parametrize("m", [1, 2, 15, 16, 17, 63, 64, 65, 79, 127, 128, 129, 191, 193, 257, 320, 385])
def test_dense_front_residual(m):
    print("dense system m=%d" % m, flush=True)
    a = gen.deterministic_indefinite_matrix(m, 40 + m, 0.1)
    s = rs.SparseLDLT.analyze_with_matrix(_csc(a), rs.AnalyzeOptions(rs.OrderingStrategy.Metis))
    s.factor(_csc(a))
    b = np.random.default_rng(m).standard_normal((m, 3))
    x = s.solve(np.asfortranarray(b))
    norm = np.abs(a).sum(axis=1).max()
    bound = 8 * m * np.finfo(float).eps * (norm * np.abs(x).max(axis=0) + np.abs(b).max(axis=0))
    assert np.all(np.abs(a @ x - b).max(axis=0) <= bound)


def _csc(a):
    m = a.shape[0]
    col_ptr = np.arange(0, m * m + 1, m, dtype=np.int64)
    row_idx = np.tile(np.arange(m, dtype=np.int64), m)
    return rs.SparseColMat(m, col_ptr, row_idx, np.ascontiguousarray(a.T).ravel())
