"""Levels of many threshold-pivoting fronts, where a front's size and the number of its kind choose
how many wavefronts take it and what is staged: every factor against the oracle, bitwise (the
kernels do the oracle's operations in the oracle's order)."""
import numpy as np
import pytest

import oracle
import rivrs_sparse as rs

pytestmark = pytest.mark.gpu


def _systems(shapes, seed):
    """Independent systems (k, r): two leaves of k columns coupled to a dense border of r rows; k = 0:
    a dense system of order r, k = -1: one with large couplings between its halves, whose blocks of 32
    columns have few acceptable pivots.  Small diagonals, so that most pivots are 2x2 or moved."""
    rng = np.random.default_rng(seed)
    rows, cols, vals, at = [], [], [], 0
    for k, r in shapes:
        n = 2 * max(k, 0) + r
        a = rng.standard_normal((n, n))
        a[np.arange(n), np.arange(n)] *= 0.1
        if k < 0:
            a[n - n // 2 + np.arange(n // 2), rng.permutation(n // 2)] += 1e4
        keep = np.tril(np.ones((n, n), dtype=bool))
        if k > 0:
            keep[k:2 * k, :k] = False
        i, j = np.nonzero(keep)
        rows.append(at + i)
        cols.append(at + j)
        vals.append(a[i, j])
        at += n
    return rs.SparseColMat.from_lower_triplets(at, np.concatenate(rows), np.concatenate(cols), np.concatenate(vals))


# One wavefront per front (more than 1024 of at most 64 rows), beside fronts of 65 rows and more; the
# number one below.  A border and one of its leaves are one front: more than 512 of 100 to 141 rows in
# parts, beside 96 to 99 and 142; fewer of them staged whole.
CASES = {
    "waves": [(0, r) for r in (1, 2, 3, 7, 8, 9, 16, 24, 31)] * 115 + [(16, 48), (16, 49), (8, 56), (31, 33)] * 4,
    "fewer": [(0, 1 + q % 31) for q in range(1024)],
    "parts": [(30, 66 + q % 47) for q in range(600)],
    "whole": [(30, 66 + q % 47) for q in range(400)],
    # columns that block pivoting leaves over, in some of more fronts than workgroups take them
    "left over": [(-1 if q % 3 else 0, 40 + q % 60) for q in range(600)],
}


@pytest.mark.parametrize("name", sorted(CASES))
def test_levels_match_oracle(name):
    A = _systems(CASES[name], 31)
    s = rs.SparseLDLT.analyze(A, rs.AnalyzeOptions(rs.OrderingStrategy.Metis))
    print("tpp level %s n=%d" % (name, A.n), flush=True)
    s.factor(A, rs.FactorOptions(update_precision="fp64_exact"))
    ref = oracle.OracleFactor(A, s.structure())
    inert = s.inertia()
    assert (inert.positive, inert.negative, inert.zero) == ref.inertia()
    for f in range(ref.num_supernodes()):
        want, got = ref.front(f), s.export_front(f)
        for key in ("l11", "l21", "dkind", "ddiag", "doff", "col_indices", "row_indices"):
            assert np.array_equal(got[key], want[key]), (f, key)
