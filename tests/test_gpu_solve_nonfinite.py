"""NaN and infinity in a right-hand side: they spread through their own column of their own system and
no further, and the sweeps end (a reader of a block of x tells it from one not yet written by a NaN
of its own, which an input may hold too)."""
import numpy as np
import pytest
import scipy.sparse as sp

import gen
import rivrs_sparse as rs

pytestmark = pytest.mark.gpu

SENTINEL = float(np.array([0x7FF4A5A55A5A5A4A], dtype=np.uint64).view(np.float64)[0])
ORDERS = [300, 40, 129, 5, 257]  # fronts of several blocks of 128 columns, and single ones


@pytest.fixture(scope="module")
def factored():
    A = rs.SparseColMat.from_scipy(
        sp.block_diag([gen.deterministic_indefinite_matrix(m, 60 + m, 0.1) for m in ORDERS], format="csc"))
    s = rs.SparseLDLT.analyze(A, rs.AnalyzeOptions(rs.OrderingStrategy.Metis))
    s.factor(A)
    return s, A.n


@pytest.mark.parametrize("value", [np.nan, np.inf, -np.inf, SENTINEL], ids=["nan", "inf", "-inf", "sentinel"])
@pytest.mark.parametrize("nrhs", [1, 3, 9, 40])
def test_stays_in_its_column_and_system(factored, nrhs, value):
    s, n = factored
    rng = np.random.default_rng(nrhs)
    b = np.asfortranarray(rng.standard_normal((n, nrhs)))
    clean = s.solve(b)
    for block in range(len(ORDERS)):
        first = sum(ORDERS[:block])
        rows = np.arange(first, first + ORDERS[block])
        i, c = int(rng.choice(rows)), int(rng.integers(nrhs))
        print("non-finite %r nrhs=%d row %d column %d" % (value, nrhs, i, c), flush=True)
        bad = b.copy(order="F")
        bad[i, c] = value
        x = s.solve(bad)
        same = np.ones((n, nrhs), dtype=bool)
        same[rows, c] = False
        assert np.array_equal(x[same], clean[same])
        assert not np.isfinite(x[rows, c]).any()


def test_every_entry_is_the_sentinel(factored):
    s, n = factored
    assert np.isnan(s.solve(np.full((n, 5), SENTINEL, order="F"))).all()
