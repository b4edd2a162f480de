"""Failed columns of a front of more than 1 GiB: the line swaps leave the 32-bit offsets of a buffer
resource and move entry by entry.

The matrix is diagonal but for 40 dense rows and columns whose own block is tiny, so the first block
of columns fails and is moved twice, to the end of its outer block and of the front.  Its inertia follows
from the 40 x 40 Schur complement; the two launch forms agree bitwise."""
import os

import numpy as np
import pytest
import scipy.sparse as sp

import rivrs_sparse as rs

pytestmark = pytest.mark.gpu

N, DENSE = 11600, 40


def test_swaps_beyond_one_gib():
    rng = np.random.default_rng(3)
    d = 1e-4 * (1.0 + np.arange(DENSE))
    c = np.where(rng.random(N - DENSE) < 0.3, -1.0, 1.0) * rng.uniform(4.0, 8.0, N - DENSE)
    B = rng.standard_normal((N - DENSE, DENSE))
    A = rs.SparseColMat.from_scipy(sp.bmat([[sp.diags(d), sp.csr_matrix(B.T)], [sp.csr_matrix(B), sp.diags(c)]], format="csc"))
    schur = np.linalg.eigvalsh(np.diag(d) - B.T @ (B / c[:, None]))
    negative = int((c < 0).sum() + (schur < 0).sum())
    st = rs.Structure(N, np.array([0], np.int32), np.array([N], np.int32), np.array([0, 0], np.int64),
                      np.zeros(0, np.int32), np.array([-1], np.int32), np.arange(N, dtype=np.int32))
    b = rng.standard_normal(N)
    xs = []
    old = os.environ.get("RV_APTP_CHAIN")
    try:
        for chain in ("1", "0"):
            print("large front persistent=%s" % chain, flush=True)
            os.environ["RV_APTP_CHAIN"] = chain
            s = rs.SparseLDLT.from_structure(st)
            s.factor(A)
            assert (s.chain_launches() > 0) == (chain == "1")
            inert = s.inertia()
            assert (inert.positive, inert.negative, inert.zero) == (N - negative, negative, 0)
            x = s.solve(b)
            assert rs.sparse_backward_error(A, x, b) <= 1e-14
            xs.append(x)
            del s
    finally:
        if old is None:
            os.environ.pop("RV_APTP_CHAIN", None)
        else:
            os.environ["RV_APTP_CHAIN"] = old
    assert np.array_equal(xs[0], xs[1])
