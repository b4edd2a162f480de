"""Failed columns whose swaps to the end of the outer block chain into cycles, with the persistent
launches and with the launches per inner block, against the oracle, bitwise.

The first block of 32 columns has `good` columns and then fails; `gap` columns follow it in the outer
block.  The 32 - good swaps by that distance form cycles of about (32 - good) / gap + 1 lines: 33
(longer than a round in registers), 32, 18, 17, 16 and 2, 3, ... of shorter ones."""
import os

import numpy as np
import pytest

import oracle
import rivrs_sparse as rs

pytestmark = pytest.mark.gpu


def _matrix(m, good, gap, seed):
    rng = np.random.default_rng(seed)
    a = rng.standard_normal((m, m))
    a = np.tril(a) + np.tril(a, -1).T
    a[:32, :32] = 0.0
    # a good column's multipliers stay below 1; the others' exceed the bound of 100
    a[np.arange(good), np.arange(good)] = 8.0 + np.arange(good)
    j = np.arange(good, 32)
    a[j, j] = 1e-4 * (1.0 + j)
    return a


@pytest.mark.parametrize("m", [70, 300, 900])
@pytest.mark.parametrize("good,gap", [(0, 1), (0, 2), (1, 1), (1, 2), (15, 1), (16, 1), (17, 1), (3, 5), (0, 31), (1, 32)])
def test_cycles_match_oracle(m, good, gap):
    p = 32 + gap
    a = _matrix(m, good, gap, 1000 * good + gap + m)
    M = rs.SparseColMat(m, np.arange(0, m * m + 1, m, dtype=np.int64), np.tile(np.arange(m, dtype=np.int64), m),
                        a.ravel(order="F"))
    st = rs.Structure(m, np.array([0, p], np.int32), np.array([p, m], np.int32), np.array([0, m - p, m - p], np.int64),
                      np.arange(p, m, dtype=np.int32), np.array([1, -1], np.int32), np.arange(m, dtype=np.int32))
    ref = oracle.OracleFactor(M, st, opts=oracle.options(nemin=1, small_leaf=0)).front(0)
    old = os.environ.get("RV_APTP_CHAIN")
    try:
        for chain in ("1", "0"):
            print("swap cycles m=%d good=%d gap=%d persistent=%s" % (m, good, gap, chain), flush=True)
            os.environ["RV_APTP_CHAIN"] = chain
            s = rs.SparseLDLT.from_structure(st)
            s.factor(M, rs.FactorOptions(nemin=1, small_leaf_threshold=0))
            assert (s.chain_launches() > 0) == (chain == "1")
            got = s.export_front(0)
            for key in ("dkind", "ddiag", "doff", "l11", "l21", "row_indices", "local_perm"):
                assert np.array_equal(got[key], ref[key]), (chain, key)
    finally:
        if old is None:
            os.environ.pop("RV_APTP_CHAIN", None)
        else:
            os.environ["RV_APTP_CHAIN"] = old
