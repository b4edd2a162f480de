"""Inner and outer block sizes other than 32 and 256 and thresholds other than 0.01, and left-over
columns on either side of what fits in LDS: dense factors against the oracle, bitwise."""
import numpy as np
import pytest

import gen
import oracle
import rivrs_sparse as rs

pytestmark = pytest.mark.gpu


def _pairs(m, seed):
    """Large couplings of columns m / 2 apart: no block of 32 columns has an acceptable pivot."""
    a = gen.deterministic_indefinite_matrix_fast(m, seed, 0.1)
    i, j = m - m // 2 + np.arange(m // 2), np.arange(m // 2)
    a[i, j] += 1e6
    a[j, i] += 1e6
    return a


def _same(a, p, ib=32, nb=256, u=0.01):
    ref = oracle.dense_factor(a, p, oracle.options(threshold=u, nb=nb, ib=ib))
    got = rs.dense_aptp_factor(a, p, rs.FactorOptions(threshold=u, outer_block_size=nb, inner_block_size=ib))
    ne = ref["num_eliminated"]
    assert got["num_eliminated"] == ne
    assert np.array_equal(got["perm"], ref["perm"])
    for key in ("dkind", "ddiag", "doff"):
        assert np.array_equal(got[key][:ne], ref[key][:ne]), key
    lower = np.tril(np.ones(a.shape, dtype=bool))
    lower[:, p:] = False
    assert np.array_equal(got["a"][lower], ref["a"][lower])


@pytest.mark.parametrize("ib,nb", [(1, 32), (3, 100), (8, 64), (16, 256), (31, 64), (32, 32), (32, 100)])
@pytest.mark.parametrize("u", [0.01, 0.5])
def test_block_sizes_match_oracle(ib, nb, u):
    for m, p in ((150, 101), (400, 300)):
        print("blocks %d of %d, threshold %g, m=%d p=%d" % (ib, nb, u, m, p), flush=True)
        a = gen.deterministic_indefinite_matrix_fast(m, 700 + ib + m, 0.1)
        _same(a, p, ib, nb, u)
        _same(gen.cause_delays(a, ib, 1000.0), p, ib, nb, u)


# 141 columns are the last staged whole; past 1024 left-over columns the earlier columns' rows (there are
# 70) are permuted cycle by cycle
@pytest.mark.parametrize("m,good", [(140, 0), (141, 0), (142, 0), (143, 0), (200, 59), (201, 59), (1200, 70)])
def test_left_over_columns_at_the_lds_switch(m, good):
    print("left-over columns m=%d after %d" % (m, good), flush=True)
    a = gen.deterministic_indefinite_matrix_fast(m, 800 + m, 0.1)
    a[good:, good:] = _pairs(m - good, 900 + m)
    a[np.arange(good), np.arange(good)] = 40.0 + np.arange(good)
    assert oracle.dense_factor(a, m, oracle.options(tpp=False))["num_eliminated"] == good
    _same(a, m)
