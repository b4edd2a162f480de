"""Pivots within a block at the ends of the exponent range, against the oracle, bitwise.

The search for the largest entry works on 32-bit keys for blocks whose entries are all below 2^1000 and
winners above the pivot floor (1e-20); everything else takes the exact rule.  The diagonals dominate
where products of two entries would overflow, so every value stays finite."""
import numpy as np
import pytest

import gen
import oracle
import rivrs_sparse as rs

pytestmark = pytest.mark.gpu


def _diagonal(m, seed, lo, hi, off):
    """Distinct diagonal entries of random sign in 2^[lo, hi), the rest up to 2^off."""
    rng = np.random.default_rng(seed)
    a = rng.uniform(-1.0, 1.0, (m, m)) * 2.0 ** off
    a = np.tril(a) + np.tril(a, -1).T
    a[np.arange(m), np.arange(m)] = np.where(rng.random(m) < 0.5, -1.0, 1.0) * 2.0 ** rng.uniform(lo, hi, m)
    return a


def _matrix(m, kind):
    seed = 500 + m
    if kind == "above":  # every block takes the exact rule
        return _diagonal(m, seed, 1000.5, 1010.0, 980.0)
    if kind == "below":  # keys, up to the largest they are used for
        return _diagonal(m, seed, 990.0, 999.99, 970.0)
    if kind == "one above":  # one entry decides for its block alone
        a = _diagonal(m, seed, 990.0, 999.99, 970.0)
        a[m // 2, m // 2] = 2.0 ** 1003
        return a
    if kind == "growth":  # off-diagonal entries as large as the diagonal's: updates grow the block
        a = _diagonal(m, seed, 499.0, 500.0, 499.9)
        return a
    # winners that cross the floor during the block, and blocks wholly below it
    a = gen.deterministic_indefinite_matrix(m, seed, 0.5)
    return a * {"floor": 2e-20, "under": 0.9e-20, "over": 1e-17}[kind]


@pytest.mark.parametrize("m", [33, 64, 65, 95, 300])
@pytest.mark.parametrize("kind", ["above", "below", "one above", "growth", "floor", "under", "over"])
def test_block_pivots_match_oracle(m, kind):
    print("pivot range m=%d %s" % (m, kind), flush=True)
    a = _matrix(m, kind)
    ref = oracle.dense_factor(a, m)
    got = rs.dense_aptp_factor(a, m)
    for key in ("num_eliminated", "num_1x1", "num_2x2", "num_delayed"):
        assert got[key] == ref[key], key
    ne = ref["num_eliminated"]
    assert np.array_equal(got["perm"], ref["perm"])
    for key in ("dkind", "ddiag", "doff"):
        assert np.array_equal(got[key][:ne], ref[key][:ne]), key
    lower = np.tril(np.ones((m, m), dtype=bool))
    assert np.all(np.isfinite(ref["a"][lower]))
    assert np.array_equal(got["a"][lower], ref["a"][lower])
