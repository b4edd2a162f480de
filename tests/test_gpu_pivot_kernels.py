"""Pivot kernels at the sizes where their layouts change, against the oracle, bitwise.

The kernels do the oracle's operations in the oracle's order, so every compared value is equal to
the last bit and no tolerance enters.
"""
import numpy as np
import pytest

import gen
import oracle
import rivrs_sparse as rs

pytestmark = pytest.mark.gpu


def _same(a, p):
    ref = oracle.dense_factor(a, p)
    got = rs.dense_aptp_factor(a, p)
    for key in ("num_eliminated", "num_1x1", "num_2x2", "num_delayed"):
        assert got[key] == ref[key], (key, got[key], ref[key])
    ne = ref["num_eliminated"]
    assert np.array_equal(got["perm"], ref["perm"])
    for key in ("dkind", "ddiag", "doff"):
        assert np.array_equal(got[key][:ne], ref[key][:ne]), key
    lower = np.tril(np.ones(a.shape, dtype=bool))
    lower[:, p:] = False
    assert np.array_equal(got["a"][lower], ref["a"][lower])
    return ref


# Threshold partial pivoting (fewer than 32 columns): one and several wavefronts' rows, their
# remainders, the last front staged in LDS (31 columns, 651 rows) and the first worked on in place.
@pytest.mark.parametrize("m,p", [(1, 1), (3, 2), (31, 31), (63, 31), (64, 16), (65, 31), (256, 30), (257, 31),
                                 (300, 1), (651, 31), (652, 31), (653, 31), (900, 31)])
@pytest.mark.parametrize("kind", ["indefinite", "delays", "saddle", "ties"])
def test_threshold_pivots_match_oracle(m, p, kind):
    print("tpp m=%d p=%d %s" % (m, p, kind), flush=True)
    _same(_matrix(m, 100 + m + p, kind), p)


# Pivots within a block (32 columns, a last block of 1 .. 32): ties are decided by position, a
# saddle's zero diagonal takes 2x2 pivots only, and entries of 2^400 leave the keys' common range.
@pytest.mark.parametrize("m", [33, 34, 47, 63, 64, 65, 95, 129])
@pytest.mark.parametrize("kind", ["indefinite", "saddle", "ties", "huge", "tiny"])
def test_block_pivots_match_oracle(m, kind):
    print("block pivots m=%d %s" % (m, kind), flush=True)
    _same(_matrix(m, 200 + m, kind), m)


# Failed columns are swapped out of their block: rows beyond one workgroup's, a last block of one
# column, swaps that chain into long cycles; what is left goes to threshold pivoting, in LDS or,
# for wide remainders, in place.
@pytest.mark.parametrize("m,p", [(96, 64), (129, 97), (257, 256), (288, 257), (513, 160), (520, 513)])
@pytest.mark.parametrize("kind", ["delays", "saddle", "ties"])
def test_swapped_columns_match_oracle(m, p, kind):
    print("swaps m=%d p=%d %s" % (m, p, kind), flush=True)
    _same(_matrix(m, 300 + m + p, kind), p)


# A root whose columns mostly fail: threshold pivoting takes them in memory until the rest fits in
# LDS (140 square), then there; a remainder that fits from the start, one just above, wide ones.
@pytest.mark.parametrize("m", [150, 180, 300, 420])
@pytest.mark.parametrize("kind", ["delays", "pairs"])
def test_left_over_columns_match_oracle(m, kind):
    print("left-over columns m=%d %s" % (m, kind), flush=True)
    ref = _same(_matrix(m, 400 + m, kind), m)
    assert ref["num_eliminated"] == m


def _matrix(m, seed, kind):
    rng = np.random.default_rng(seed)
    if kind == "ties":
        a = rng.integers(-2, 3, size=(m, m)).astype(np.float64)
        return np.tril(a) + np.tril(a, -1).T
    a = gen.deterministic_indefinite_matrix(m, seed, 0.1)
    if kind == "delays":
        return gen.cause_delays(a, seed, 1000.0)
    if kind == "pairs":  # large couplings between the halves: no block of 32 has an acceptable pivot
        d = rng.permutation(m // 2)
        a[m - m // 2 + np.arange(m // 2), d] += 1e4
        a[d, m - m // 2 + np.arange(m // 2)] += 1e4
        return a
    if kind == "saddle":
        a[np.arange(m), np.arange(m)] = np.where(rng.random(m) < 0.5, 0.0, np.diag(a))
        return a
    return a * {"indefinite": 1.0, "huge": 2.0 ** 400, "tiny": 2.0 ** -40}[kind]
