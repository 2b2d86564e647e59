"""Factors that are representable come out exactly: matrices L L^T with small
integer entries of L, whose every pivot, quotient and update is an integer, in
FP64 and FP32, through the launch for the bottom of the tree (order <= 128) and
the 64-column steps (whose 64 x 64 blocks are uncoupled here: the panel's rows
below a diagonal block are formed with its inverse, which is no integer).  So
an exactly singular matrix is refused at its zero pivot instead of passing with
a rounding error in its place."""
import numpy as np
import pytest

import mfdag
from mfdag import problems as P


def integer_factor(n, seed):
    """Lower triangular, integer, off-diagonal entries -15 .. 15, pivots 1 .. 63;
    L L^T and every partial sum of it stay below 2^24."""
    rng = np.random.Generator(np.random.PCG64(seed))
    L = np.tril(rng.integers(-15, 16, (n, n)).astype(np.float64), -1)
    np.fill_diagonal(L, rng.integers(1, 64, n))
    if n > 128:
        L *= np.arange(n)[:, None] // 64 == np.arange(n) // 64
    assert (np.abs(L) @ np.abs(L).T).max() < 2 ** 24
    return L


def open_dense(n):
    i, j = np.tril_indices(n)
    cc, rr, order = P.lower_ccs(n, i, j, np.arange(len(i)))
    order = order.astype(np.int64)
    s = mfdag.Solver(nb=64)
    s.analyze(cc, rr, 0, np.arange(1, n + 1, dtype=np.int32))
    assert s.num_node == 1
    return s, lambda A: np.ascontiguousarray(A[i[order], j[order]])


@pytest.mark.gpu
@pytest.mark.parametrize("n", [2, 16, 17, 48, 64, 65, 100, 128, 129, 200, 333])
def test_integer_factors_are_exact(n):
    s, values = open_dense(n)
    for seed in range(4):
        L = integer_factor(n, seed)
        for prec in (mfdag.FP64, mfdag.FP32_IR):
            assert s.factorize(values(L @ L.T), prec) == 0
            assert s.stats()["precision"] == prec
            assert np.array_equal(np.tril(s.front(1)), L), (n, seed, prec)
    s.close()


@pytest.mark.gpu
@pytest.mark.parametrize("n,col", [(2, 1), (40, 7), (64, 33), (100, 99), (128, 15), (129, 100), (200, 64), (200, 199)])
def test_zero_pivots_are_refused(n, col):
    """Pivot `col` (0-based) exactly zero: the reported column is its own."""
    s, values = open_dense(n)
    for seed in range(4):
        L = integer_factor(n, seed)
        L[col, col] = 0.0
        with pytest.raises(mfdag.NotPositiveDefinite) as e:
            s.factorize(values(L @ L.T))
        assert e.value.code == col + 1, seed
    s.close()


@pytest.mark.gpu
def test_singular_pairs_are_refused():
    """[[s^2, s l], [s l, l^2]] for all integers up to 64, in one matrix of
    2 x 2 blocks each time but for one singular block."""
    pairs = [(a, b) for a in range(1, 65) for b in range(1, 65)]
    n = 2 * len(pairs)
    diag = np.arange(n)
    rows, cols = np.concatenate([diag, diag[1::2]]), np.concatenate([diag, diag[::2]])
    cc, rr, order = P.lower_ccs(n, rows, cols, np.arange(len(rows)))
    order = order.astype(np.int64)
    a, b = (np.array(v, dtype=np.float64) for v in zip(*pairs))
    s = mfdag.Solver(nb=64)
    systems = [(np.array([1, 3, 4], dtype=np.int32), np.array([1, 2, 2], dtype=np.int32))] * len(pairs)
    s.analyze_batch(systems, 0, None)
    vals = np.stack([a * a, a * b, b * b + 1.0], axis=1)
    assert s.factorize(vals.ravel()) == 0
    for k in range(len(pairs)):
        v = vals.copy()
        v[k, 2] -= 1.0
        with pytest.raises(mfdag.NotPositiveDefinite) as e:
            s.factorize(v.ravel())
        assert e.value.code == 2 * k + 2, pairs[k]
    s.close()
