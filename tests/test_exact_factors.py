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


def integer_factor(n, seed, coupled):
    """Lower triangular, integer, off-diagonal entries -15 .. 15, pivots 1 .. 63;
    L L^T and every partial sum of it stay below 2^24."""
    rng = np.random.Generator(np.random.PCG64(seed))
    L = np.tril(rng.integers(-15, 16, (n, n)).astype(np.float64), -1)
    np.fill_diagonal(L, rng.integers(1, 64, n))
    if not coupled:
        L *= np.arange(n)[:, None] // 64 == np.arange(n) // 64
    assert (np.abs(L) @ np.abs(L).T).max() < 2 ** 24
    return L


def open_dense(n, launch):
    """A dense matrix by itself (factored level by level), or beside a grid
    that keeps the launch for the bottom of the tree in use; the function that
    makes the values, and the number of unknowns before it."""
    i, j = np.tril_indices(n)
    cc, rr, order = P.lower_ccs(n, i, j, np.arange(len(i)))
    order = order.astype(np.int64)
    grid = P.laplacian_2d(40)
    s = mfdag.Solver(nb=64)
    natural = np.arange(1, n + 1, dtype=np.int32)
    if launch:
        s.analyze_batch([(grid.ccs_col, grid.ccs_row), (cc, rr)], 0, [grid.perm, natural])
        return s, lambda A: np.concatenate([grid.val, A[i[order], j[order]]]), grid.n
    s.analyze(cc, rr, 0, natural)
    assert s.num_node == 1
    return s, lambda A: np.ascontiguousarray(A[i[order], j[order]]), 0


@pytest.mark.gpu
@pytest.mark.parametrize("n,launch", [(2, 0), (16, 0), (17, 0), (48, 0), (64, 0), (65, 0), (129, 0), (200, 0), (333, 0),
                                      (2, 1), (16, 1), (17, 1), (48, 1), (64, 1), (65, 1), (100, 1), (128, 1)])
def test_integer_factors_are_exact(n, launch):
    s, values, _ = open_dense(n, launch)
    for seed in range(4):
        L = integer_factor(n, seed, coupled=launch or n <= 64)
        for prec in (mfdag.FP64, mfdag.FP32_IR):
            assert s.factorize(values(L @ L.T), prec) == 0
            assert s.stats()["precision"] == prec
            assert np.array_equal(np.tril(s.front(s.num_node)), L), (seed, prec)
    s.close()


@pytest.mark.gpu
@pytest.mark.parametrize("n,col,launch", [(2, 1, 0), (40, 7, 0), (64, 33, 0), (129, 100, 0), (200, 64, 0), (200, 199, 0),
                                          (2, 1, 1), (40, 7, 1), (64, 33, 1), (100, 99, 1), (128, 15, 1)])
def test_zero_pivots_are_refused(n, col, launch):
    """Pivot `col` (0-based) exactly zero: the reported column is its own."""
    s, values, before = open_dense(n, launch)
    for seed in range(4):
        L = integer_factor(n, seed, coupled=launch or n <= 64)
        L[col, col] = 0.0
        with pytest.raises(mfdag.NotPositiveDefinite) as e:
            s.factorize(values(L @ L.T))
        assert e.value.code == before + col + 1, seed
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
