"""The launch for the bottom of the tree (mfd_tree_plan.cpp, mfd_tree.hip):
every wait satisfied by earlier tasks (CPU), and factors at the orders where
a front changes shape -- panels of 16 pivot columns, diagonal blocks of 64,
the largest order 128 -- with many children, a child of order above 128 in
the way, and each form of the values."""
import numpy as np
import pytest

import mfdag
from mfdag import problems as P
from parity import front_errors, oracle_for
from test_solve_tasks import arrow

# (pivot columns, update rows, leaves): orders 1 to 17, around 64 and 80,
# 112, and the last inside (128) and first outside (129)
SHAPES = [(1, 0, 1), (1, 1, 2), (15, 1, 3), (16, 1, 3), (17, 15, 9), (48, 15, 2), (16, 48, 5), (64, 1, 3), (63, 2, 2),
          (64, 15, 2), (65, 15, 2), (47, 65, 4), (100, 27, 2), (127, 1, 2), (64, 64, 3), (1, 127, 7), (128, 0, 1),
          (113, 16, 2), (80, 48, 3), (64, 65, 2)]


def open_arrow(c, w, leaves, **kw):
    p = arrow(c, w, leaves, seed=c + 200 * w)
    s = mfdag.Solver(nb=64, **kw)
    s.analyze(p.ccs_col, p.ccs_row, 0, np.arange(1, p.n + 1, dtype=np.int32))
    return s, p


@pytest.mark.parametrize("rule", [1, 0])
@pytest.mark.parametrize("make,max_zero", [
    (lambda: P.laplacian_2d(60), 16),
    (lambda: P.weighted_laplacian_3d(16, seed=2), 1024),
    (lambda: arrow(100, 28, 4, 1), 0),
    (lambda: arrow(100, 29, 4, 1), 0),
], ids=["lap2d_60", "wlap3d_16", "arrow_128", "arrow_129"])
def test_every_wait_is_for_earlier_tasks(make, max_zero, rule):
    p = make()
    s = mfdag.Solver(nb=64, host_only=True)
    s.analyze(p.ccs_col, p.ccs_row, max_zero, p.perm)
    s.level_rule = rule
    assert s.check_schedule(0) == (0, "")
    # some fronts of order 65 to 128 medium: they and their ancestors leave the launch
    s.set_front_kinds(np.random.default_rng(3).integers(0, 2, s.num_node).astype(np.int32))
    assert s.check_schedule(0) == (0, "")
    s.close()


@pytest.mark.gpu
@pytest.mark.parametrize("c,w,leaves", SHAPES, ids=lambda v: str(v))
def test_fronts_against_oracle(c, w, leaves):
    """FP64 1e-12 (the suite's bound).  FP32: the factor's relative error is
    at most about (order) * 2^-24 * the condition number, here below 4."""
    s, p = open_arrow(c, w, leaves)
    assert s.factorize(p.val) == 0
    f, st, info = oracle_for(s, p.val)
    assert info == 0
    assert front_errors(s, f, st).max() <= 1e-12
    _, b = P.rhs(p, 2, seed=4)
    assert P.backward_error(p, s.solve(b.copy()), b) <= 1e-14
    assert s.factorize(p.val, mfdag.FP32_IR) == 0
    assert front_errors(s, f, st).max() <= 4 * (c + w + 1) * 2.0 ** -24
    for prec in (mfdag.FP32_IR, mfdag.FP16_IR, mfdag.BF16_IR):
        assert s.factorize(p.val, prec) == 0
        assert P.backward_error(p, s.solve(b.copy()), b) <= 1e-14
    s.close()


@pytest.mark.gpu
@pytest.mark.parametrize("col", [0, 15, 16, 63, 64, 99, 100, 127])
def test_first_bad_pivot_is_reported(col):
    """A diagonal entry far below zero stops the factorization at its column
    in the panel or the front where it stands."""
    s, p = open_arrow(100, 28, 1)
    val = p.val.copy()
    val[p.ccs_col[col] - 1] = -1e6
    for prec in (mfdag.FP64, mfdag.FP32_IR):
        with pytest.raises(mfdag.NotPositiveDefinite) as e:
            s.factorize(val, prec)
        assert e.value.code == col + 1
        assert s.factorize(p.val, prec) == 0
    s.close()


def subsets(c, w, leaves, order, seed):
    """`leaves` dense blocks of order c, each coupled to w random columns of a
    dense block of the given order (> 128): children in the bottom-of-the-tree
    launch whose parent is not, their update rows scattered over its columns."""
    rng = np.random.Generator(np.random.PCG64(seed))
    n = c * leaves + order
    A = np.zeros((n, n))
    for k in range(leaves):
        s = slice(c * k, c * k + c)
        A[s, s] = rng.uniform(-1.0, 1.0, (c, c))
        A[np.ix_(c * leaves + rng.choice(order, w, replace=False), range(s.start, s.stop))] = rng.uniform(-1, 1, (w, c))
    A[c * leaves:, c * leaves:] = rng.uniform(-1.0, 1.0, (order, order))
    L = np.tril(A, -1)
    A = L + L.T
    np.fill_diagonal(A, np.abs(A).sum(axis=1) + 1.0)
    i, j = np.nonzero(np.tril(A))
    cc, rr, vv = P.lower_ccs(n, i, j, A[i, j])
    return P.Problem(n, cc, rr, vv, None, f"subsets_{c}_{w}_{leaves}_{order}")


@pytest.mark.gpu
@pytest.mark.parametrize("c,w,leaves,order", [(1, 1, 1, 129), (3, 31, 2, 144), (20, 32, 5, 160), (20, 33, 5, 161),
                                              (5, 64, 3, 191), (63, 65, 4, 192), (1, 127, 9, 193), (28, 100, 33, 260)],
                         ids=lambda v: str(v))
def test_children_added_into_a_larger_parent(c, w, leaves, order):
    p = subsets(c, w, leaves, order, seed=c + w)
    s = mfdag.Solver(nb=64)
    s.analyze(p.ccs_col, p.ccs_row, 0, np.arange(1, p.n + 1, dtype=np.int32))
    n = s.structure()["supernode_size"] + s.structure()["work_size"]
    assert n.max() > 128 and n.min() <= 128
    assert s.check_schedule(0) == (0, "")
    _, b = P.rhs(p, 2, seed=4)
    for prec in (mfdag.FP32_IR, mfdag.FP16_IR, mfdag.BF16_IR, mfdag.FP64):
        assert s.factorize(p.val, prec) == 0
        assert P.backward_error(p, s.solve(b.copy()), b) <= 1e-14
    f, st, info = oracle_for(s, p.val)
    assert info == 0
    assert front_errors(s, f, st).max() <= 1e-12
    s.close()
