"""Matrices whose CCS gives an entry more than once: the fronts are assembled
from the last one of each in the order of the analysed structure, as the
reference stores them one after another (coefficient_setter_m.f90:26-41),
wherever the copies fall among the threads of a workgroup.  (FP32: the copies
differ by 30% and more.)"""
import numpy as np
import pytest

import mfdag
from mfdag import problems as P
from parity import front_errors, oracle_for


def repeated(p, seed):
    """p with up to two earlier copies of its entries below the diagonal, of
    other values."""
    rng = np.random.Generator(np.random.PCG64(seed))
    copies = rng.integers(0, 3, len(p.val))
    copies[p.ccs_col[:-1] - 1] = 0
    at = np.repeat(np.arange(len(p.val)), copies + 1)
    is_last = np.append(at[1:] != at[:-1], True)
    val = np.where(is_last, p.val[at], p.val[at] * rng.uniform(0.2, 0.7, len(at)))
    col = np.concatenate([[0], np.cumsum(copies + 1)])[p.ccs_col - 1] + 1
    return col.astype(np.int32), p.ccs_row[at].astype(np.int32), val


@pytest.mark.gpu
@pytest.mark.parametrize("name,make,max_zero", [
    ("lap2d_60", lambda: P.laplacian_2d(60), 16), ("wlap3d_14", lambda: P.weighted_laplacian_3d(14, seed=2), 1024),
    ("st27_8", lambda: P.stencil27_3d(8, seed=3), 64), ("blk3_6", lambda: P.block_stencil_3dof(6, seed=4), 256),
], ids=lambda v: v if isinstance(v, str) else "")
def test_last_copy_is_assembled(name, make, max_zero):
    p = make()
    col, row, val = repeated(p, seed=5)
    s = mfdag.Solver(nb=64)
    s.analyze(col, row, max_zero, p.perm)
    f, st, info = oracle_for(s, val)
    assert info == 0
    for prec, bound in ((mfdag.FP64, 1e-12), (mfdag.FP32_IR, 1e-4)):
        for _ in range(3):
            assert s.factorize(val, prec) == 0
            assert s.stats()["precision"] == prec
            assert front_errors(s, f, st).max() <= bound
        # the refinement is of the same matrix
        b = P.rhs(p, 2, seed=3)[1]
        x = s.solve(b.copy())
        if prec == mfdag.FP64:
            want = x
        assert s.stats()["precision"] == prec
        assert np.max(np.abs(x - want)) <= 1e-8 * np.max(np.abs(want))
    s.close()
