"""The bound of the waits between running workgroups.  With a bound far below
the time that a chain of fronts takes, waits give up: every kernel ends, the
call returns MFD_ERR_INTERNAL, and the GPU serves the next handle."""
import numpy as np
import pytest

import mfdag
from mfdag import problems as P
from test_front_kinds import chain, natural

MFD_ERR_INTERNAL = -6


def tridiagonal(n):
    i = np.concatenate([np.arange(n), np.arange(1, n)])
    j = np.concatenate([np.arange(n), np.arange(n - 1)])
    cc, rr, vv = P.lower_ccs(n, i, j, np.where(i == j, 4.0, -1.0))
    return P.Problem(n, cc, rr, vv, None, f"tridiagonal_{n}")


@pytest.mark.gpu
def test_waits_that_give_up(monkeypatch):
    tri, blocks = tridiagonal(4000), chain(64, 50)
    monkeypatch.setenv("MFD_WAIT_POLLS", "1")
    # 4000 fronts of one column, one after another, in the bottom-of-the-tree launch
    s = mfdag.Solver(nb=64)
    s.analyze(tri.ccs_col, tri.ccs_row, 0, natural(tri))
    with pytest.raises(mfdag.MfdError) as e:
        s.factorize(tri.val)
    assert e.value.code == MFD_ERR_INTERNAL
    s.close()
    # 50 fronts, factored level by level, their solve one after another
    s = mfdag.Solver(nb=64)
    s.analyze(blocks.ccs_col, blocks.ccs_row, 0, natural(blocks))
    assert s.factorize(blocks.val) == 0
    _, b = P.rhs(blocks, 2, seed=1)
    with pytest.raises(mfdag.MfdError) as e:
        s.solve(b.copy())
    assert e.value.code == MFD_ERR_INTERNAL
    s.close()
    monkeypatch.delenv("MFD_WAIT_POLLS")
    for p in (tri, blocks):
        s = mfdag.Solver(nb=64)
        s.analyze(p.ccs_col, p.ccs_row, 0, natural(p))
        _, b = P.rhs(p, 2, seed=1)
        for prec in (mfdag.FP64, mfdag.FP32_IR):
            assert s.factorize(p.val, prec) == 0
            assert P.backward_error(p, s.solve(b.copy()), b) <= 1e-14
        s.close()
