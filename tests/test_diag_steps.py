"""The 64-column steps of the large fronts (k_diag, k_upd_diag and its TRSM
tiles) at the block widths where a step changes shape: last blocks of one
column, around 16 and 64, one to eight blocks, and up to three pending panels
(update periods), against the oracle."""
import numpy as np
import pytest

import mfdag
from mfdag import problems as P
from parity import front_errors, oracle_for
from test_solve_tasks import arrow


@pytest.mark.gpu
@pytest.mark.parametrize("period", [1, 2, 3])
@pytest.mark.parametrize("c,w", [(65, 64), (127, 2), (128, 1), (129, 0), (143, 1), (144, 0), (145, 5), (191, 3), (192, 1),
                                 (193, 1), (208, 70), (257, 1), (320, 65), (449, 3)], ids=lambda v: str(v))
def test_steps_against_oracle(c, w, period):
    """FP64 1e-12 (the suite's bound).  FP32: at most about (order) * 2^-24 *
    the condition number, here below 4."""
    p = arrow(c, w, 1, seed=c + w)
    s = mfdag.Solver(nb=64)
    s.analyze(p.ccs_col, p.ccs_row, 0, np.arange(1, p.n + 1, dtype=np.int32))
    s.update_period = period
    assert s.factorize(p.val) == 0
    f, st, info = oracle_for(s, p.val)
    assert info == 0
    assert front_errors(s, f, st).max() <= 1e-12
    _, b = P.rhs(p, 2, seed=4)
    assert P.backward_error(p, s.solve(b.copy()), b) <= 1e-14
    assert s.factorize(p.val, mfdag.FP32_IR) == 0
    assert front_errors(s, f, st).max() <= 4 * (c + w + 1) * 2.0 ** -24
    s.close()


@pytest.mark.gpu
@pytest.mark.parametrize("col", [0, 15, 16, 63, 64, 127, 128, 143, 199])
def test_first_bad_pivot_is_reported(col):
    p = arrow(200, 0, 1, seed=3)
    s = mfdag.Solver(nb=64)
    s.analyze(p.ccs_col, p.ccs_row, 0, np.arange(1, p.n + 1, dtype=np.int32))
    val = p.val.copy()
    val[p.ccs_col[col] - 1] = -1e6
    for prec in (mfdag.FP64, mfdag.FP32_IR):
        with pytest.raises(mfdag.NotPositiveDefinite) as e:
            s.factorize(val, prec)
        assert e.value.code == col + 1
        assert s.factorize(p.val, prec) == 0
    s.close()
