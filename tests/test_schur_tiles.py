"""The 64 x 64 tile product (tile_mma in mfd_kernels.hip) at the lengths of its
K loop where the chunks in flight change -- 16 columns a chunk, two chunks
ahead -- and with tiles past one square of the order in which a launch's tiles
are handed out, against the oracle."""
import numpy as np
import pytest

import mfdag
from mfdag import problems as P
from parity import front_errors, oracle_for
from test_solve_tasks import arrow


@pytest.mark.gpu
@pytest.mark.parametrize("c,w,leaves", [(1, 130, 2), (15, 129, 2), (16, 191, 2), (17, 192, 2), (32, 193, 3), (33, 130, 2),
                                        (48, 130, 2), (49, 130, 2), (64, 130, 3), (65, 130, 2), (81, 600, 3),
                                        (129, 130, 2), (257, 70, 2)], ids=lambda v: str(v))
def test_schur_update_against_oracle(c, w, leaves):
    p = arrow(c, w, leaves, seed=c + w)
    s = mfdag.Solver(nb=64)
    s.analyze(p.ccs_col, p.ccs_row, 0, np.arange(1, p.n + 1, dtype=np.int32))
    assert s.factorize(p.val) == 0
    f, st, info = oracle_for(s, p.val)
    assert info == 0
    assert front_errors(s, f, st).max() <= 1e-12
    _, b = P.rhs(p, 2, seed=4)
    for prec in (mfdag.FP64, mfdag.FP32_IR, mfdag.FP16_IR, mfdag.BF16_IR):
        assert s.factorize(p.val, prec) == 0
        assert P.backward_error(p, s.solve(b.copy()), b) <= 1e-14
    s.close()
