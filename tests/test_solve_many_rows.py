"""Solves on levels with so many update rows that a forward task takes 64 of
them (more than 512 tasks of 16): fronts below and above one block, one
superblock and one 64-row tile, odd numbers of rows."""
import numpy as np
import pytest

import mfdag
from mfdag import problems as P
from test_front_kinds import natural
from test_solve_tasks import arrow

SHAPES = [(1, 129, 70), (20, 200, 50), (64, 191, 50), (65, 193, 50), (257, 400, 22)]


@pytest.mark.parametrize("block", [0, 256])
@pytest.mark.parametrize("c,w,leaves", SHAPES[:3])
def test_every_wait_is_for_earlier_tasks(c, w, leaves, block):
    p = arrow(c, w, leaves, seed=c + w)
    s = mfdag.Solver(nb=64, host_only=True)
    s.analyze(p.ccs_col, p.ccs_row, 0, natural(p))
    s.solve_block = block
    assert s.check_schedule(0) == (0, "")
    s.close()


@pytest.mark.gpu
@pytest.mark.parametrize("c,w,leaves", SHAPES)
def test_solutions(c, w, leaves):
    """Normwise backward error at most 1e-14, the bound every form is held to."""
    p = arrow(c, w, leaves, seed=c + w)
    s = mfdag.Solver(nb=64)
    s.analyze(p.ccs_col, p.ccs_row, 0, natural(p))
    assert int(s.structure()["work_size"].sum()) > 16 * 512
    for block in (0, 256):
        s.solve_block = block
        for prec in (mfdag.FP64, mfdag.FP32_IR):
            assert s.factorize(p.val, prec) == 0
            for nrhs in (1, 17):
                _, b = P.rhs(p, nrhs, seed=nrhs)
                assert P.backward_error(p, s.solve(b), b) <= 1e-14
    s.close()
