"""The solves' task list (mfd_solve_plan.cpp) and kernel (mfd_solve.hip): every
wait satisfied by earlier tasks (CPU), and solutions at the sizes where a
task changes shape -- blocks of 64 and superblocks of 256 pivot columns,
chunks of 16, 64 and 256 update rows, more than two children of one front,
groups of 16 right-hand sides."""
import numpy as np
import pytest

import mfdag
from mfdag import problems as P


def arrow(c, w, leaves, seed):
    """`leaves` dense diagonal blocks of order c, each coupled to one dense
    block of order w (w = 0: a single dense block): one front of c pivot
    columns and w update rows per block, and a root of w columns."""
    rng = np.random.Generator(np.random.PCG64(seed))
    n = c * leaves + w
    A = np.zeros((n, n))
    for k in range(leaves):
        s = slice(c * k, c * k + c)
        A[s, s] = rng.uniform(-1.0, 1.0, (c, c))
        A[c * leaves:, s] = rng.uniform(-1.0, 1.0, (w, c))
    A[c * leaves:, c * leaves:] = rng.uniform(-1.0, 1.0, (w, w))
    L = np.tril(A, -1)
    A = L + L.T
    np.fill_diagonal(A, np.abs(A).sum(axis=1) + 1.0)
    i, j = np.nonzero(np.tril(A))
    cc, rr, vv = P.lower_ccs(n, i, j, A[i, j])
    return P.Problem(n, cc, rr, vv, None, f"arrow_{c}_{w}_{leaves}")


@pytest.mark.parametrize("block", [0, 1, 65, 256])
@pytest.mark.parametrize("name,make,max_zero", [
    ("lap2d_60", lambda: P.laplacian_2d(60), 16),
    ("wlap3d_20", lambda: P.weighted_laplacian_3d(20, seed=2), 4096),
    ("blk3_9", lambda: P.block_stencil_3dof(9, seed=7), 256),
    ("arrow_300_270", lambda: arrow(300, 270, 3, 1), 0),
], ids=lambda v: v if isinstance(v, str) else "")
def test_every_wait_is_for_earlier_tasks(name, make, max_zero, block):
    p = make()
    s = mfdag.Solver(nb=64, host_only=True)
    s.analyze(p.ccs_col, p.ccs_row, max_zero, p.perm)
    for rule in (1, 0):
        s.level_rule = rule
        s.solve_block = block
        n, rep = s.check_schedule(0)
        assert n == 0, rep
    s.close()


def test_every_wait_is_for_earlier_tasks_in_a_batch():
    systems = P.batch_anisotropic(30, seed=4, lo=4, hi=60)
    s = mfdag.Solver(nb=64, host_only=True)
    s.analyze_batch([(p.ccs_col, p.ccs_row) for p in systems], 256, [p.perm for p in systems])
    n, rep = s.check_schedule(0)
    assert n == 0, rep
    s.close()


# (pivot columns, update rows, fronts below the root)
SHAPES = [(1, 0, 1), (63, 0, 1), (64, 0, 1), (65, 0, 1), (255, 0, 1), (257, 0, 1), (600, 0, 1), (1, 1, 5), (2, 17, 3),
          (64, 64, 3), (65, 65, 4), (130, 128, 2), (200, 129, 2), (256, 16, 2), (257, 256, 2), (300, 257, 3),
          (520, 300, 2)]


@pytest.mark.gpu
@pytest.mark.parametrize("precision", [mfdag.FP64, mfdag.FP32_IR], ids=["fp64", "fp32_ir"])
@pytest.mark.parametrize("c,w,leaves", SHAPES)
def test_solutions_at_task_edges(c, w, leaves, precision):
    """Normwise backward error at most 1e-14, the bound every form is held to,
    through the 64-column blocks, the explicit superblocks, and the default."""
    p = arrow(c, w, leaves, seed=c + w)
    s = mfdag.Solver(nb=64)
    s.analyze(p.ccs_col, p.ccs_row, 0, None)
    for block in (0, 1, 256):
        s.solve_block = block
        assert s.factorize(p.val, precision) == 0
        for nrhs in (1, 5, 16, 17, 33):
            print(f"c={c} w={w} leaves={leaves} block={block} nrhs={nrhs}", flush=True)
            _, b = P.rhs(p, nrhs, seed=nrhs)
            x = s.solve(b)
            eta = P.backward_error(p, x, b)
            assert eta <= 1e-14, (block, nrhs, eta)
    s.close()
