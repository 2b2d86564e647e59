"""Which fronts the launch for the bottom of the tree takes: by
mfd_set_front_kinds (0 gives the fronts of order 65 to 128 64-column steps, 1 a
workgroup each, -1 leaves them to the launch), and by their tree (all of order
<= 128 where it branches, none of the larger ones, or none at all, where fronts
follow one another in few chains)."""
import numpy as np
import pytest

import mfdag
from mfdag import problems as P, tune
from parity import front_errors, oracle_for
from test_solve_tasks import arrow


def front_flops(c, w):
    return float(sum(np.sum(np.arange(wi + 1.0, wi + ci + 1.0) ** 2) for ci, wi in zip(c, w)))


def launch_flops(st, order):
    """Flops of the class MFD_K_SMALL_FRONT with the launch taking the fronts
    of order <= `order` (and the other fronts of order <= 64, one by one)."""
    c, w, par = st["supernode_size"], st["work_size"], st["parent"]
    tree = tune.bottom_of_tree(c + w, par, order)
    inside = tree | (c + w <= 64)
    adds = tree & (par > 0) & tree[par - 1]  # into a parent of the same launch
    return front_flops(c[inside], w[inside]) + float(np.sum(w[adds] * (w[adds] + 1.0) / 2.0))


@pytest.mark.gpu
@pytest.mark.parametrize("kind", [0, 1, -1])
def test_kind_decides_the_route(kind):
    p = P.laplacian_2d(100)
    s = mfdag.Solver(nb=64)
    s.analyze(p.ccs_col, p.ccs_row, 256, p.perm)
    st = s.structure()
    c, w = st["supernode_size"], st["work_size"]
    n = c + w
    low = tune.bottom_of_tree(n, st["parent"])
    assert (low & (n > 64)).sum() >= 8
    s.set_front_kinds(np.full(s.num_node, kind, dtype=np.int32))
    assert s.factorize(p.val) == 0
    f, st, info = oracle_for(s, p.val)
    assert info == 0
    assert front_errors(s, f, st).max() <= 1e-12
    work = {k: v[0] for k, v in s.kernel_work().items()}
    assert work["small_front"] == pytest.approx(launch_flops(st, 128 if kind == -1 else 64), rel=1e-12)
    large = (n > 64) & (~low if kind == -1 else True)
    assert (work["potrf"] > 0) == (kind != 1 and large.any())
    assert (work["front"] > 0) == (kind == 1)
    s.close()


def chain(b, length):
    """A block tridiagonal matrix of dense b x b blocks: one front of b pivot
    columns and b update rows after another."""
    i = np.arange(b * length) // b
    A = np.where(np.abs(i[:, None] - i) <= 1, 0.5, 0.0)
    np.fill_diagonal(A, A.sum(axis=1) + 1.0)
    r, c = np.nonzero(np.tril(A))
    cc, rr, vv = P.lower_ccs(len(A), r, c, A[r, c])
    return P.Problem(len(A), cc, rr, vv, None, f"chain_{b}_{length}")


def natural(p):
    return np.arange(1, p.n + 1, dtype=np.int32)


def check_fronts(s, val):
    assert s.factorize(val) == 0
    f, st, info = oracle_for(s, val)
    assert info == 0
    assert front_errors(s, f, st).max() <= 1e-12
    return st, {k: v[0] for k, v in s.kernel_work().items()}


# the largest order of the launch's fronts (0: it takes none)
@pytest.mark.gpu
@pytest.mark.parametrize("name,make,order", [
    ("dense_30", lambda: arrow(30, 0, 1, 1), 0), ("dense_64", lambda: arrow(64, 0, 1, 1), 0),
    ("dense_128", lambda: arrow(128, 0, 1, 1), 0), ("chain_8", lambda: chain(8, 16), 128),
    ("chain_64", lambda: chain(64, 12), 0), ("grid_60", lambda: P.laplacian_2d(60), 128),
    ("star_100", lambda: arrow(100, 28, 40, 1), 128), ("star_60", lambda: arrow(60, 3, 100, 1), 128),
], ids=lambda v: v if isinstance(v, str) else "")
def test_chains_of_large_fronts_are_left_to_the_levels(name, make, order):
    p = make()
    s = mfdag.Solver(nb=64)
    s.analyze(p.ccs_col, p.ccs_row, 0, p.perm if p.perm is not None else natural(p))
    st, work = check_fronts(s, p.val)
    if order == 0:  # no extend-add inside the class
        n = st["supernode_size"] + st["work_size"]
        want = front_flops(st["supernode_size"][n <= 64], st["work_size"][n <= 64])
    else:
        want = launch_flops(st, order)
    assert work["small_front"] == pytest.approx(want, rel=1e-12)
    s.close()


# the shapes at which a front in the launch changes: 16-column panels, 64-column
# blocks of the inverse, the largest order, many children; beside a grid whose
# fronts keep the launch in use
@pytest.mark.gpu
@pytest.mark.parametrize("c,w,leaves", [(1, 1, 2), (15, 1, 3), (16, 1, 1), (17, 15, 9), (48, 15, 1), (16, 48, 5), (64, 1, 1),
                                        (63, 2, 2), (64, 15, 1), (65, 15, 2), (47, 65, 1), (100, 27, 2), (127, 1, 1),
                                        (64, 64, 3), (1, 127, 7), (128, 0, 1), (113, 15, 1), (80, 48, 1)],
                         ids=lambda v: str(v))
def test_front_shapes_in_the_launch(c, w, leaves):
    grid, p = P.laplacian_2d(70), arrow(c, w, leaves, seed=c + 200 * w)
    s = mfdag.Solver(nb=64)
    s.analyze_batch([(q.ccs_col, q.ccs_row) for q in (grid, p)], 0, [grid.perm, natural(p)])
    val = np.concatenate([grid.val, p.val])
    st, work = check_fronts(s, val)
    assert work["small_front"] == pytest.approx(launch_flops(st, 128), rel=1e-12)
    both = P.batch_problem([grid, p])
    _, b = P.rhs(both, 2, seed=3)
    for prec in (mfdag.FP64, mfdag.FP32_IR, mfdag.FP16_IR, mfdag.BF16_IR):
        assert s.factorize(val, prec) == 0
        assert P.backward_error(both, s.solve(b.copy()), b) <= 1e-14
    s.close()
