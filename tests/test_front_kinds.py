"""What mfd_set_front_kinds chooses for the fronts of order 65 to 128 at the
bottom of the tree: 0 gives them 64-column steps, 1 a workgroup each, -1 leaves
them to the launch that factors the bottom of the tree."""
import numpy as np
import pytest

import mfdag
from mfdag import problems as P, tune
from parity import front_errors, oracle_for


def front_flops(c, w):
    return float(sum(np.sum(np.arange(wi + 1.0, wi + ci + 1.0) ** 2) for ci, wi in zip(c, w)))


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
    tree = low if kind == -1 else tune.bottom_of_tree(n, st["parent"], 64)
    inside = tree | (n <= 64)
    adds = tree & (st["parent"] > 0) & tree[st["parent"] - 1]  # into a parent of the same launch
    flops = front_flops(c[inside], w[inside]) + float(np.sum(w[adds] * (w[adds] + 1.0) / 2.0))
    assert work["small_front"] == pytest.approx(flops, rel=1e-12)
    large = (n > 64) & (~low if kind == -1 else True)
    assert (work["potrf"] > 0) == (kind != 1 and large.any())
    assert (work["front"] > 0) == (kind == 1)
    s.close()
