"""Two handles driven from two threads at the same time.  The launches for the
bottom of the tree and for the solves fill the GPU with workgroups that wait
for each other; beside the other handle's they end all the same, and, every sum
having a fixed order, with the results that they give alone."""
import threading

import numpy as np
import pytest

import mfdag
from mfdag import problems as P


def opened(p, max_zero, graph):
    s = mfdag.Solver(nb=64, graph=graph)
    if isinstance(p, list):
        s.analyze_batch([(q.ccs_col, q.ccs_row) for q in p], max_zero, [q.perm for q in p])
        p = P.batch_problem(p)
    else:
        s.analyze(p.ccs_col, p.ccs_row, max_zero, p.perm)
    _, b = P.rhs(p, 3, seed=1)
    return s, p, b


@pytest.mark.gpu
@pytest.mark.parametrize("precision", [mfdag.FP64, mfdag.FP32_IR], ids=["fp64", "fp32_ir"])
@pytest.mark.parametrize("graph", [False, True])
def test_results_beside_another_handle(graph, precision):
    pair = [opened(P.weighted_laplacian_3d(24, seed=4), 4096, graph),
            opened(P.batch_anisotropic(60, seed=6, lo=8, hi=60), 256, graph)]
    alone = []
    for s, p, b in pair:
        assert s.factorize(p.val, precision) == 0
        alone.append(s.solve(b.copy()))
    start, wrong = threading.Barrier(2), []

    def drive(k):
        s, p, b = pair[k]
        start.wait()
        for it in range(25):
            ok = s.factorize(p.val, precision) == 0 and np.array_equal(s.solve(b.copy()), alone[k])
            if not ok:
                wrong.append((k, it))

    threads = [threading.Thread(target=drive, args=(k,)) for k in range(2)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert wrong == []
    for s, _, _ in pair:
        s.close()
