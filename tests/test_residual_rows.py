"""The refinement residual at the row lengths where its number of lanes per row
changes (12, 40 and 72 entries on average), odd orders, and right-hand sides
around its groups of four."""
import numpy as np
import pytest

import mfdag
from mfdag import problems as P


def band(n, k, seed):
    """Half bandwidth k: 2 k + 1 entries in a row."""
    rng = np.random.Generator(np.random.PCG64(seed))
    j = np.concatenate([np.arange(n - d) for d in range(1, k + 1)])
    i = np.concatenate([np.arange(d, n) for d in range(1, k + 1)])
    v = rng.uniform(-1.0, 1.0, len(i))
    diag = 1.0 + np.bincount(i, abs(v), n) + np.bincount(j, abs(v), n)
    cc, rr, vv = P.lower_ccs(n, np.concatenate([np.arange(n), i]), np.concatenate([np.arange(n), j]),
                             np.concatenate([diag, v]))
    return P.Problem(n, cc, rr, vv, None, f"band_{n}_{k}")


@pytest.mark.gpu
@pytest.mark.parametrize("n,k", [(515, 2), (515, 6), (515, 7), (1031, 20), (1031, 21), (1031, 36), (1031, 40), (77, 76)],
                         ids=lambda v: str(v))
def test_residual_against_numpy(n, k):
    """r = b - A x in FP64: to the rounding of rows of 2 k + 1 products and a
    right-hand side, (2 k + 3) 2^-53 of |b| + |A| |x|."""
    p = band(n, k, seed=n + k)
    s = mfdag.Solver(nb=64)
    s.analyze(p.ccs_col, p.ccs_row, 256, np.arange(1, n + 1, dtype=np.int32))
    A = p.scipy()
    norm, dense = abs(A).sum(axis=1).max(), A.toarray().astype(np.longdouble)
    for prec in (mfdag.FP64, mfdag.FP32_IR):
        assert s.factorize(p.val, prec) == 0
        for nrhs in (1, 4, 7):
            _, b = P.rhs(p, nrhs, seed=nrhs)
            x = s.solve(b.copy())
            assert P.backward_error(p, x, b) <= 1e-14
            eta = s.solve_errors(nrhs)["eta"]
            r = np.abs(b.astype(np.longdouble) - dense @ x.astype(np.longdouble)).max(axis=0)
            scale = norm * np.abs(x).max(axis=0) + np.abs(b).max(axis=0)
            assert np.all(np.abs(eta - r / scale) <= (2 * k + 3) * 2.0 ** -53)
    s.close()
