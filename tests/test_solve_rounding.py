"""Rounding of the solves' long sums.  Two 256-column blocks coupled to `w` rows
by B with L = [I; B] and an identity Schur complement, all exact by
construction: with b = (b1, 0) the solution's last w entries are -B b1, a sum
of 256 positive products per front formed by the forward sweep, and with
b = (0, b2) its first ones are -B^T b2, w products formed by the backward one.

A running sum s rounds by ulp(s) / sqrt(12) rms at every step.  With ulp(s)
about 0.72 * 2^-52 s, summing K equal terms in one chain gives 0.208 sqrt(K /
3) 2^-52 of the sum: 1.9 for K = 256, 1.36 for K = 128; in chains of at most
64 entries, added to each other, at most 0.72.  The bound is 1."""
import numpy as np
import pytest

import mfdag
from mfdag import problems as P

C, NRHS = 256, 16


def exact_blocks(w, seed):
    rng = np.random.Generator(np.random.PCG64(seed))
    B = [rng.integers(512, 1024, (w, C)) * 2.0 ** -10 for _ in range(2)]
    n = 2 * C + w
    A = np.zeros((n, n))
    A[:2 * C, :2 * C] = np.eye(2 * C)
    for k in range(2):
        A[2 * C:, C * k:C * k + C] = B[k]
    A[2 * C:, 2 * C:] = np.eye(w) + sum(b @ b.T for b in B)  # exact: 20-bit products, 512 of them
    pat = np.zeros((n, n), dtype=bool)
    pat[:C, :C] = pat[C:2 * C, C:2 * C] = pat[2 * C:, :] = True
    i, j = np.nonzero(np.tril(pat))
    cc, rr, vv = P.lower_ccs(n, i, j, A[i, j])
    return n, cc, rr, vv, B, rng


@pytest.mark.gpu
@pytest.mark.parametrize("block", [0, 256])
@pytest.mark.parametrize("w", [128, 300])
def test_long_sums(w, block):
    n, cc, rr, vv, B, rng = exact_blocks(w, seed=w)
    s = mfdag.Solver(nb=64)
    s.analyze(cc, rr, 0, np.arange(1, n + 1, dtype=np.int32))
    s.solve_block = block
    st = s.structure()  # the second block and the rows form the root
    assert st["supernode_size"][0] == C and st["work_size"][0] == w
    assert s.factorize(vv) == 0
    F = np.tril(s.front(1))
    assert np.array_equal(F[:C, :C], np.eye(C)) and np.array_equal(F[C:, :C], B[0])
    L = np.longdouble
    b = np.zeros((n, NRHS))
    b[:C] = rng.uniform(1.0, 2.0, (C, NRHS))
    got, want = s.solve(b.copy())[2 * C:], -(B[0].astype(L) @ b[:C].astype(L))
    rms = float(np.sqrt(np.mean(((got - want) / want) ** 2))) * 2.0 ** 52
    print(f"forward, w={w} block={block}: {rms:.3f}", flush=True)
    assert rms <= 1.0
    b = np.zeros((n, NRHS))
    b[2 * C:] = rng.uniform(1.0, 2.0, (w, NRHS))
    got, want = s.solve(b.copy())[:C], -(B[0].T.astype(L) @ b[2 * C:].astype(L))
    rms = float(np.sqrt(np.mean(((got - want) / want) ** 2))) * 2.0 ** 52
    print(f"backward, w={w} block={block}: {rms:.3f}", flush=True)
    assert rms <= 1.0
    s.close()
