"""Device memory of a solve.  mfd_solve_device_noalloc takes every vector from a
fixed 128 MiB array; a solve needs at most one entry per update row of the
elimination tree and four per unknown and right-hand side, whatever the shape
of the fronts: chains and stars of large fronts, whose partial sums would
otherwise take the most, are solved up to that many right-hand sides."""
import numpy as np
import pytest

import mfdag
from mfdag import problems as P
from test_front_kinds import chain, natural
from test_solve_tasks import arrow
from test_zz_no_alloc import DeviceArray


@pytest.mark.parametrize("block", [0, 1, 256])
@pytest.mark.parametrize("name,make", [
    ("chain_300", lambda: chain(300, 8)), ("chain_64", lambda: chain(64, 12)), ("chain_1", lambda: chain(1, 40)),
    ("star_600", lambda: arrow(600, 1500, 3, 1)), ("star_2", lambda: arrow(2, 140, 9, 1)),
], ids=lambda v: v if isinstance(v, str) else "")
def test_every_wait_is_for_earlier_tasks(name, make, block):
    p = make()
    s = mfdag.Solver(nb=64, host_only=True)
    s.analyze(p.ccs_col, p.ccs_row, 0, natural(p))
    s.solve_block = block
    assert s.check_schedule(0) == (0, "")
    s.close()


@pytest.mark.gpu
@pytest.mark.parametrize("precision", [mfdag.FP64, mfdag.FP32_IR], ids=["fp64", "fp32_ir"])
@pytest.mark.parametrize("block", [0, 256])
def test_partial_sums_over_many_rows(block, precision):
    """Fronts of 600 columns and 1500 update rows, whose partial sums are formed
    over 512 rows at a time."""
    p = arrow(600, 1500, 3, 1)
    s = mfdag.Solver(nb=64)
    s.analyze(p.ccs_col, p.ccs_row, 0, natural(p))
    s.solve_block = block
    assert s.factorize(p.val, precision) == 0
    for nrhs in (1, 17):
        _, b = P.rhs(p, nrhs, seed=nrhs)
        assert P.backward_error(p, s.solve(b.copy()), b) <= 1e-14
    s.close()


@pytest.mark.gpu
@pytest.mark.parametrize("name,make", [
    ("chain_512", lambda: chain(512, 6)), ("chain_1024", lambda: chain(1024, 4)),
    ("star_1024", lambda: arrow(1024, 700, 3, 1)), ("star_300", lambda: arrow(300, 2000, 3, 1)),
    ("chain_300", lambda: chain(300, 8)), ("grid3d_14", lambda: P.weighted_laplacian_3d(14, seed=3)),
], ids=lambda v: v if isinstance(v, str) else "")
def test_solves_up_to_the_fixed_array(name, make):
    p = make()
    s = mfdag.Solver(nb=64)
    s.analyze(p.ccs_col, p.ccs_row, 0, p.perm if p.perm is not None else natural(p))
    assert s.factorize(p.val) == 0
    per = 8 * (int(s.structure()["work_size"].sum()) + 4 * p.n)
    nrhs = (128 << 20) // per // 16 * 16
    _, few = P.rhs(p, 16, seed=2)
    b = np.asfortranarray(np.tile(few, nrhs // 16))
    d_b = DeviceArray(b)
    print(f"{name}: n={p.n} nrhs={nrhs}", flush=True)
    assert s.solve_device_noalloc(d_b.ptr.value, nrhs, p.n) == 0
    x = d_b.download()
    d_b.free()
    assert P.backward_error(p, x[:, :16], few) <= 1e-14
    assert all(np.array_equal(x[:, k:k + 16], x[:, :16]) for k in range(16, nrhs, 16))
    s.close()
