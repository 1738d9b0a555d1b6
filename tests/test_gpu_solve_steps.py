"""The solver's queued Arnoldi steps where a step is the last one: restarts of
one and of a few steps, iteration limits on either side of a restart, a
converged start and a zero right side; twice, for the same bits.

Tolerance: the solver's own and the host's residual differ by rounding of the
products (relative 1e-13 of ||b|| and less), so 1e-11 ||b|| bounds it."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

g = pytest.importorskip("goal_amd")


@pytest.mark.parametrize("precond", [g.PRECOND_AMG, g.PRECOND_BLOCK_JACOBI])
@pytest.mark.parametrize("restart,limit", [(1, 0), (1, 1), (1, 5), (4, 3), (4, 4), (4, 9), (50, 200)])
def test_last_steps(restart, limit, precond):
    disc = g.Disc.box(6, 5, 4, order=2, jitter=0.1, seed=2)
    rp, cols = disc.graph()
    rng = np.random.default_rng(9)
    n = disc.num_dofs
    vals = rng.uniform(-1.0, 1.0, disc.nnz)
    rows = np.repeat(np.arange(n), np.diff(rp))
    off = rows != cols
    vals[~off] = 1.2 * np.bincount(rows[off], np.abs(vals[off]), n) + 0.1
    b = rng.standard_normal(n)
    si = g.SolInfo(disc)
    si.set(vals=vals)
    bd, xd = g.DeviceArray.from_host(b), g.DeviceArray(n)
    runs = []
    for _ in range(2):
        xd.fill(0.0)
        its, relres = si.solve(bd, xd, rtol=1e-9, max_iters=limit, restart=restart, precond=precond)
        x = xd.numpy()
        res = np.linalg.norm(b - np.bincount(rows, vals * x[cols], n)) / np.linalg.norm(b)
        assert its <= limit and (relres <= 1e-9 or its == limit)
        assert abs(res - relres) < 1e-11
        runs.append((its, relres, x))
    assert runs[0][:2] == runs[1][:2] and np.array_equal(runs[0][2], runs[1][2])
    if limit == 200:
        assert relres <= 1e-9
        assert si.solve(bd, xd, rtol=2.0, max_iters=limit, restart=restart, precond=precond)[0] == 0  # met at the start
        zero = g.DeviceArray(n)
        zero.fill(0.0)
        xd.fill(0.0)
        assert si.solve(zero, xd, max_iters=limit, restart=restart, precond=precond) == (0, 0.0)
        assert not xd.numpy().any()
