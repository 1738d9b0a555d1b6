"""The solver's matrix products where rows are ragged: nodes of few and of many
neighbours (more than a group of lanes reads at once), meshes of one and of
several multigrid levels.  The matrix is random on the mesh's graph and
diagonally dominant by a factor of two, so the solve converges in a few steps
and the true residual can be held to the requested one: the solver stops at
rtol ||b|| by its own products; the host's differ from them by rounding
(relative 1e-13 and less), so 1.01 rtol bounds the host's residual."""
import numpy as np
import pytest

from tests.helpers import fan_mesh

pytestmark = pytest.mark.gpu

g = pytest.importorskip("goal_amd")


def disc_of(kind, order):
    if kind == "fan":
        return g.Disc.from_arrays(order, *fan_mesh(order=order, subdiv=2))
    return g.Disc.box(*dict(cell=(1, 1, 1), ragged=(9, 1, 2), block=(7, 6, 5))[kind], order=order, jitter=0.1, seed=2)


@pytest.mark.parametrize("precond", [g.PRECOND_AMG, g.PRECOND_BLOCK_JACOBI])
@pytest.mark.parametrize("order", [1, 2])
@pytest.mark.parametrize("kind", ["cell", "ragged", "block", "fan"])
def test_solve_meets_its_residual(kind, order, precond):
    disc = disc_of(kind, order)
    rp, cols = disc.graph()
    rng = np.random.default_rng(9)
    n = disc.num_dofs
    vals = rng.uniform(-1.0, 1.0, disc.nnz)
    rows = np.repeat(np.arange(n), np.diff(rp))
    off = rows != cols
    vals[~off] = 2.0 * np.bincount(rows[off], np.abs(vals[off]), n) + 0.1
    b = rng.standard_normal(n)
    si = g.SolInfo(disc)
    si.set(vals=vals)
    bd, xd = g.DeviceArray.from_host(b), g.DeviceArray(n)
    xd.fill(0.0)
    rtol = 1e-9
    its, relres = si.solve(bd, xd, rtol=rtol, max_iters=200, precond=precond)
    x = xd.numpy()
    r = b - np.bincount(rows, vals * x[cols], n)
    assert relres <= rtol and its < 60
    assert np.linalg.norm(r) <= 1.01 * rtol * np.linalg.norm(b)
