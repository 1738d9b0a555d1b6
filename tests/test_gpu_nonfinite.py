"""States that are not finite, or that turn an element inside out: the rows of R
that the oracle answers with NaN or infinity, and no others, are not finite, in
residuals, localizations and the Jacobian kinds' residuals, for every pair of
shape, points and model; the finite rows agree to RTOL of the parity tests (1e-11
normwise, over the rows that no such element touches)."""
import numpy as np
import pytest

import oracle as O
from tests.helpers import MATS, RTOL, mat_row, oracle_mesh_from, random_history, random_state, rel

pytestmark = pytest.mark.gpu

g = pytest.importorskip("goal_amd")


def states(n, seed):
    """A state, and the same with one node's u or p NaN, infinite or far off."""
    x = random_state(n, seed, scale_u=0.002)
    at = 4 * (n // 2)
    for name, k, v in (("nan", at, np.nan), ("nan p", at + 3, np.nan), ("inf", at + 1, np.inf), ("far", at + 2, 0.9)):
        y = x.copy()
        y[k] = v
        yield name, y


def same(a, b):
    bad = ~np.isfinite(b)
    return np.array_equal(~np.isfinite(a), bad) and rel(a[~bad], b[~bad]) < RTOL


@pytest.mark.parametrize("model", [0, 1, 2])
@pytest.mark.parametrize("order,quad", [(1, 1), (1, 2), (2, 1), (2, 2)])
def test_rows_that_are_not_finite(order, quad, model):
    disc = g.Disc.box(3, 2, 2, order=order, jitter=0.1, seed=1)
    st = g.States(disc, model, quad)
    m = MATS[model]
    mech = g.Mechanics(disc, st, [g.MaterialSpec(**m)], quad_order=quad)
    mech.set_option("check", 0)  # a return map that fails is part of the answer
    om = oracle_mesh_from(disc)
    ost = O.States(om, model, quad)
    if model == 2:
        Fp, eq = random_history(disc.num_elems * st.nq, 8)
        for name, v in (("Fp_old", Fp), ("Fp", Fp), ("eqps_old", eq), ("eqps", eq)):
            st.set(name, v)
            getattr(ost, name)[:] = v
    z = random_state(disc.num_nodes, 9)
    dz = g.DeviceArray.from_host(z)
    si = g.SolInfo(disc)
    rows = [mat_row(m)]
    for name, x in states(disc.num_nodes, 6):
        disc.set_soln(x)
        with np.errstate(all="ignore"):
            Ro, _ = O.assemble(O.K_RESIDUAL, om, model, rows, x, ost, quad_order=quad, save=False)
            Lo, _ = O.assemble(O.K_LOCALIZE, om, model, rows, x, ost, quad_order=quad, save=False, z_diff=z,
                               z_coarse=z)
        si.zero_R()
        mech.residual(si, save_states=False)
        assert same(si.R(), Ro), name
        si.zero_R()
        mech.localize(si, dz.ptr.value, dz.ptr.value)
        assert same(si.R(), Lo), name
        si.zero_all()
        mech.jacobian(si, save_states=False)
        assert same(si.R(), Ro), name
