"""The residual kinds' point-per-thread kernel and its sums by node, for every
pair of shape, points and model, against the oracle (RTOL of the parity tests,
1e-11 normwise): meshes whose points end inside a block, stabilization on and
off, sums added to earlier ones, and the localization's weights.  Where the random
iterate turns a point inside out (J < 0, which J2's J^(-2/3) answers with NaN),
the same entries have to be NaN as in the oracle's answer."""
import numpy as np
import pytest

import oracle as O
from tests.helpers import MATS, RTOL, mat_row, oracle_mesh_from, random_history, random_state, rel

pytestmark = pytest.mark.gpu

g = pytest.importorskip("goal_amd")


def close(a, b):
    a, b = np.ravel(a), np.ravel(b)
    bad = np.isnan(b)
    return np.array_equal(np.isnan(a), bad) and rel(a[~bad], b[~bad]) < RTOL


@pytest.mark.parametrize("model", [0, 1, 2])
@pytest.mark.parametrize("order,quad", [(1, 1), (1, 2), (2, 1), (2, 2)])
@pytest.mark.parametrize("dims", [(1, 1, 1), (5, 3, 2)])
def test_residual_kinds_match_oracle(dims, order, quad, model):
    disc = g.Disc.box(*dims, order=order, jitter=0.1, seed=5)
    st = g.States(disc, model, quad)
    m = MATS[model]
    mech = g.Mechanics(disc, st, [g.MaterialSpec(**m)], quad_order=quad)
    x = random_state(disc.num_nodes, 6)
    disc.set_soln(x)
    om = oracle_mesh_from(disc)
    ost = O.States(om, model, quad)
    if model == 2:
        Fp, eq = random_history(disc.num_elems * st.nq, 8)
        for name in ("Fp_old", "Fp"):
            st.set(name, Fp)
            getattr(ost, name)[:] = Fp
        for name in ("eqps_old", "eqps"):
            st.set(name, eq)
            getattr(ost, name)[:] = eq
    si = g.SolInfo(disc)
    for stab in (True, False):
        mech.set_option("stabilization", int(stab))
        si.zero_R()
        mech.residual(si, save_states=True)
        mech.residual(si, save_states=False)  # added
        Ro, _ = O.assemble(O.K_RESIDUAL, om, model, [mat_row(m)], x, ost, quad_order=quad, stabilization=stab)
        assert close(si.R(), 2 * Ro)
        assert close(st.get("sigma"), ost.sigma)
        if model == 2:
            assert close(st.get("Fp"), ost.Fp) and close(st.get("eqps"), ost.eqps)
        zd, zc = random_state(disc.num_nodes, 9), random_state(disc.num_nodes, 10)
        dd, dc = g.DeviceArray.from_host(zd), g.DeviceArray.from_host(zc)
        si.zero_R()
        mech.localize(si, dd.ptr.value, dc.ptr.value)
        Lo, _ = O.assemble(O.K_LOCALIZE, om, model, [mat_row(m)], x, ost, quad_order=quad, stabilization=stab,
                           save=False, z_diff=zd, z_coarse=zc)
        assert close(si.R(), Lo)
