"""Sums over a node's elements: the functionals' derivative (element values by
incidence record, then summed) and the recovered nodal means of the features,
at nodes with one, a few and 80 or 320 elements and with element sets left out.

Tolerances: RTOL of the parity tests (FP64 on both sides, at most 320 terms a
node); the features' as in their own tests, through the recovered means."""
import numpy as np
import pytest

import oracle as O
from oracle import learned as L
from tests.helpers import MATS, RTOL, fan_mesh, mat_row, random_history, random_state, rel

pytestmark = pytest.mark.gpu

g = pytest.importorskip("goal_amd")


@pytest.mark.parametrize("order", [1, 2])
@pytest.mark.parametrize("model", [0, 1, 2])
@pytest.mark.parametrize("subdiv", [0, 1, 2])
def test_qoi_derivative_sums(order, model, subdiv):
    X, conn = fan_mesh(order=order, subdiv=subdiv, jitter=0.05, seed=3)
    ne = conn.shape[0]
    sets = (np.arange(ne) % 3 == 0).astype(np.int32)
    mats = [dict(MATS[model]), dict(MATS[model], E=700.0)]
    x = random_state(X.shape[0], 4, scale_u=0.005)
    om = O.Mesh(order, X, conn, sets)
    disc = g.Disc.from_arrays(order, X, conn, sets)
    disc.set_elem_sets(2, sets)
    disc.set_soln(x)
    st, ost = g.States(disc, model, order), O.States(om, model, order)
    mech = g.Mechanics(disc, st, [g.MaterialSpec(**m) for m in mats], quad_order=order)
    if model == 2:
        Fp, eq = random_history(ne * st.nq, 9)
        for f, v in (("Fp_old", Fp), ("Fp", Fp), ("eqps_old", eq), ("eqps", eq)):
            getattr(ost, f)[:] = v
            st.set(f, v)
    si = g.SolInfo(disc)
    for kind, only in ((g.QOI_AVG_DISP, -1), (g.QOI_AVG_VM, -1), (g.QOI_AVG_VM, 1)):
        val, ev, dm = O.qoi(kind, om, model, [mat_row(m) for m in mats], x, ost, quad_order=order, derivative=True,
                            qoi_set=only)
        si.zero_dMdu()
        v, e = mech.qoi(kind, si, elem_set=only, elem_values=True)
        assert abs(v - val) <= RTOL * abs(val) and rel(e, ev) < RTOL
        assert rel(si.dMdu(), dm) < RTOL
        mech.qoi(kind, si, elem_set=only)  # added to what is there
        assert rel(si.dMdu(), 2 * dm) < RTOL


@pytest.mark.parametrize("order", [1, 2])
@pytest.mark.parametrize("subdiv", [0, 1, 2])
def test_recovered_means(order, subdiv):
    X, conn = fan_mesh(order=order, subdiv=subdiv, jitter=0.05, seed=3)
    ne = conn.shape[0]
    disc = g.Disc.from_arrays(order, X, conn, np.zeros(ne, dtype=np.int32))
    x = random_state(X.shape[0], 4, scale_u=0.005)
    disc.set_soln(x)
    st = g.States(disc, 1, order)
    mech = g.Mechanics(disc, st, [g.MaterialSpec(**MATS[1])], quad_order=order)
    _, ev = mech.qoi(g.QOI_AVG_VM, None, elem_set=-1, elem_values=True)
    feat = g.learn_features(mech, 0.25).numpy(ne * 12).reshape(ne, 12)
    ref = L.features(X, conn, x.reshape(-1, 4), ev, MATS[1]["E"], MATS[1]["nu"], None, 0.25)
    assert np.allclose(feat, ref, rtol=2e-6, atol=2e-6)
